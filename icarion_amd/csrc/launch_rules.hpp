// launch_rules.hpp - how the EHSS and surrogate kernels spread a cloud over the
// chip's 1024 SIMDs (host code, without HIP).
#pragma once

#include <cstdint>

namespace icarion {

constexpr uint32_t kSimds = 1024;   // 256 CUs of four

// Wavefronts per SIMD of the geometry EHSS kernel: two (256 registers and 64 KB of
// LDS per workgroup), except for RK4 in a field array and fields of several terms,
// whose registers leave room for one (two would spill 50 and more).
constexpr uint32_t ehss_waves_per_simd(int integrator, bool field_array, bool general_array) {
    return general_array || (field_array && integrator == 0) ? 1u : 2u;
}

// Ions per wavefront of the geometry EHSS kernel.  A wavefront works through its
// colliding ions one after another, so the ions are spread evenly over the least
// number of full rounds of the wavefronts that the chip holds at a time.
inline uint32_t ehss_ions_per_wave(uint32_t n_ions, uint32_t waves_per_simd) {
    const uint64_t slots = uint64_t(kSimds) * waves_per_simd;
    const uint64_t rounds = (n_ions + 64 * slots - 1) / (64 * slots);
    if (rounds == 0) return 1;
    const uint64_t g = (n_ions + rounds * slots - 1) / (rounds * slots);
    return g > 64 ? 64u : static_cast<uint32_t>(g);
}

// The surrogate kernel's instantiation for large clouds (four wavefronts per SIMD
// instead of three): from where the ions are more than two full wavefronts per SIMD.
constexpr uint32_t kSurrogateLargeIons = 64 * 2 * kSimds;
inline bool surrogate_large(uint32_t n_ions) { return n_ions > kSurrogateLargeIons; }

// Ions per wavefront of the surrogate kernel: up to 131,072 ions one or two
// wavefronts per SIMD, evenly filled (a step lasts as long as the workgroup's
// chain, which is shorter with fewer colliding ions: 30,000 ions x 1000 steps
// 5.7 ms with 64 per wavefront, 4.0 ms spread); above that full wavefronts, for
// full MLP blocks.
inline uint32_t surrogate_ions_per_wave(uint32_t n_ions) {
    if (surrogate_large(n_ions)) return 64;
    const uint32_t rounds = n_ions > 64 * kSimds ? 2 : 1;
    const uint32_t g = (n_ions + rounds * kSimds - 1) / (rounds * kSimds);
    return g < 1 ? 1 : g;
}

}  // namespace icarion
