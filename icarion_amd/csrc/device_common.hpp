// device_common.hpp - device-side building blocks of the gfx950 ion-step
// kernels: 3-vectors, the Philox4x32-10 counter RNG and per-(ion, step)
// random streams.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace icarion {

// ---- physical constants (reference src/utils/constants.h:13-65) ----------
constexpr double kPi = 3.14159265358979323846;
constexpr double kBoltzmann = 1.380649e-23;
constexpr double kLoschmidt = 2.6867811e25;
constexpr double kEpsilon0 = 8.854187817e-12;
constexpr double kStpTemp = 273.15;
// thresholds (HSSCollisionHandler.cpp:20, CollisionKernels.h:172-178,
// CylindricalGeometry.h:245, AnalyticalFieldModel.cpp:12)
constexpr double kMinRelativeVelocity = 1e-10;
constexpr double kMinVelocityMag = 1e-12;
constexpr double kMinContactDistSq = 1e-24;
constexpr int kEhssMaxAttempts = 256;
constexpr int kBmaxExpansionAttempt = 64;
constexpr double kBmaxExpansionFactor = 1.5;
constexpr double kGeomEpsilon = 1e-12;
constexpr double kMinVoltage = 1e-12;

// Keeps a wave-uniform branch a branch: without it the compiler computes both
// sides in every step and selects.  MEM: the kernel's uniform records lie in memory
// (the general field arrays' axes and terms; everything in a unit that defines
// KEEP_BRANCH_READS_ONLY): its branches are held by a scheduling barrier that nothing
// is bound by, since an asm statement counts as a write to memory and takes the
// scalar loads, and the loop's own constants, away from every record read after it
// (RK4 steps of 300,000 ions in a field of three terms took 6 % longer).
#ifdef KEEP_BRANCH_READS_ONLY
constexpr bool kRecordsInMemory = true;
#else
constexpr bool kRecordsInMemory = false;
#endif
template <bool MEM = kRecordsInMemory>
__device__ __forceinline__ void keep_branch() {
    if constexpr (MEM) __builtin_amdgcn_sched_barrier(0x7ff);
    else asm volatile("");
}

template <typename T>
struct vec3 {
    T x, y, z;
};
template <typename T>
__device__ __forceinline__ vec3<T> operator+(vec3<T> a, vec3<T> b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
template <typename T>
__device__ __forceinline__ vec3<T> operator-(vec3<T> a, vec3<T> b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
template <typename T>
__device__ __forceinline__ vec3<T> operator*(vec3<T> a, T s) { return {a.x * s, a.y * s, a.z * s}; }
template <typename T>
__device__ __forceinline__ T dot(vec3<T> a, vec3<T> b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
template <typename T>
__device__ __forceinline__ vec3<T> cross(vec3<T> a, vec3<T> b) {
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ vec3<double> mat_mul(const double m[9], vec3<double> v) {
    return {m[0] * v.x + m[1] * v.y + m[2] * v.z,
            m[3] * v.x + m[4] * v.y + m[5] * v.z,
            m[6] * v.x + m[7] * v.y + m[8] * v.z};
}

// ---- Philox4x32-10 (Salmon et al., SC'11), published round constants -----
struct u32x4 {
    uint32_t v[4];
};

// One round takes two 32 x 32 -> 64-bit products, each a single v_mad_u64_u32
// (as a 64-bit product; a low and a high 32-bit multiply issue twice), and two
// three-way exclusive ors, each a single v_bitop3_b32 (truth table 0x96).  The
// FP32 step kernels are bound by vector issue and the rounds were a third of
// it: with the keys below, 200,003 ions x 10,000 HSS steps went from 28.0 to
// 23.6 ms and 1M ions x 20,000 Boris + kick steps from 143 to 123 ms.
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}

__device__ __forceinline__ u32x4 philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                               uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint64_t p0 = static_cast<uint64_t>(0xD2511F53u) * c0;
        const uint64_t p1 = static_cast<uint64_t>(0xCD9E8D57u) * c2;
        // the step's streams have a wave-uniform block, step and key: then c2
        // stays uniform in the first round and c0 in the second, and a plain
        // exclusive or keeps them (and their products) on the scalar unit
        const uint32_t h1 = static_cast<uint32_t>(p1 >> 32), h0 = static_cast<uint32_t>(p0 >> 32);
        c0 = r == 1 ? h1 ^ c1 ^ k0 : xor3(h1, c1, k0);
        c2 = r == 0 ? h0 ^ c3 ^ k1 : xor3(h0, c3, k1);
        c1 = static_cast<uint32_t>(p1);
        c3 = static_cast<uint32_t>(p0);
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    u32x4 o;
    o.v[0] = c0; o.v[1] = c1; o.v[2] = c2; o.v[3] = c3;
    return o;
}

// 53-bit uniform on (0, 1] from two words: k*2^-53 + 2^-54, k = hi[31:5]:lo[31:6].
__device__ __forceinline__ double uniform53(uint32_t hi, uint32_t lo) {
    const uint64_t k = (static_cast<uint64_t>(hi >> 5) << 26) | static_cast<uint64_t>(lo >> 6);
    return static_cast<double>(k) * 0x1.0p-53 + 0x1.0p-54;
}

// 24-bit uniform on (0, 1) from one word.
__device__ __forceinline__ float uniform24(uint32_t w) {
    return static_cast<float>(w >> 8) * 0x1.0p-24f + 0x1.0p-25f;
}

// ---- FP64 functions of the random draws ------------------------------------
// The general sin, cos and log were a third of the FP64 HSS step's instructions:
// they reduce any argument.  A draw is a uniform in (0, 1], so the angle is
// reduced exactly in revolutions before it meets 2 pi, and the logarithm has no
// special values.  The polynomials interpolate at Chebyshev nodes (evaluated in
// extended precision; relative error of the fit below 5e-18).  Largest errors
// over 4e5 draws against extended precision: sine and cosine 1.5e-16 absolute,
// where the general functions of the rounded product 2 pi u had 6.9e-16;
// logarithm 0.9 units in the last place.
template <int N>
__device__ __forceinline__ double horner(const double (&p)[N], double w) {
    double r = p[N - 1];
#pragma unroll
    for (int i = N - 2; i >= 0; --i) r = fma(r, w, p[i]);
    return r;
}

// sine and cosine of u revolutions, 0 <= u <= 1: u = k / 4 + r with |r| <= 1/8
__device__ __forceinline__ void sincos_rev(double u, double& sn, double& cs) {
    constexpr double ps[] = {6.283185307179586, -41.341702240399634, 81.60524927594857,
                             -76.70585970444363, 42.058685043183644, -15.09380560388465,
                             3.7808998789812995};
    constexpr double pc[] = {-19.739208802178716, 64.93939402266825, -85.45681720664702,
                             60.244641353320404, -26.426253328264924, 7.903208845913531,
                             -1.699058459304078};
    const double k = rint(4.0 * u);
    const double r = fma(k, -0.25, u);
    const double w = r * r;
    const double s = r * horner(ps, w);
    const double c = fma(w, horner(pc, w), 1.0);
    const int q = static_cast<int>(k);
    const double a = (q & 1) ? c : s, b = (q & 1) ? s : c;
    sn = (q & 2) ? -a : a;
    cs = ((q + 1) & 2) ? -b : b;
}

// natural logarithm of 0 < u <= 1 (a normal number): u = 2^e m, m in
// [sqrt(1/2), sqrt(2)), log m = 2 atanh(s) with s = (m - 1) / (m + 1)
__device__ __forceinline__ double log_unit(double u) {
    constexpr double pa[] = {0.3333333333333335, 0.1999999999994975, 0.14285714312988573,
                             0.11111105567284828, 0.09091444569747409, 0.07665860591894315,
                             0.0730822712981302};
    double m = __builtin_amdgcn_frexp_mant(u);
    int e = __builtin_amdgcn_frexp_exp(u);
    const bool low = m < 0.70710678118654752;
    m = low ? m + m : m;
    e = low ? e - 1 : e;
    const double f = m - 1.0, d = m + 1.0;
    double y = __builtin_amdgcn_rcp(d);
    y = fma(y, fma(-d, y, 1.0), y);
    y = fma(y, fma(-d, y, 1.0), y);
    double s = f * y;
    s = fma(fma(-d, s, f), y, s);
    const double z = s * s;
    const double ed = static_cast<double>(e);
    // 2 s = f - s f; ln 2 in two parts, the first times e exact
    const double t = s * (f - 2.0 * (z * horner(pa, z)));
    return fma(ed, 0.6931471805598903, f - fma(ed, -5.497924164543644e-14, t));
}

// Per-(ion, step) stream, counter = (block, ion, step_lo, step_hi), key =
// (seed_lo, seed_hi).  FP64 draws take two words (the oracle's PhiloxStream
// hands out the identical sequence); FP32 draws take one word.
struct PhiloxStream {
    uint32_t k0, k1, ion, s_lo, s_hi;
    uint32_t block;
    uint32_t buf[4];
    int pos;
    bool n_have;       // normal_f64: the second value of the last pair is pending
    double n_cached;

    __device__ __forceinline__ PhiloxStream(uint64_t seed, uint32_t ion_index, uint64_t step)
        : k0(static_cast<uint32_t>(seed)), k1(static_cast<uint32_t>(seed >> 32)), ion(ion_index),
          s_lo(static_cast<uint32_t>(step)), s_hi(static_cast<uint32_t>(step >> 32)), block(0),
          pos(4), n_have(false), n_cached(0.0) {}

    // The round keys as scalar adds in this call (the key words, wave-uniform,
    // are tied to the step's counter).  Hoisted out of the step loop the 18 keys
    // overflow the scalar registers and come back by v_readlane, on the vector
    // pipe that bounds the step kernels.
    __device__ __forceinline__ void refill() {
        uint32_t r0 = __builtin_amdgcn_readfirstlane(k0), r1 = __builtin_amdgcn_readfirstlane(k1);
        asm("" : "+s"(r0), "+s"(r1) : "s"(__builtin_amdgcn_readfirstlane(s_lo)));
        const u32x4 o = philox4x32_10(block, ion, s_lo, s_hi, r0, r1);
        buf[0] = o.v[0]; buf[1] = o.v[1]; buf[2] = o.v[2]; buf[3] = o.v[3];
        ++block;
        pos = 0;
    }
    // The words are selected rather than indexed by pos, so that the block
    // stays in registers where the compiler cannot resolve pos (draws inside
    // data-dependent loops); an indexed buffer goes to private memory there.
    // A stream takes FP64 draws only (pos 0 or 2) or FP32 draws only.
    __device__ __forceinline__ double uniform_f64() {
        if (pos >= 4) refill();
        const bool second = pos >= 2;
        const double u = uniform53(second ? buf[2] : buf[0], second ? buf[3] : buf[1]);
        pos += 2;
        return u;
    }
    // Standard normal by Box-Muller on two FP64 draws, the pair's second value
    // kept for the next call (the oracle's stream and std::normal_distribution
    // hand out both values of a pair), so consecutive collision substeps share
    // pairs as the engine's one stream per ion does.
    __device__ __forceinline__ double normal_f64() {
        if (n_have) {
            n_have = false;
            return n_cached;
        }
        const double u1 = uniform_f64();
        const double u2 = uniform_f64();
        const double r = sqrt(-2.0 * log_unit(u1));
        double sn, cs;
        sincos_rev(u2, sn, cs);
        n_cached = r * sn;
        n_have = true;
        return r * cs;
    }
    __device__ __forceinline__ float uniform_f32() {
        if (pos >= 4) refill();
        const uint32_t w = pos == 0 ? buf[0] : pos == 1 ? buf[1] : pos == 2 ? buf[2] : buf[3];
        const float u = uniform24(w);
        pos += 1;
        return u;
    }
};

}  // namespace icarion
