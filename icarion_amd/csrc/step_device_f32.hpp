// step_device_f32.hpp - device functions of the FP32 + Kahan path shared by
// the fixed-step, surrogate, batch and RK45 kernels: compensated accumulation,
// hardware transcendentals, fields, containment, collisions and acceleration
// in FP32 (time and RF phase stay FP64).
#pragma once

#include "step_device.hpp"

namespace icarion {

using f3 = vec3<float>;

// The products and sums of the push are written with their rounding (fmaf): left
// to the compiler, a product is fused with its sum only where both end up in one
// basic block, so that another branch or another kernel around the same lines
// would give other last bits, and an ion another course from its next collision
// test on.
__device__ __forceinline__ f3 fma3(f3 a, float s, f3 b) {
    return f3{fmaf(a.x, s, b.x), fmaf(a.y, s, b.y), fmaf(a.z, s, b.z)};
}
__device__ __forceinline__ float dot(f3 a, f3 b) { return fmaf(a.z, b.z, fmaf(a.x, b.x, a.y * b.y)); }
// |v|^2 of a relative velocity after a push by INTEG (0 RK4, 1 Boris): their
// kernels have always begun the sum with another component.
template <int INTEG>
__device__ __forceinline__ float speed2_f32(f3 v) {
    return fmaf(v.z, v.z, INTEG == 0 ? fmaf(v.x, v.x, v.y * v.y) : fmaf(v.y, v.y, v.x * v.x));
}
__device__ __forceinline__ f3 cross(f3 a, f3 b) {
    return f3{fmaf(a.y, b.z, -(a.z * b.y)), fmaf(a.z, b.x, -(a.x * b.z)), fmaf(a.x, b.y, -(a.y * b.x))};
}
__device__ __forceinline__ f3 mat_mul(const float m[9], f3 v) {
    return f3{dot(f3{m[0], m[1], m[2]}, v), dot(f3{m[3], m[4], m[5]}, v), dot(f3{m[6], m[7], m[8]}, v)};
}

// compensated accumulation: (hi, lo) <- hi + lo + d  (Kahan / Fast2Sum)
__device__ __forceinline__ void kahan_sum(float& hi, float& lo, float y) {
    const float t = hi + y;
    lo = y - (t - hi);
    hi = t;
}
__device__ __forceinline__ void kahan_add(float& hi, float& lo, float d) { kahan_sum(hi, lo, d + lo); }
// the same with d = a s, the product unrounded
__device__ __forceinline__ void kahan_fma(float& hi, float& lo, float a, float s) { kahan_sum(hi, lo, fmaf(a, s, lo)); }

// hardware transcendentals: v_log_f32 (log2), v_exp_f32 (exp2), v_sin/cos_f32
// (argument in revolutions), v_sqrt_f32, v_rcp_f32
__device__ __forceinline__ float fast_ln(float u) { return __builtin_amdgcn_logf(u) * 0.69314718056f; }
__device__ __forceinline__ float fast_cos_rev(float r) { return __builtin_amdgcn_cosf(r); }
__device__ __forceinline__ float fast_sin_rev(float r) { return __builtin_amdgcn_sinf(r); }
__device__ __forceinline__ float fast_sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }


// The corner values of the grid cell an ion is in.  An ion crosses a cell in
// hundreds to thousands of steps, so a caller that keeps this across the stages
// and steps reloads the eight corners only when the cell changes (24 registers
// more).  Gathering them at every stage, the RK4 kernel waited on four dependent
// gathers per step: 1M ions x 2000 HSS steps on a 96 x 96 x 192 grid took 71 ms
// of kernel time, now bound by vector issue and 29 ms; an in-cell test in place
// of the cell search saves another 2 ms (3001 ions x 800: 3.69, 1.96, 1.61 ms),
// the node's address formed for a new cell alone another 4 % (300,000 x 300: 1.58
// and 1.51 ms).
struct CellF32 {
    uint64_t node = ~0ull;   // the cell's first node
    f3 e[8];                 // corner 4 dx + 2 dy + dz
    // the cell's indices for the in-cell test of field_f32; NaN (none passes it)
    // while there is no cell and in the last cell of an axis, where positions
    // past the grid are clamped
    f3 index{__builtin_nanf(""), 0.0f, 0.0f};
};

// c: the stage's RF coefficient (analytic fields) or the stage time (field
// arrays, always in FP64); T: float where the caller holds rounded values.
template <int FIELD, class T>
__device__ __forceinline__ f3 field_f32(const StepParams& P, const FastConst& C, f3 p, T c, T ez, CellF32& kept) {
    if constexpr (FIELD == FIELD_LINEAR) {
        const float c_rf = (float)c;
        f3 E{0.0f, 0.0f, (float)ez};
        if (P.has_rf) {
            E.x = -2.0f * p.x * c_rf;
            E.y = 2.0f * p.y * c_rf;
        }
        return E;
    } else if constexpr (FIELD == FIELD_ORBITRAP) {
        const f3 s{p.x - C.ox, p.y - C.oy, p.z - C.oz};
        f3 l = s;
        if (!P.rot_identity) {
            keep_branch();
            l = mat_mul(C.g2l, s);
        }
        const float r_sq = fmaxf(1e-18f, l.x * l.x + l.y * l.y);
        const float Cf = 1.0f - C.R_char_sq * __builtin_amdgcn_rcpf(r_sq);
        f3 E{C.orbi_hk * l.x * Cf, C.orbi_hk * l.y * Cf, -C.orbi_k * l.z};
        if (!P.rot_identity) {
            keep_branch();
            E = mat_mul(C.l2g, E);
        }
        return E;
    } else {
        // trilinear on float4 nodes; the axis search of the FP64 path on
        // non-uniform axes
        // The cell (rounded down) and the coordinate in it of f = (v - v0) / spacing:
        // the cell from the rounded product, the coordinate rounded once.
        auto cell_of = [](float v, float v0, float inv_d, float& cell_i, float& a) {
            cell_i = floorf((v - v0) * inv_d);
            a = fmaf(v - v0, inv_d, -cell_i);
        };
        // clamped to the grid (branch-free: the ends are selected over the interior)
        auto clamp_cell = [](float v, float v0, float vl, float inv_d, int n, float cell_i, int& i0, float& a) {
            const int i = min(static_cast<int>(cell_i), n - 2);   // negative only below v0
            const bool below = v <= v0, above = v >= vl;
            const float in = static_cast<float>(i) < cell_i ? fmaf(v - v0, inv_d, -static_cast<float>(i)) : a;
            a = below ? 0.0f : above ? 1.0f : in;
            i0 = below ? 0 : above ? n - 2 : i;
        };
        auto loc_axis = [](const float* __restrict__ ax, int n, float v, int& i0, float& a) {
            if (v <= ax[0]) { i0 = 0; a = 0.0f; }
            else if (v >= ax[n - 1] || v != v) { i0 = n - 2; a = 1.0f; }
            else {
                int first = 0, len = n - 1;
                while (len > 0) {
                    const int half = len >> 1;
                    if (ax[first + 1 + half] < v) { first += half + 1; len -= half + 1; }
                    else len = half;
                }
                i0 = first;
                const float dv = ax[first + 1] - ax[first];
                a = dv > 0.0f ? (v - ax[first]) / dv : 0.0f;
            }
        };
        constexpr bool GEN = FIELD == FIELD_ARRAY_X;
        // non-uniform axes and several terms gather the corners each time: the
        // registers of a kept cell cost their kernels a wavefront per SIMD (300,000
        // ions x 150 RK4 steps, one term: 4.7 ms with and 4.3 ms without; three
        // terms, which read other nodes each time: 8.8 and 7.6 ms)
        CellF32 fresh;
        CellF32& cell = GEN ? fresh : kept;
        int ix = 0, iy = 0, iz = 0;
        float ax, ay, az;
        // Still in the kept cell?  The cell follows from the position alone, not from
        // where the ion was before or where its launches begin.  (The coordinate
        // against [0, 1) would decide otherwise within rounding of a face.)
        bool inside = false;
        f3 at{0.0f, 0.0f, 0.0f};
        if (!GEN || !P.axf_x) {
            cell_of(p.x, C.fa_first[0], C.fa_inv[0], at.x, ax);
            cell_of(p.y, C.fa_first[1], C.fa_inv[1], at.y, ay);
            cell_of(p.z, C.fa_first[2], C.fa_inv[2], at.z, az);
        }
        if constexpr (!GEN) inside = (at.x == cell.index.x) & (at.y == cell.index.y) & (at.z == cell.index.z);
        f3 r{0.0f, 0.0f, 0.0f};
        const size_t sy = static_cast<size_t>(P.nx), sz = static_cast<size_t>(P.nx) * P.ny;
        if (!inside) {
            if (GEN && P.axf_x) {
                loc_axis(P.axf_x, P.nx, p.x, ix, ax);
                loc_axis(P.axf_y, P.ny, p.y, iy, ay);
                loc_axis(P.axf_z, P.nz, p.z, iz, az);
            } else {
                clamp_cell(p.x, C.fa_first[0], C.fa_last[0], C.fa_inv[0], P.nx, at.x, ix, ax);
                clamp_cell(p.y, C.fa_first[1], C.fa_last[1], C.fa_inv[1], P.ny, at.y, iy, ay);
                clamp_cell(p.z, C.fa_first[2], C.fa_last[2], C.fa_inv[2], P.nz, at.z, iz, az);
            }
            if (!GEN || P.n_terms <= 1) {
                // the cell's first node by two 32 x 32 -> 64-bit multiply-adds, the
                // other three rows by one 64-bit add each; the second node of a
                // row is an offset of the load
                const uint32_t row = static_cast<uint32_t>(iy) + static_cast<uint32_t>(P.ny) * static_cast<uint32_t>(iz);
                const uint64_t node = static_cast<uint64_t>(row) * static_cast<uint32_t>(P.nx) + static_cast<uint32_t>(ix);
                const char* const p00 = reinterpret_cast<const char*>(P.fa_f32) + 16 * node;
                if (node != cell.node) {
                    cell.node = node;
                    if constexpr (!GEN) {
                        const bool last = ix == P.nx - 2 || iy == P.ny - 2 || iz == P.nz - 2;
                        cell.index = f3{last ? __builtin_nanf("") : static_cast<float>(ix), static_cast<float>(iy),
                                        static_cast<float>(iz)};
                    }
#pragma unroll
                    for (int c4 = 0; c4 < 4; ++c4) {
                        const float4* const q =
                            reinterpret_cast<const float4*>(p00 + 16 * ((c4 >> 1) * sy + (c4 & 1) * sz));
                        const float4 lo4 = q[0], hi4 = q[1];
                        cell.e[c4] = f3{lo4.x, lo4.y, lo4.z};
                        cell.e[4 + c4] = f3{hi4.x, hi4.y, hi4.z};
                    }
                }
            }
        }
        if (!GEN || P.n_terms <= 1) {
#pragma unroll
            for (int c8 = 0; c8 < 8; ++c8) {
                const int dx = c8 >> 2, dy = (c8 >> 1) & 1, dzz = c8 & 1;
                const float w = (dx ? ax : 1.0f - ax) * (dy ? ay : 1.0f - ay) * (dzz ? az : 1.0f - az);
                r.x += w * cell.e[c8].x;
                r.y += w * cell.e[c8].y;
                r.z += w * cell.e[c8].z;
            }
        } else {
            // the time factors in FP64 (phase never in FP32), applied in FP32
            const int nt = P.n_terms;
            const size_t base = ix + sy * iy + sz * iz;
            for (int j = 0; j < nt; ++j) {
                const float sj = (float)term_scale_f64(P, j, c);
                f3 e{0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int c8 = 0; c8 < 8; ++c8) {
                    const int dx = c8 >> 2, dy = (c8 >> 1) & 1, dzz = c8 & 1;
                    const float w = (dx ? ax : 1.0f - ax) * (dy ? ay : 1.0f - ay) * (dzz ? az : 1.0f - az);
                    const float4 v4 = P.fa_f32[(base + dx + dy * sy + dzz * sz) * nt + j];
                    e.x += w * v4.x;
                    e.y += w * v4.y;
                    e.z += w * v4.z;
                }
                r = r + e * sj;
            }
        }
        const float s = C.fa_scale;
        if (s != 1.0f) r = r * s;
        return r;
    }
}

// Domain containment in FP32 (same predicates as contains_f64; the FP32
// position is good to ~1e-7 relative, far finer than any domain feature).
template <bool MEM = kRecordsInMemory>
__device__ __forceinline__ bool contains_f32(const StepParams& P, const FastConst& C, float px,
                                             float py, float pz) {
    const f3 s{px - C.ox, py - C.oy, pz - C.oz};
    f3 l = s;
    if (!P.rot_identity) {
        keep_branch<MEM>();
        l = mat_mul(C.g2l, s);
    }
    const float r2 = fmaf(l.x, l.x, l.y * l.y);
    if (P.instrument == 3) {
        const float z_abs = fabsf(l.z);
        if (z_abs > C.half_L) return false;
        if (r2 > C.R_out_sq) return false;
        const float ln_r = 0.5f * fast_ln(r2);
        const float z2 = z_abs * z_abs;
        const float f_in = z2 - 0.5f * (r2 - C.R_in_sq) - C.R_char_sq * (C.ln_R_in - ln_r);
        const float f_out = z2 - 0.5f * (r2 - C.R_out * C.R_out) - C.R_char_sq * (C.ln_R_out - ln_r);
        return f_in >= 0.0f && f_out <= 0.0f;
    }
    return !(l.z < 0.0f) & !(l.z >= C.L) & (r2 <= C.R_eps_sq);
}

// 1 - exp(-x), small x by its series
__device__ __forceinline__ float collision_probability_f32(float x) {
    return x < 1e-3f ? x * fmaf(-0.5f * x, fmaf(x, -1.0f / 3.0f, 1.0f), 1.0f)
                     : 1.0f - __builtin_amdgcn_exp2f(-x * 1.44269504089f);
}

__device__ __forceinline__ f3 iso_dir_f32(PhiloxStream& rng) {
    const float u1 = rng.uniform_f32();
    const float u2 = rng.uniform_f32();
    const float cosT = 2.0f * u1 - 1.0f;
    const float sinT = fast_sqrt(fmaxf(0.0f, 1.0f - cosT * cosT));
    return f3{sinT * fast_cos_rev(u2), sinT * fast_sin_rev(u2), cosT};
}

// FLOW: the neutrals move with ug (the gas velocity at the ion's position),
// else with the constant gas velocity.  FIXED: the sums of the HSS collision after
// a push by this integrator with their rounding written out (the field-array
// kernels, single cloud and batch); -1: the compiler's choice.
template <int COLL, bool FLOW = false, int FIXED = -1>
__device__ __forceinline__ bool collide_f32(const StepParams& P, const FastConst& C,
                                            const SpeciesDev& sp, uint32_t sidx, float m,
                                            float inv_m_plus, float lpre, float kbt2_dt_over_m, f3& v,
                                            PhiloxStream& rng, float dt, float n_dt,
                                            f3 ug = f3{0.0f, 0.0f, 0.0f}) {
    const f3 u_gas = FLOW ? ug : f3{C.u_gas[0], C.u_gas[1], C.u_gas[2]};
    if constexpr (COLL == COLL_HSS_MIX) {
        {
            // the mixture path of collide_f64 in FP32 (rates, test and partner
            // choice as there; neutrals from two Box-Muller pairs)
            const double* sg = P.mix_sigma + static_cast<size_t>(sidx) * P.n_mix;
            f3 vn[kMaxGasComponents];
            float k[kMaxGasComponents];
            float k_total = 0.0f;
#pragma unroll
            for (int c = 0; c < kMaxGasComponents; ++c) {
                k[c] = -1.0f;
                vn[c] = f3{0.0f, 0.0f, 0.0f};
                if (c < P.n_mix) {
                    const float sn = (float)P.mix_sig[c];
                    const float u1 = rng.uniform_f32(), u2 = rng.uniform_f32();
                    const float u3 = rng.uniform_f32(), u4 = rng.uniform_f32();
                    const float r1 = sn * fast_sqrt(-2.0f * fast_ln(u1));
                    const float r2 = sn * fast_sqrt(-2.0f * fast_ln(u3));
                    vn[c] = f3{r1 * fast_cos_rev(u2) + u_gas.x, r1 * fast_sin_rev(u2) + u_gas.y,
                               r2 * fast_cos_rev(u4) + u_gas.z};
                    const f3 vr = v - vn[c];
                    const float vm = fast_sqrt(dot<float>(vr, vr));
                    if (vm >= (float)kMinRelativeVelocity) {
                        k[c] = (float)(P.mix_n[c] * sg[c]) * vm;
                        k_total += k[c];
                    }
                }
            }
            if (!(k_total > 0.0f)) return false;
            const float x = k_total * dt;
            const float Pc = x < 1e-3f ? x * (1.0f - 0.5f * x * (1.0f - x * (1.0f / 3.0f)))
                                       : (x <= 50.0f ? 1.0f - __builtin_amdgcn_exp2f(-x * 1.44269504089f) : 1.0f);
            if (rng.uniform_f32() >= Pc) return false;
            const float r = rng.uniform_f32() * k_total;
            int sel = -1, first = -1;
            float cum = 0.0f;
#pragma unroll
            for (int c = 0; c < kMaxGasComponents; ++c) {
                if (k[c] >= 0.0f) {
                    if (first < 0) first = c;
                    cum += k[c];
                    if (sel < 0 && r < cum) sel = c;
                }
            }
            if (sel < 0) sel = first;
            f3 vs{0.0f, 0.0f, 0.0f};
            float ms = 0.0f;
#pragma unroll
            for (int c = 0; c < kMaxGasComponents; ++c) {
                if (c == sel) {
                    vs = vn[c];
                    ms = (float)P.mix_m[c];
                }
            }
            const f3 vr = v - vs;
            const float vm = fast_sqrt(dot<float>(vr, vr));
            const f3 nd = iso_dir_f32(rng);
            const float inv_mt = 1.0f / (m + ms);
            const f3 Vcom = (v * m + vs * ms) * inv_mt;
            v = Vcom + nd * (vm * ms * inv_mt);
            return true;
        }
    } else if constexpr (COLL == COLL_HSS) {
        const float sigma = (float)sp.sigma_hss;
        if (!(sigma > 0.0f)) return false;
        // three Maxwellian components from two Box-Muller pairs (both branches)
        const float u1 = rng.uniform_f32(), u2 = rng.uniform_f32();
        const float u3 = rng.uniform_f32(), u4 = rng.uniform_f32();
        const float r1 = C.sigma_neutral * fast_sqrt(-2.0f * fast_ln(u1));
        const float r2 = C.sigma_neutral * fast_sqrt(-2.0f * fast_ln(u3));
        const f3 vn{r1 * fast_cos_rev(u2) + u_gas.x, r1 * fast_sin_rev(u2) + u_gas.y,
                    r2 * fast_cos_rev(u4) + u_gas.z};
        const f3 vrel = v - vn;
        const float vm = fast_sqrt(FIXED < 0 ? dot<float>(vrel, vrel) : speed2_f32<FIXED>(vrel));
        if (vm < (float)kMinRelativeVelocity) return false;
        const float Pc = collision_probability_f32(n_dt * sigma * vm);
        if (rng.uniform_f32() >= Pc) return false;
        const f3 nd = iso_dir_f32(rng);
        // centre of mass velocity + relative velocity times the neutral's share
        const f3 share = nd * (vm * C.m_gas * inv_m_plus);
        v = FIXED < 0 ? (v * m + vn * C.m_gas) * inv_m_plus + share
                      : fma3(fma3(vn, C.m_gas, v * m), inv_m_plus, share);
        return true;
    } else if constexpr (COLL == COLL_DAMPING) {
        if (P.ou_kicks) {
            const float g = (P.damping_model == 3) ? lpre / fmaxf(1e-6f, fast_sqrt(dot<float>(v, v))) : lpre;
            if (!(g > 0.0f)) return false;
            const float s = fast_sqrt(g * kbt2_dt_over_m);
            const float u1 = rng.uniform_f32(), u2 = rng.uniform_f32();
            const float u3 = rng.uniform_f32(), u4 = rng.uniform_f32();
            const float r1 = s * fast_sqrt(-2.0f * fast_ln(u1));
            const float r2 = s * fast_sqrt(-2.0f * fast_ln(u3));
            v.x += r1 * fast_cos_rev(u2);
            v.y += r1 * fast_sin_rev(u2);
            v.z += r2 * fast_cos_rev(u4);
        }
        return false;
    } else {
        return false;
    }
}

// gas_velocity_f64 in FP32: the constant gas velocity, or the AxialParabolic
// profile at p.
__device__ __forceinline__ f3 gas_velocity_f32(const StepParams& P, const FastConst& C, f3 p) {
    if (!P.flow_parabolic) return f3{C.u_gas[0], C.u_gas[1], C.u_gas[2]};
    float uz = C.flow_umax;
    if (C.flow_R2 > 0.0f) {
        const float dx = p.x - C.ox, dy = p.y - C.oy, dz = p.z - C.oz;
        const float lx = C.g2l[0] * dx + C.g2l[1] * dy + C.g2l[2] * dz;
        const float ly = C.g2l[3] * dx + C.g2l[4] * dy + C.g2l[5] * dz;
        uz = C.flow_umax * fmaxf(0.0f, 1.0f - (lx * lx + ly * ly) / C.flow_R2);
    }
    return f3{C.l2g[2] * uz, C.l2g[5] * uz, C.l2g[8] * uz};
}

// FLOW: the gas velocity at p (gas_velocity_f32), else the constant one.
template <int FIELD, int COLL, bool FLOW = false, class T>
__device__ __forceinline__ f3 accel_f32(const StepParams& P, const FastConst& C, f3 p, f3 v,
                                        T c, T ez, float qm, float lpre, CellF32& cell) {
    f3 a = field_f32<FIELD>(P, C, p, c, ez, cell) * qm;
    if constexpr (COLL == COLL_DAMPING) {
        const float g = (P.damping_model == 3) ? lpre / fmaxf(1e-6f, fast_sqrt(dot<float>(v, v))) : lpre;
        if (g > 0.0f) {
            const f3 u = FLOW ? gas_velocity_f32(P, C, p) : f3{C.u_gas[0], C.u_gas[1], C.u_gas[2]};
            a = a - f3{v.x - u.x, v.y - u.y, v.z - u.z} * g;
        }
    }
    return a;
}

template <int FIELD, int COLL, bool FLOW = false, class T>
__device__ __forceinline__ f3 accel_f32(const StepParams& P, const FastConst& C, f3 p, f3 v,
                                        T c, T ez, float qm, float lpre) {
    CellF32 cell;
    return accel_f32<FIELD, COLL, FLOW>(P, C, p, v, c, ez, qm, lpre, cell);
}

// RF coefficient (or time) and axial field of stage S (0 start, 1 middle, 2 end):
// FP64 for scaled field arrays (WIDE), rounded otherwise.
template <bool WIDE, int S>
__device__ __forceinline__ auto stage_c(const StepEntry& te) {
    if constexpr (WIDE) return S == 0 ? te.c0 : S == 1 ? te.ch : te.c1;
    else return S == 0 ? te.c0f : S == 1 ? te.chf : te.c1f;
}
template <bool WIDE, int S>
__device__ __forceinline__ auto stage_e(const StepEntry& te) {
    if constexpr (WIDE) return S == 0 ? te.e0 : S == 1 ? te.eh : te.e1;
    else return S == 0 ? te.e0f : S == 1 ? te.ehf : te.e1f;
}

// The stages of RK4 along x (two = -2) or y (two = 2) of an RF field E = two p c(t).
__device__ __forceinline__ void rk4_rf_axis(float p0, float v0, float two, const StepEntry& te, float qm, float dt,
                                            float half_dt, float& dpos, float& dvel) {
    const float k1a = two * p0 * te.c0f * qm;
    const float k2v = fmaf(k1a, half_dt, v0);
    const float k2a = two * fmaf(v0, half_dt, p0) * te.chf * qm;
    const float k3v = fmaf(k2a, half_dt, v0);
    const float k3a = two * fmaf(k2v, half_dt, p0) * te.chf * qm;
    const float k4v = fmaf(k3a, dt, v0);
    const float e4 = two * fmaf(k3v, dt, p0) * te.c1f;
    dpos = fmaf(k3v, 2.0f, fmaf(k2v, 2.0f, v0)) + k4v;
    dvel = fmaf(e4, qm, fmaf(k3a, 2.0f, fmaf(k2a, 2.0f, k1a)));
}

// One RK4 or Boris push of the FP32 path from (p0, v0).  The increments are
// returned as apply_push_f32 takes them, RK4's in units of h6 = dt / 6, Boris'
// position increment in units of dt.
template <int INTEG, int FIELD, int COLL, bool FLOW = false>
__device__ __forceinline__ void push_f32(const StepParams& P, const FastConst& C, const StepEntry& te, f3 p0, f3 v0,
                                         float qm, float lp, float dt, float half_dt, CellF32& cell, f3& dpos,
                                         f3& dvel) {
    constexpr bool X = FIELD == FIELD_ARRAY_X;
    if constexpr (INTEG == 0) {
        if constexpr (FIELD == FIELD_LINEAR && COLL != COLL_DAMPING) {
            // E = (-2 x c(t), 2 y c(t), E_z(t)): the stages below by component, z first
            const float az1 = te.e0f * qm, az2 = te.ehf * qm;
            const float k2z = fmaf(az1, half_dt, v0.z), k3z = fmaf(az2, half_dt, v0.z), k4z = fmaf(az2, dt, v0.z);
            f3 dp{0.0f, 0.0f, fmaf(k3z, 2.0f, fmaf(k2z, 2.0f, v0.z)) + k4z};
            f3 dv{0.0f, 0.0f, fmaf(te.e1f, qm, fmaf(az2, 2.0f, fmaf(az2, 2.0f, az1)))};
            if (P.has_rf) {
                rk4_rf_axis(p0.x, v0.x, -2.0f, te, qm, dt, half_dt, dp.x, dv.x);
                rk4_rf_axis(p0.y, v0.y, 2.0f, te, qm, dt, half_dt, dp.y, dv.y);
            } else {   // no acceleration in x and y
                dp.x = fmaf(v0.x, 2.0f, fmaf(v0.x, 2.0f, v0.x)) + v0.x;
                dp.y = fmaf(v0.y, 2.0f, fmaf(v0.y, 2.0f, v0.y)) + v0.y;
            }
            dpos = dp;
            dvel = dv;
            return;
        }
        const auto ch = stage_c<X, 1>(te), eh = stage_e<X, 1>(te), c1 = stage_c<X, 2>(te), e1 = stage_e<X, 2>(te);
        const f3 k1a = accel_f32<FIELD, COLL, FLOW>(P, C, p0, v0, stage_c<X, 0>(te), stage_e<X, 0>(te), qm, lp, cell);
        const f3 k2v = fma3(k1a, half_dt, v0);
        const f3 k2a = accel_f32<FIELD, COLL, FLOW>(P, C, fma3(v0, half_dt, p0), k2v, ch, eh, qm, lp, cell);
        const f3 k3v = fma3(k2a, half_dt, v0);
        const f3 k3a = accel_f32<FIELD, COLL, FLOW>(P, C, fma3(k2v, half_dt, p0), k3v, ch, eh, qm, lp, cell);
        const f3 k4v = fma3(k3a, dt, v0);
        const f3 p4 = fma3(k3v, dt, p0);
        const f3 a3 = fma3(k3a, 2.0f, fma3(k2a, 2.0f, k1a));
        f3 a4;
        // the last stage's field times q / m unrounded, without a damping force
        if constexpr (COLL == COLL_DAMPING)
            a4 = a3 + accel_f32<FIELD, COLL, FLOW>(P, C, p4, k4v, c1, e1, qm, lp, cell);
        else
            a4 = fma3(field_f32<FIELD>(P, C, p4, c1, e1, cell), qm, a3);
        dpos = fma3(k3v, 2.0f, fma3(k2v, 2.0f, v0)) + k4v;
        dvel = a4;
    } else {
        const f3 a = accel_f32<FIELD, COLL, FLOW>(P, C, p0, v0, stage_c<X, 0>(te), stage_e<X, 0>(te), qm, lp, cell);
        const f3 vm = fma3(a, half_dt, v0);
        f3 rot{0.0f, 0.0f, 0.0f};
        if (P.magnetic) {
            const f3 tv = f3{(float)P.B[0], (float)P.B[1], (float)P.B[2]} * (qm * half_dt);
            const float s_f = 2.0f / (1.0f + dot(tv, tv));
            const f3 vprime = vm + cross(vm, tv);
            rot = cross(vprime, tv * s_f);
        }
        // x += v+ dt, v = v+ + a dt/2 = v0 + a dt + rot (no cancellation)
        dpos = vm + rot;
        dvel = fma3(a, dt, rot);
    }
}

template <int INTEG>
__device__ __forceinline__ void apply_push_f32(float hi[6], float lo[6], f3 dpos, f3 dvel, float dt, float h6) {
    const float s = INTEG == 0 ? h6 : dt;
    kahan_fma(hi[0], lo[0], dpos.x, s);
    kahan_fma(hi[1], lo[1], dpos.y, s);
    kahan_fma(hi[2], lo[2], dpos.z, s);
    if constexpr (INTEG == 0) {
        kahan_fma(hi[3], lo[3], dvel.x, s);
        kahan_fma(hi[4], lo[4], dvel.y, s);
        kahan_fma(hi[5], lo[5], dvel.z, s);
    } else {
        kahan_add(hi[3], lo[3], dvel.x);
        kahan_add(hi[4], lo[4], dvel.y);
        kahan_add(hi[5], lo[5], dvel.z);
    }
}

}  // namespace icarion
