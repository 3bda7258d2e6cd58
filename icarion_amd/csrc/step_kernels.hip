// step_kernels.hip - fused multi-step ion kernels for gfx950.
//
// One ion per lane (four lanes in FP64 for small clouds, a wavefront's lanes
// together through geometry EHSS).  A lane loads its ion once (coalesced SoA), runs
// params.n_steps engine steps with the state in registers, and stores it
// once; per step it does what the reference engine does to one ion:
//   prepare  (SimulationEngineLifecycle.cpp:86-107): birth, domain lookup;
//   push     (RK4Strategy.cpp:181-361 or BorisStrategy.cpp:18-98);
//   collide  (HSS: HSSCollisionHandler.cpp:257-376, EHSS:
//             EHSSCollisionHandler.cpp:222-455, OU kick: CollisionKernels.cpp:171-214);
//   finalize (SimulationEngineLifecycle.cpp:137-192): boundary elimination with
//             death at the step-start time, NaN kill.
// Ions never interact, so running these phases back to back per ion gives
// the reference's per-ion result.  Per-step wave-uniform values (engine time,
// RF coefficient) come from a table read with scalar loads.  Counters are
// reduced per wavefront before one atomic per wave.
#include "launch_rules.hpp"
#include "step_device.hpp"
#include "step_device_f32.hpp"
#include "surrogate.hpp"

namespace icarion {

// An index whose addresses are formed where it is used: hoisted out of the step
// loop, the addresses of rare events take registers all along.
__device__ __forceinline__ uint32_t here(uint32_t i) {
    asm volatile("" : "+v"(i));
    return i;
}

// The per-ion factor of the damping coefficient (DampingForce.cpp:150-177 / :269-271).
__device__ __forceinline__ double damping_factor_f64(const StepParams& P, const SpeciesDev& sp, double m, double q) {
    if (P.damping_model == 3) {
        if (P.alpha_gas > 0.0 && P.n > 0.0 && P.v_th > 0.0 && P.m_gas > 0.0) {
            const double mu = (m * P.m_gas) / (m + P.m_gas);
            const double cs1 = kPi * q * sqrt(P.alpha_gas / (4.0 * kPi * kEpsilon0 * mu));
            return P.n * cs1 * P.v_th * P.m_gas / (P.m_gas + m);
        }
    } else {
        const double K0 = sp.K0_cm2_Vs;
        if (K0 > 0.0 && m > 0.0 && P.n > 0.0) {
            const double K0t = K0 * 1e-4 * sqrt(kStpTemp / fmax(P.T, 1.0));
            return q / ((K0t * (kLoschmidt / P.n)) * m);
        }
    }
    return 0.0;
}

// SUB: collision substeps; FLOW: the AxialParabolic gas flow (both read from P
// at run time, instantiated apart because they cost the plain kernels
// registers).
template <int INTEG, int FIELD, int COLL, bool SUB = false, bool FLOW = false>
__device__ __forceinline__ void f64_ion(const StepParams& P, const IonPtrs& S, const uint32_t i,
        uint32_t& pushed, uint32_t& ncoll_launch) {
    d3 pos{S.x[i], S.y[i], S.z[i]};
    d3 vel{S.vx[i], S.vy[i], S.vz[i]};
    const double m = S.mass[i];
    const double q = S.charge[i];
    const uint32_t sidx = S.species[i];
    const SpeciesDev sp = P.species[sidx];
    uint8_t flags = S.flags[i];
    bool active = flags & 1, born = (flags >> 1) & 1;
    const double birth = S.birth ? S.birth[i] : -INFINITY;
    double death = S.death[i];
    double arrival = S.arrival[i];
    uint32_t nc = S.ncoll[i];
    const double inv_m = 1.0 / m;
    double lpre = 0.0;
    if constexpr (COLL == COLL_DAMPING) lpre = damping_factor_f64(P, sp, m, q);
    // 0: done, 1: stepping, 2: unborn, 3: stepping, position not yet known to
    // be inside (see f32_ion: the loop is wave-uniform, its body masked)
    uint32_t state = !born ? 2u : active ? 3u : 0u;
    const double dt = P.dt;
    const double half_dt = dt * 0.5;
    for (uint32_t k = 0; k < P.n_steps; ++k) {
        if (__ballot(state != 0u) == 0ull) break;
        const StepEntry& te = P.table[k];
        const double t = te.t;
        if (__ballot(state > 1u) != 0ull) {   // before an ion's first step only
            if (state == 2u && t >= birth) {
                born = true;
                state = 3u;
            }
            if (state == 3u) {
                state = 1u;
                if (!contains_f64<FIELD == FIELD_ARRAY_X>(P, pos)) {
                    state = 0u;
                    death = t;
                }
            }
        }
        if (state != 1u) continue;
        const double z_before = pos.z;
        // the step's gas density (update_dynamic_environments at the step
        // start, SimulationEngine.cpp:380): the damping coefficient and the
        // collision rates scale with it
        const double lp = lpre * te.nrel;
        if constexpr (INTEG == 0) {
            // RK4Strategy::step_batch_with_stage_refresh (RK4Strategy.cpp:181-361)
            const d3 p0 = pos, v0 = vel;
            const d3 k1v = v0;
            const d3 k1a = force_f64<FIELD, COLL, FLOW>(P, p0, v0, te.c0, te.e0, q, m, lp) * inv_m;
            const d3 k2v = v0 + k1a * half_dt;
            const d3 k2a = force_f64<FIELD, COLL, FLOW>(P, p0 + k1v * half_dt, k2v, te.ch, te.eh, q, m, lp) * inv_m;
            const d3 k3v = v0 + k2a * half_dt;
            const d3 k3a = force_f64<FIELD, COLL, FLOW>(P, p0 + k2v * half_dt, k3v, te.ch, te.eh, q, m, lp) * inv_m;
            const d3 k4v = v0 + k3a * dt;
            const d3 k4a = force_f64<FIELD, COLL, FLOW>(P, p0 + k3v * dt, k4v, te.c1, te.e1, q, m, lp) * inv_m;
            const double h6 = dt / 6.0;
            pos = p0 + (k1v + k2v * 2.0 + k3v * 2.0 + k4v) * h6;
            vel = v0 + (k1a + k2a * 2.0 + k3a * 2.0 + k4a) * h6;
        } else {
            // BorisStrategy::step (BorisStrategy.cpp:18-98)
            const d3 a = force_f64<FIELD, COLL, FLOW>(P, pos, vel, te.c0, te.e0, q, m, lp) * inv_m;
            const d3 vm = vel + a * half_dt;
            d3 vp = vm;
            if (P.magnetic) {
                const double qm = q * inv_m;
                const d3 tv = d3{P.B[0], P.B[1], P.B[2]} * (qm * dt * 0.5);
                const double s_f = 2.0 / (1.0 + dot(tv, tv));
                const d3 sv = tv * s_f;
                const d3 vprime = vm + cross(vm, tv);
                vp = vm + cross(vprime, sv);
            }
            pos = pos + vp * dt;
            vel = vp + a * half_dt;
        }
        ++pushed;
        if constexpr (COLL != COLL_NONE) {
            PhiloxStream rng(P.seed, i, P.step0 + k);
            // collision substeps, each an event of its own, in the SUB
            // instantiation (the loop costs the one-stage kernels registers)
            const int ns = SUB ? P.n_sub : 1;
            const double dtc = SUB ? dt / static_cast<double>(P.n_sub) : dt;
            // a rate n sigma |v| dt takes the density ratio through dt; the OU
            // kick's variance 2 gamma kT dt / m through gamma alone
            const double dtn = COLL == COLL_DAMPING ? dtc : dtc * te.nrel;
            // the gas velocity at the pushed position, for every substep
            // (SimulationEngineCollisionRuntime.cpp:122-130)
            const d3 ug = FLOW ? gas_velocity_f64(P, pos) : d3{0.0, 0.0, 0.0};
            for (int s = 0; s < ns; ++s) {
                if (collide_f64<COLL, FLOW>(P, sp, sidx, m, lp, vel, rng, dtn, ug)) {
                    ++nc;
                    ++ncoll_launch;
                }
            }
        }
        if (P.detect) {
            keep_branch<FIELD == FIELD_ARRAY_X>();
            if (isnan(arrival) && z_before < P.det_z && pos.z >= P.det_z)
                arrival = t + dt * (P.det_z - z_before) / (pos.z - z_before);
        }
        if (!(contains_f64<FIELD == FIELD_ARRAY_X>(P, pos) & isfinite(pos.x) & isfinite(pos.y) & isfinite(pos.z) & isfinite(vel.x) &
              isfinite(vel.y) & isfinite(vel.z))) {
            state = 0u;
            death = t;
        }
    }
    if (state != 2u) active = state != 0u;
    S.x[i] = pos.x; S.y[i] = pos.y; S.z[i] = pos.z;
    S.vx[i] = vel.x; S.vy[i] = vel.y; S.vz[i] = vel.z;
    S.flags[i] = static_cast<uint8_t>((active ? 1 : 0) | (born ? 2 : 0));
    S.death[i] = death;
    S.arrival[i] = arrival;
    S.ncoll[i] = nc;
}

// Two wavefronts per SIMD where the compiler would take registers for one: Boris in
// general field arrays (256 and up to 30 spilled; with 282 registers 300,000 ions x
// 60 HSS steps took 1.89 ms, now 1.38 ms), EHSS with offline sets and over mixtures
// in linear fields (256 and up to 12 spilled; 150,000 ions x 40 steps, offline sets
// for one of three species 5.64 ms, now 4.24 ms).
template <int INTEG, int FIELD, int COLL, bool SUB = false>
__global__ void __launch_bounds__(256, (FIELD == FIELD_LINEAR && (COLL == COLL_EHSS_TAB || COLL == COLL_EHSS_MIX)) ||
                                       (INTEG == 1 && FIELD == FIELD_ARRAY_X) ? 2 : 1)
    step_f64_kernel(const StepParams P, const IonPtrs S) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t pushed = 0, ncoll_launch = 0;
    if (i < P.n_ions) f64_ion<INTEG, FIELD, COLL, SUB, SUB>(P, S, P.order ? P.order[i] : i, pushed, ncoll_launch);
    add_counters(P, pushed, ncoll_launch);
}

// ======================= FP64, four lanes per ion ============================
//
// The step of f64_ion for the analytic linear fields (no magnetic field) with
// one ion on four lanes: lanes 0-2 hold the x, y and z components.  Lane 3 starts
// as z and serves the draws alone: after a collision its position and velocity
// mean nothing, and nothing reads them.  The draws of a step are four or five Philox blocks, three or four
// Box-Muller transforms and a direction: lane c takes block c, so one block, one
// logarithm, one sine and cosine per lane replace them (lane 3 draws the
// collision test and the direction).  Scalars of an ion (speeds, tests) are
// formed on all four lanes from broadcast components, in f64_ion's order of
// operations: the results agree with it to rounding.
// A wavefront's step is a third of f64_ion's instructions for a quarter of the
// ions, and a cloud that does not fill the chip is bound by exactly that chain
// (10,000 ions x 5000 HSS steps: 19.4 ms with f64_ion and the general sine,
// cosine and logarithm, 7.6 ms here; 30,000 x 1000: 4.5 and 2.7 ms).  From three
// wavefronts per SIMD on the lanes repeated by an ion cost what the chain gains:
// 65,000 ions x 1000 steps took 4.6 ms here and 4.9 ms before both.
constexpr uint32_t kQuadMaxIons = 49152;

// Component K (0-3) of the ion's four lanes, on each of them.
template <int K>
__device__ __forceinline__ double quad_f64(double x) {
    const int lo = __double2loint(x), hi = __double2hiint(x);
    return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, K * 0x55, 0xf, 0xf, false),
                            __builtin_amdgcn_update_dpp(lo, lo, K * 0x55, 0xf, 0xf, false));
}
__device__ __forceinline__ d3 quad_d3(double x) { return d3{quad_f64<0>(x), quad_f64<1>(x), quad_f64<2>(x)}; }

template <int INTEG, int COLL>
__global__ void __launch_bounds__(256) step_f64_quad_kernel(const StepParams P, const IonPtrs S) {
    const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t c = tid & 3u;
    const bool valid = (tid >> 2) < P.n_ions;
    const uint32_t i = valid ? tid >> 2 : 0u;
    const int comp = c < 2u ? static_cast<int>(c) : 2;
    double* const px = comp == 0 ? S.x : comp == 1 ? S.y : S.z;
    double* const pv = comp == 0 ? S.vx : comp == 1 ? S.vy : S.vz;
    double p = px[i], v = pv[i];
    const double m = S.mass[i], q = S.charge[i];
    const uint32_t sidx = S.species[i];
    const SpeciesDev sp = P.species[sidx];
    const uint8_t flags = S.flags[i];
    bool active = flags & 1, born = (flags >> 1) & 1;
    const double birth = S.birth ? S.birth[i] : -INFINITY;
    double death = S.death[i], arrival = S.arrival[i];
    uint32_t nc = S.ncoll[i];
    const double inv_m = 1.0 / m;
    double lpre = 0.0;
    if constexpr (COLL == COLL_DAMPING) lpre = damping_factor_f64(P, sp, m, q);
    const double rf_sign = comp == 0 ? -2.0 : 2.0;
    const double u_gas = comp == 0 ? P.u_gas[0] : comp == 1 ? P.u_gas[1] : P.u_gas[2];
    const double inv_mt = 1.0 / (m + P.m_gas);
    uint32_t pushed = 0, ncoll_launch = 0;
    uint32_t state = !valid ? 0u : !born ? 2u : active ? 3u : 0u;   // as in f64_ion, alike on the ion's lanes
    const double dt = P.dt;
    const double half_dt = dt * 0.5;
    for (uint32_t k = 0; k < P.n_steps; ++k) {
        if (__ballot(state != 0u) == 0ull) break;
        const StepEntry& te = P.table[k];
        const double t = te.t;
        if (__ballot(state > 1u) != 0ull) {   // before an ion's first step only
            if (state == 2u && t >= birth) {
                born = true;
                state = 3u;
            }
            const bool in = contains_f64(P, quad_d3(p));
            if (state == 3u) {
                state = in ? 1u : 0u;
                if (!in) death = t;
            }
        }
        if (state != 1u) continue;
        const double p_before = p;
        const double lp = lpre * te.nrel;
        // this lane's component of force / mass at (pc, vc)
        auto accel = [&](double pc, double vc, double c_rf, double ez) {
            double E = comp == 2 ? ez : 0.0;
            if (P.has_rf && comp != 2) E = rf_sign * pc * c_rf;
            double F = E * q;
            if constexpr (COLL == COLL_DAMPING) {
                const double g = gamma_f64(P, lp, quad_d3(vc));
                if (g > 0.0) F = F + (vc - u_gas) * (-g * m);
            }
            return F * inv_m;
        };
        if constexpr (INTEG == 0) {
            const double k1a = accel(p, v, te.c0, te.e0);
            const double k2v = v + k1a * half_dt;
            const double k2a = accel(p + v * half_dt, k2v, te.ch, te.eh);
            const double k3v = v + k2a * half_dt;
            const double k3a = accel(p + k2v * half_dt, k3v, te.ch, te.eh);
            const double k4v = v + k3a * dt;
            const double k4a = accel(p + k3v * dt, k4v, te.c1, te.e1);
            const double h6 = dt / 6.0;
            p = p + (v + k2v * 2.0 + k3v * 2.0 + k4v) * h6;
            v = v + (k1a + k2a * 2.0 + k3a * 2.0 + k4a) * h6;
        } else {
            const double a = accel(p, v, te.c0, te.e0);
            const double vm = v + a * half_dt;
            p = p + vm * dt;
            v = vm + a * half_dt;
        }
        ++pushed;
        if constexpr (COLL == COLL_HSS) {
            if (sp.sigma_hss > 0.0) {
                const uint32_t s_lo = static_cast<uint32_t>(P.step0 + k), s_hi = static_cast<uint32_t>((P.step0 + k) >> 32);
                const uint32_t k0 = static_cast<uint32_t>(P.seed), k1 = static_cast<uint32_t>(P.seed >> 32);
                // draws 2 c and 2 c + 1 on lane c; draw 8 (the direction's angle) on all
                const u32x4 o = philox4x32_10(c, i, s_lo, s_hi, k0, k1);
                const u32x4 o4 = philox4x32_10(4u, i, s_lo, s_hi, k0, k1);
                const double ua = uniform53(o.v[0], o.v[1]), ub = uniform53(o.v[2], o.v[3]);
                double sn, cs;
                sincos_rev(c == 3u ? uniform53(o4.v[0], o4.v[1]) : ub, sn, cs);
                const double vn = P.sigma_neutral * (sqrt(-2.0 * log_unit(ua)) * cs) + u_gas;
                const double vm = speed_f64(quad_d3(v - vn));
                const double Pc = 1.0 - exp(-P.n * sp.sigma_hss * vm * (dt * te.nrel));
                // lane 3's draws, on every lane (before any lane-dependent choice:
                // a broadcast reads its source lane only while that is active)
                const double u_test = quad_f64<3>(ua), u_dir = quad_f64<3>(ub);
                const double sn3 = quad_f64<3>(sn), cs3 = quad_f64<3>(cs);
                // vm below kMinRelativeVelocity: no collision (above it hss_collision's
                // smaller bound never applies)
                if (vm >= kMinRelativeVelocity && u_test < Pc) {
                    const double cosT = 2.0 * u_dir - 1.0;
                    const double sinT = sqrt(fmax(0.0, 1.0 - cosT * cosT));
                    const double nd = comp == 2 ? cosT : sinT * (comp == 0 ? cs3 : sn3);
                    v = hss_velocity_f64(v, m, vn, P.m_gas, inv_mt, nd, vm, P.m_gas * inv_mt);
                    ++nc;
                    ++ncoll_launch;
                }
            }
        } else if constexpr (COLL == COLL_DAMPING) {
            if (P.ou_kicks) {
                const double g = gamma_f64(P, lp, quad_d3(v));
                if (g > 0.0 && dt > 0.0) {
                    // draws 0, 1 for x (cosine) and y (sine), 2, 3 for z (cosine)
                    const u32x4 o = philox4x32_10(c >> 1, i, static_cast<uint32_t>(P.step0 + k),
                                                  static_cast<uint32_t>((P.step0 + k) >> 32),
                                                  static_cast<uint32_t>(P.seed), static_cast<uint32_t>(P.seed >> 32));
                    double sn, cs;
                    sincos_rev(uniform53(o.v[2], o.v[3]), sn, cs);
                    const double r = sqrt(-2.0 * log_unit(uniform53(o.v[0], o.v[1])));
                    const double kBT_over_m = kBoltzmann * P.T / m;
                    const double s = sqrt(2.0 * g * kBT_over_m * dt);
                    v += s * (r * (comp == 1 ? sn : cs));
                }
            }
        }
        if (P.detect) {
            keep_branch();
            const double zb = quad_f64<2>(p_before), za = quad_f64<2>(p);
            if (isnan(arrival) && zb < P.det_z && za >= P.det_z) arrival = t + dt * (P.det_z - zb) / (za - zb);
        }
        const d3 pos = quad_d3(p), vel = quad_d3(v);
        if (!(contains_f64(P, pos) & isfinite(pos.x) & isfinite(pos.y) & isfinite(pos.z) & isfinite(vel.x) &
              isfinite(vel.y) & isfinite(vel.z))) {
            state = 0u;
            death = t;
        }
    }
    if (state != 2u) active = state != 0u;
    if (valid) {
        if (c < 3u) {
            px[i] = p;
            pv[i] = v;
        } else {
            S.flags[i] = static_cast<uint8_t>((active ? 1 : 0) | (born ? 2 : 0));
            S.death[i] = death;
            S.arrival[i] = arrival;
            S.ncoll[i] = nc;
        }
    }
    add_counters(P, c == 3u ? pushed : 0u, c == 3u ? ncoll_launch : 0u);
}

// ======================= FP64 geometry EHSS, wave-cooperative ===============
//
// The plain EHSS method of ehss_f64 / ehss_core_f64 with a collision's atoms
// spread over the wavefront and everything else done by all lanes at once.
// A wavefront owns P.ions_per_wave ions (lanes below that number).  Per step:
//   * every owner lane pushes its ion and runs its collision test (the
//     handler's Maxwellian neutral, P = 1 - exp(-n sigma_eff |v_rel| dt)), and
//     forms its random orientation, all lanes together;
//   * the first impact parameters of every ion are drawn by all lanes together
//     too: the stream is counter-based (attempt a is Philox block 5 + a), so
//     lane g * ions_per_wave + l draws attempt g of ion l;
//   * then the colliding ions one after another: the orientation goes to
//     scalar registers, atom j of the cluster is handled by lane j mod 64.
//     The method's geometry is taken in the collision frame, in which the
//     relative velocity is the z axis and the rotation is the orientation
//     alone: b_max is a wave max over the atoms' extents about the axis; for
//     each impact parameter the first contact is a wave min over (s_hit, atom
//     index), the sequential loop's choice (CollisionKernels.cpp:283-381);
//   * the contact normals of all ions are turned to the global frame and the
//     velocities reflected by all lanes together.
// What bounds it: FP64 issue in the atom loops and the chain of one collision.
// Done once per collision, the orientation, the draws and the reflection were
// two thirds of the instructions; a row of atoms was waited for at a time; and
// 64 ions on every wavefront left SIMDs idle below 131,072 ions
// (ehss_ions_per_wave).  Two wavefronts per SIMD hide the chain: birth, death and
// arrival times stay in memory until their event and the table entry is read where
// it is used, which leaves 256 registers and 4 spilled ones (with all of them in
// registers 282, and one wavefront).  First, with one wavefront, and now:
// 701 ions x 200 steps 56.0, 1.4 and 1.4 ms, 9001 x 200 59.6, 6.2 and 4.5 ms,
// 40,000 x 100 33.3, 11.4 and 6.9 ms, 250,000 x 40 33.3, 25.2 and 16.2 ms.

__device__ __forceinline__ uint32_t readlane_u32(uint32_t x, int lane) {
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(x), lane));
}

__device__ __forceinline__ double readlane_f64(double x, int lane) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(x), lane);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(x), lane);
    return __hiloint2double(hi, lo);
}

// x moved between lanes by a DPP control; lanes without a source keep x.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_f64(double x) {
    const int lo = __double2loint(x), hi = __double2hiint(x);
    return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xf, false),
                            __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xf, false));
}

// The maximum / minimum over the wavefront (all 64 lanes active), wave-uniform:
// row shifts within 16 lanes, then row broadcasts, read from lane 63.
template <class Op>
__device__ __forceinline__ double wave_reduce_f64(double v, Op&& op) {
    v = op(v, dpp_f64<0x111, 0xf>(v));
    v = op(v, dpp_f64<0x112, 0xf>(v));
    v = op(v, dpp_f64<0x114, 0xf>(v));
    v = op(v, dpp_f64<0x118, 0xf>(v));
    v = op(v, dpp_f64<0x142, 0xa>(v));
    v = op(v, dpp_f64<0x143, 0xc>(v));
    return readlane_f64(v, 63);
}

// Rotated atoms of the collision in progress, per wavefront: the first
// kWaveAtoms atoms of a cluster, (x, y) and (z, (r_atom + r_gas)^2) in the
// collision frame, each written and read by its own lane; atoms past that are
// rotated again from the table on every impact parameter.
constexpr int kWaveRows = 8;
constexpr uint32_t kWaveAtoms = 64 * kWaveRows;
struct WaveAtoms {
    double2 xy[kWaveAtoms];
    double2 zr[kWaveAtoms];
};

// Impact parameters of an ion drawn ahead, in units of b_max, per pass over the
// lanes (64 / ions_per_wave attempts each).
constexpr int kAheadPasses = 3;

// The draws of the step's streams by block number: pair(b, ion) is draws 2 b and
// 2 b + 1 of the ion's stream (0-5 the neutral, 6 the test, 7-9 the orientation,
// 10 + 2 a and 11 + 2 a impact parameter a).
struct EhssDraws {
    uint32_t k0, k1, s_lo, s_hi;
    __device__ __forceinline__ EhssDraws(uint64_t seed, uint64_t step)
        : k0(static_cast<uint32_t>(seed)), k1(static_cast<uint32_t>(seed >> 32)), s_lo(static_cast<uint32_t>(step)),
          s_hi(static_cast<uint32_t>(step >> 32)) {
        // the round keys as scalar adds in each use (see PhiloxStream::refill)
        k0 = __builtin_amdgcn_readfirstlane(k0);
        k1 = __builtin_amdgcn_readfirstlane(k1);
        asm("" : "+s"(k0), "+s"(k1) : "s"(__builtin_amdgcn_readfirstlane(s_lo)));
    }
    __device__ __forceinline__ void pair(uint32_t block, uint32_t ion, double& u1, double& u2) const {
        const u32x4 o = philox4x32_10(block, ion, s_lo, s_hi, k0, k1);
        u1 = uniform53(o.v[0], o.v[1]);
        u2 = uniform53(o.v[2], o.v[3]);
    }
    // the impact point of one attempt over b_max: sqrt(u1) (cos 2 pi u2, sin 2 pi u2)
    __device__ __forceinline__ void impact(uint32_t attempt, uint32_t ion, double& ux, double& uy) const {
        double u1, u2, sn, cs;
        pair(5u + attempt, ion, u1, u2);
        const double b = sqrt(u1);
        sincos_rev(u2, sn, cs);
        ux = b * cs;
        uy = b * sn;
    }
};

template <int INTEG, int FIELD>
__global__ void __launch_bounds__(256, ehss_waves_per_simd(INTEG, FIELD == FIELD_ARRAY, FIELD == FIELD_ARRAY_X))
    step_f64_ehss_kernel(const StepParams P, const IonPtrs S) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t G = P.ions_per_wave;
    const uint32_t first = (blockIdx.x * (blockDim.x >> 6) + wave) * G;
    const uint32_t ahead = lane / G, owner = lane - ahead * G;   // the attempt and ion this lane draws for
    const uint32_t reps = 64u / G;                               // attempts drawn per pass
    const uint32_t passes = reps >= 3u ? 1u : reps == 2u ? 2u : 3u;
    const uint32_t i = first + lane;
    const bool have = lane < G && i < P.n_ions;
    d3 pos{0.0, 0.0, 0.0}, vel{0.0, 0.0, 0.0};
    double m = 1.0, q = 0.0;
    uint32_t sidx = 0, nc = 0;
    bool active = false, born = true;
    if (have) {
        pos = d3{S.x[i], S.y[i], S.z[i]};
        vel = d3{S.vx[i], S.vy[i], S.vz[i]};
        m = S.mass[i];
        q = S.charge[i];
        sidx = S.species[i];
        const uint8_t flags = S.flags[i];
        active = flags & 1;
        born = (flags >> 1) & 1;
        nc = S.ncoll[i];
    }
    const SpeciesDev sp = P.species[sidx];
    const double inv_m = 1.0 / m;
    uint32_t pushed = 0, ncoll_launch = 0;
    bool checked = false;
    const double dt = P.dt;
    const double half_dt = dt * 0.5;
    __shared__ WaveAtoms s_atoms[4];   // 256 threads = 4 wavefronts
    WaveAtoms& lds = s_atoms[threadIdx.x >> 6];
    for (uint32_t k = 0; k < P.n_steps; ++k) {
        // unborn ions wait for their birth, live ones step; none left: the
        // whole wavefront leaves together
        if (__ballot(have && (!born || active)) == 0ull) break;
        const StepEntry& te = P.table[k];
        const double t = te.t;
        bool live = false;
        if (have) {
            if (!born && (!S.birth || t >= S.birth[here(i)])) {
                born = true;
                active = true;
                checked = false;
            }
            if (born && active) {
                if (!checked && !contains_f64(P, pos)) {
                    active = false;
                    S.death[here(i)] = t;
                } else {
                    live = true;
                }
            }
        }
        const double z_before = pos.z;
        if (live) {
            if constexpr (INTEG == 0) {
                const d3 p0 = pos, v0 = vel;
                const d3 k1v = v0;
                const d3 k1a = force_f64<FIELD, COLL_EHSS>(P, p0, v0, te.c0, te.e0, q, m, 0.0) * inv_m;
                const d3 k2v = v0 + k1a * half_dt;
                const d3 k2a = force_f64<FIELD, COLL_EHSS>(P, p0 + k1v * half_dt, k2v, te.ch, te.eh, q, m, 0.0) * inv_m;
                const d3 k3v = v0 + k2a * half_dt;
                const d3 k3a = force_f64<FIELD, COLL_EHSS>(P, p0 + k2v * half_dt, k3v, te.ch, te.eh, q, m, 0.0) * inv_m;
                const d3 k4v = v0 + k3a * dt;
                const d3 k4a = force_f64<FIELD, COLL_EHSS>(P, p0 + k3v * dt, k4v, te.c1, te.e1, q, m, 0.0) * inv_m;
                const double h6 = dt / 6.0;
                pos = p0 + (k1v + k2v * 2.0 + k3v * 2.0 + k4v) * h6;
                vel = v0 + (k1a + k2a * 2.0 + k3a * 2.0 + k4a) * h6;
            } else {
                const d3 a = force_f64<FIELD, COLL_EHSS>(P, pos, vel, te.c0, te.e0, q, m, 0.0) * inv_m;
                const d3 vm = vel + a * half_dt;
                d3 vp = vm;
                if (P.magnetic) {
                    const double qm = q * inv_m;
                    const d3 tv = d3{P.B[0], P.B[1], P.B[2]} * (qm * dt * 0.5);
                    const double s_f = 2.0 / (1.0 + dot(tv, tv));
                    const d3 sv = tv * s_f;
                    const d3 vprime = vm + cross(vm, tv);
                    vp = vm + cross(vprime, sv);
                }
                pos = pos + vp * dt;
                vel = vp + a * half_dt;
            }
            ++pushed;
        }
        // the collision test of each lane (collide_f64<COLL_EHSS> up to the
        // geometry method)
        const EhssDraws rng(P.seed, P.step0 + k);
        bool hit = false;
        d3 vn{0.0, 0.0, 0.0}, vrel{0.0, 0.0, 0.0};
        double vrel_mag = 1.0, u_first = 0.0;   // u_first: the orientation's first draw
        if (live && sp.sigma_ehss > 0.0) {
            double u1, u2;
            rng.pair(0u, i, u1, u2);
            vn.x = P.sigma_neutral * normal_of(u1, u2);
            rng.pair(1u, i, u1, u2);
            vn.y = P.sigma_neutral * normal_of(u1, u2);
            rng.pair(2u, i, u1, u2);
            vn.z = P.sigma_neutral * normal_of(u1, u2);
            vn = vn + d3{P.u_gas[0], P.u_gas[1], P.u_gas[2]};
            vrel = vel - vn;
            vrel_mag = sqrt(dot(vrel, vrel));
            if (vrel_mag >= kMinRelativeVelocity) {
                const double Pc = 1.0 - exp(-P.n * sp.sigma_ehss * vrel_mag * (dt * te.nrel));
                rng.pair(3u, i, u1, u_first);
                hit = u1 < Pc;
            }
        }
        uint64_t pending = __ballot(hit);
        if (pending) {
            // the random orientation (CollisionGeometry::generate_random_rotation)
            double O[9];
            {
                const double u1 = u_first;
                double u2, u3;
                rng.pair(4u, i, u2, u3);
                double s2, c2, s3, c3;
                sincos_rev(u2, s2, c2);
                sincos_rev(u3, s3, c3);
                const double x = sqrt(1.0 - u1) * s2;
                const double y = sqrt(1.0 - u1) * c2;
                const double z = sqrt(u1) * s3;
                const double w = sqrt(u1) * c3;
                O[0] = 1 - 2 * (y * y + z * z); O[1] = 2 * (x * y - z * w);     O[2] = 2 * (x * z + y * w);
                O[3] = 2 * (x * y + z * w);     O[4] = 1 - 2 * (x * x + z * z); O[5] = 2 * (y * z - x * w);
                O[6] = 2 * (x * z - y * w);     O[7] = 2 * (y * z + x * w);     O[8] = 1 - 2 * (x * x + y * y);
            }
            // the first impact points: pass p draws attempts p * reps .. + reps - 1
            double ux[kAheadPasses], uy[kAheadPasses];
#pragma unroll
            for (int p = 0; p < kAheadPasses; ++p) {
                ux[p] = uy[p] = 0.0;
                if (static_cast<uint32_t>(p) < passes) rng.impact(p * reps + ahead, first + owner, ux[p], uy[p]);
            }
            bool contact = false;
            double nx = 0.0, ny = 0.0, nz = 1.0;   // the contact point about the atom, collision frame
            // The cluster of the first colliding ion; each later one is loaded
            // while the impact parameters of the ion before it are tried.  Rows of
            // 64 atoms; lanes past the last atom read it again.
            float4 row[kWaveRows];
            auto fetch = [&](int L) {
                const uint32_t nat = readlane_u32(sp.atom_count, L);
                const float4* __restrict__ atoms = P.atoms + readlane_u32(sp.atom_offset, L);
#pragma unroll
                for (int r = 0; r < kWaveRows; ++r)
                    if (64u * r < nat) row[r] = atoms[min(lane + 64u * r, nat - 1u)];
            };
            fetch(__builtin_amdgcn_readfirstlane(static_cast<int>(__builtin_ctzll(pending))));
            while (pending) {
                const int L = __builtin_amdgcn_readfirstlane(static_cast<int>(__builtin_ctzll(pending)));
                pending &= pending - 1ull;
                const uint32_t nat = readlane_u32(sp.atom_count, L);
                const float4* __restrict__ atoms = P.atoms + readlane_u32(sp.atom_offset, L);
                double Q[9];
#pragma unroll
                for (int c = 0; c < 9; ++c) Q[c] = readlane_f64(O[c], L);
                const double r_gas = P.r_gas;
                auto rotated = [&](float4 f, double2& xy, double2& zr) {
                    const d3 r = mat_mul(Q, d3{f.x, f.y, f.z});
                    const double Rsum = static_cast<double>(f.w) + r_gas;
                    xy = make_double2(r.x, r.y);
                    zr = make_double2(r.z, Rsum * Rsum);
                };
                double bm = 0.0;
#pragma unroll
                for (int r = 0; r < kWaveRows; ++r) {
                    if (64u * r < nat) {
                        double2 xy, zr;
                        rotated(row[r], xy, zr);
                        // (a lane past the last atom repeats it: the same extent)
                        const double ext = sqrt(xy.x * xy.x + xy.y * xy.y) + static_cast<double>(row[r].w);
                        bm = ext > bm ? ext : bm;
                        if (lane + 64u * r >= nat) zr.y = -1.0;   // never a contact
                        lds.xy[lane + 64u * r] = xy;
                        lds.zr[lane + 64u * r] = zr;
                    }
                }
                for (uint32_t j = kWaveAtoms + lane; j < nat; j += 64) {
                    const float4 f = atoms[j];
                    double2 xy, zr;
                    rotated(f, xy, zr);
                    bm = fmax(bm, sqrt(xy.x * xy.x + xy.y * xy.y) + static_cast<double>(f.w));
                }
                if (pending) fetch(__builtin_amdgcn_readfirstlane(static_cast<int>(__builtin_ctzll(pending))));
                if (nat == 0) continue;
                double b_max = wave_reduce_f64(bm, [](double a, double b) { return a > b ? a : b; }) + r_gas;
                // the first contact of impact point (bx, by); true: found
                auto first_contact = [&](double bx, double by) -> bool {
                    double best_s = INFINITY, cx = 0.0, cy = 0.0, ch = 0.0;
                    uint32_t best_j = 0;
                    auto test = [&](uint32_t j, double2 xy, double2 zr) {
                        const double dx = bx - xy.x, dy = by - xy.y;
                        const double dmin2 = dx * dx + dy * dy;
                        if (dmin2 <= zr.y) {
                            const double h = sqrt(zr.y - dmin2);
                            const double s_hit = -zr.x - h;
                            if (s_hit < best_s) {
                                best_s = s_hit;
                                best_j = j;
                                cx = dx;
                                cy = dy;
                                ch = h;
                            }
                        }
                    };
                    const uint32_t staged = min(nat, kWaveAtoms);
#pragma unroll 2
                    for (uint32_t base = 0; base < staged; base += 64)
                        test(base + lane, lds.xy[base + lane], lds.zr[base + lane]);
                    for (uint32_t j = kWaveAtoms + lane; j < nat; j += 64) {
                        double2 xy, zr;
                        rotated(atoms[j], xy, zr);
                        test(j, xy, zr);
                    }
                    if (__ballot(best_s < INFINITY) == 0ull) return false;
                    const double s_min = wave_reduce_f64(best_s, [](double a, double b) { return a < b ? a : b; });
                    uint64_t at = __ballot(best_s == s_min);
                    int W = __builtin_amdgcn_readfirstlane(static_cast<int>(__builtin_ctzll(at)));
                    // equal s_hit: the lowest atom index
                    for (at &= at - 1ull; at; at &= at - 1ull) {
                        const int V = __builtin_amdgcn_readfirstlane(static_cast<int>(__builtin_ctzll(at)));
                        if (readlane_u32(best_j, V) < readlane_u32(best_j, W)) W = V;
                    }
                    const double wx = readlane_f64(cx, W), wy = readlane_f64(cy, W), wh = readlane_f64(ch, W);
                    if (static_cast<int>(lane) == L) {
                        contact = true;
                        nx = wx;
                        ny = wy;
                        nz = wh;
                    }
                    return true;
                };
                // the attempts drawn ahead, then 64 at a time drawn for this ion alone
                const uint32_t drawn = passes * reps;
                double sx = ux[0], sy = uy[0];
                uint32_t from = static_cast<uint32_t>(L), last = from + (reps - 1u) * G;
                for (uint32_t attempt = 0; attempt < kEhssMaxAttempts; ++attempt) {
                    if (attempt >= drawn && ((attempt - drawn) & 63u) == 0u) {
                        rng.impact(attempt + lane, first + L, sx, sy);
                        from = 0;
                    }
                    if (attempt == kBmaxExpansionAttempt + 1) b_max *= kBmaxExpansionFactor;
                    if (first_contact(b_max * readlane_f64(sx, static_cast<int>(from)),
                                      b_max * readlane_f64(sy, static_cast<int>(from))))
                        break;
                    if (attempt + 1 >= drawn) {
                        ++from;
                    } else if (from == last) {   // the next pass
                        from = static_cast<uint32_t>(L);
                        const bool second = attempt + 1 == reps;
                        sx = second ? ux[1] : ux[2];
                        sy = second ? uy[1] : uy[2];
                    } else {
                        from += G;
                    }
                }
            }
            if (hit) {
                ++nc;
                ++ncoll_launch;
            }
            if (contact) {
                // reflection about the contact normal, which points against the axis
                d3 nb{0.0, 0.0, -1.0};
                const double phr2 = nx * nx + ny * ny + nz * nz;
                if (phr2 > kMinContactDistSq) {
                    nb = d3{nx, ny, nz} * (1.0 / sqrt(phr2));
                    if (nb.z > 0.0) nb = nb * -1.0;
                }
                const d3 ax{vrel.x / vrel_mag, vrel.y / vrel_mag, vrel.z / vrel_mag};
                d3 t1, t2;
                ortho_basis_f64(ax, t1, t2);
                nb = t1 * nb.x + t2 * nb.y + ax * nb.z;
                const double vdn = dot(vrel, nb);
                const d3 vr = vrel - nb * (2.0 * vdn);
                const double inv_mt = 1.0 / (m + P.m_gas);
                const d3 Vcom = (vel * m + vn * P.m_gas) * inv_mt;
                vel = Vcom + vr * (P.m_gas * inv_mt);
            }
        }
        if (live) {
            if (P.detect && z_before < P.det_z && pos.z >= P.det_z) {
                double& arrival = S.arrival[here(i)];
                if (isnan(arrival)) arrival = t + dt * (P.det_z - z_before) / (pos.z - z_before);
            }
            if (!contains_f64(P, pos)) {
                active = false;
                S.death[here(i)] = t;
            } else {
                checked = true;
                if (!(isfinite(pos.x) && isfinite(pos.y) && isfinite(pos.z) && isfinite(vel.x) &&
                      isfinite(vel.y) && isfinite(vel.z))) {
                    active = false;
                    S.death[here(i)] = t;
                }
            }
        }
    }
    if (have) {
        S.x[i] = pos.x; S.y[i] = pos.y; S.z[i] = pos.z;
        S.vx[i] = vel.x; S.vy[i] = vel.y; S.vz[i] = vel.z;
        S.flags[i] = static_cast<uint8_t>((active ? 1 : 0) | (born ? 2 : 0));
        S.ncoll[i] = nc;
    }
    add_counters(P, pushed, ncoll_launch);
}

// ======================= FP32 + Kahan (fast path) ===========================

// the FP32 helpers (fields, containment, collisions) are in step_device_f32.hpp

template <int INTEG, int FIELD, int COLL, bool SUB = false, bool FLOW = false>
__device__ __forceinline__ void f32_ion(const StepParams& P, const IonPtrs& S, const uint32_t i,
        uint32_t& pushed, uint32_t& ncoll_launch) {
    const FastConst& C = P.fc;
    // state: FP32 (hi, lo) pairs; hi + lo equals the FP64 value to ~2^-48
    const double X[6] = {S.x[i], S.y[i], S.z[i], S.vx[i], S.vy[i], S.vz[i]};
    float hi[6], lo[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        hi[c] = (float)X[c];
        lo[c] = (float)(X[c] - (double)hi[c]);
    }
    const double md = S.mass[i];
    const double qd = S.charge[i];
    const uint32_t sidx = S.species[i];
    const SpeciesDev sp = P.species[sidx];
    const float m = (float)md;
    const float qm = (float)(qd / md);
    const float inv_m_plus = (float)(1.0 / (md + P.m_gas));
    const float kbt2_dt_over_m = (float)(2.0 * kBoltzmann * P.T / md * P.dt);
    uint8_t flags = S.flags[i];
    bool active = flags & 1, born = (flags >> 1) & 1;
    const double birth = S.birth ? S.birth[i] : -INFINITY;
    double death = S.death[i];
    double arrival = S.arrival[i];
    uint32_t nc = S.ncoll[i];
    // damping factor in units of 1/s (force per mass): Langevin lpre/|v|
    float lpre = 0.0f;
    if constexpr (COLL == COLL_DAMPING) {
        double l = 0.0;
        if (P.damping_model == 3) {
            if (P.alpha_gas > 0.0 && P.n > 0.0 && P.v_th > 0.0 && P.m_gas > 0.0) {
                const double mu = (md * P.m_gas) / (md + P.m_gas);
                const double cs1 = kPi * qd * sqrt(P.alpha_gas / (4.0 * kPi * kEpsilon0 * mu));
                l = P.n * cs1 * P.v_th * P.m_gas / (P.m_gas + md);
            }
        } else {
            const double K0 = sp.K0_cm2_Vs;
            if (K0 > 0.0 && md > 0.0 && P.n > 0.0) {
                const double K0t = K0 * 1e-4 * sqrt(kStpTemp / fmax(P.T, 1.0));
                l = qd / ((K0t * (kLoschmidt / P.n)) * md);
            }
        }
        lpre = (float)l;
    }
    // 0: done, 1: stepping, 2: unborn, 3: stepping, position not yet known to
    // be inside.  A register rather than lane masks, which the compiler would
    // merge with the execution mask on every path through the loop.
    uint32_t state = !born ? 2u : active ? 3u : 0u;
    CellF32 cell;
    const float dt = (float)P.dt;
    const float half_dt = 0.5f * dt;
    const float h6 = dt * (1.0f / 6.0f);
    // The loop is wave-uniform and its body one masked region; lanes that leave
    // one by one cost the scalar unit a third of the step's instructions.  With
    // the uniform-field push and the FP32 table values this took 200,003 ions x
    // 10,000 HSS steps from 23.6 to 19.0 ms and 1M ions x 20,000 Boris + kick
    // steps from 123 to 103 ms (bound by vector issue, 3-4 wavefronts per SIMD).
    for (uint32_t k = 0; k < P.n_steps; ++k) {
        if (__ballot(state != 0u) == 0ull) break;
        const StepEntry& te = P.table[k];
        const double t = te.t;
        if (__ballot(state > 1u) != 0ull) {   // before an ion's first step only
            if (state == 2u && t >= birth) {
                born = true;
                state = 3u;
            }
            if (state == 3u) {
                state = 1u;
                if (!contains_f32<FIELD == FIELD_ARRAY_X>(P, C, hi[0], hi[1], hi[2])) {
                    state = 0u;
                    death = t;
                }
            }
        }
        if (state == 1u) {
            const float z_before = hi[2];
            const float z_before_lo = lo[2];
            // the step's gas density over the domain's (scales gamma and the rates)
            const float nrel = te.nrelf;
            const float lp = lpre * nrel;
            const f3 p0{hi[0], hi[1], hi[2]};
            const f3 v0{hi[3], hi[4], hi[5]};
            f3 dpos, dvel;
            push_f32<INTEG, FIELD, COLL, FLOW>(P, C, te, p0, v0, qm, lp, dt, half_dt, cell, dpos, dvel);
            apply_push_f32<INTEG>(hi, lo, dpos, dvel, dt, h6);
            ++pushed;
            if constexpr (COLL != COLL_NONE) {
                PhiloxStream rng(P.seed, i, P.step0 + k);
                f3 v{hi[3], hi[4], hi[5]};
                const f3 vin = v;
                // collision substeps: dt / n_sub each, one continuing stream, in the
                // SUB instantiation (the loop costs the one-stage kernels a
                // wavefront per SIMD)
                const int ns = SUB ? P.n_sub : 1;
                const float sub = SUB ? 1.0f / static_cast<float>(P.n_sub) : 1.0f;
                const float dtc = SUB ? static_cast<float>(P.dt / static_cast<double>(P.n_sub)) : dt;
                uint32_t hits = 0;
                const f3 ug = FLOW ? gas_velocity_f32(P, C, f3{hi[0], hi[1], hi[2]}) : f3{0.0f, 0.0f, 0.0f};
                for (int s = 0; s < ns; ++s)
                    hits += collide_f32<COLL, FLOW, FIELD == FIELD_ARRAY ? INTEG : -1>(
                                P, C, sp, sidx, m, inv_m_plus, lp, kbt2_dt_over_m * sub, v, rng, dtc * nrel,
                                C.n_dt * sub * nrel, ug) ? 1u : 0u;
                if (COLL == COLL_HSS || COLL == COLL_HSS_MIX) {
                    if (hits) {
                        // a collision replaces the velocity: restart its compensation
                        hi[3] = v.x; hi[4] = v.y; hi[5] = v.z;
                        lo[3] = 0.0f; lo[4] = 0.0f; lo[5] = 0.0f;
                        nc += hits;
                        ncoll_launch += hits;
                    }
                } else {
                    kahan_add(hi[3], lo[3], v.x - vin.x);
                    kahan_add(hi[4], lo[4], v.y - vin.y);
                    kahan_add(hi[5], lo[5], v.z - vin.z);
                }
            }
            if (P.detect) {
                keep_branch<FIELD == FIELD_ARRAY_X>();
                if (isnan(arrival)) {
                    const double zb = (double)z_before + (double)z_before_lo;
                    const double za = (double)hi[2] + (double)lo[2];
                    if (zb < P.det_z && za >= P.det_z)
                        arrival = t + P.dt * (P.det_z - zb) / (za - zb);
                }
            }
            if (!(contains_f32<FIELD == FIELD_ARRAY_X>(P, C, hi[0], hi[1], hi[2]) & isfinite(hi[0]) & isfinite(hi[1]) & isfinite(hi[2]) &
                  isfinite(hi[3]) & isfinite(hi[4]) & isfinite(hi[5]))) {
                state = 0u;
                death = t;
            }
        }
    }
    if (state != 2u) active = state != 0u;
    S.x[i] = (double)hi[0] + (double)lo[0];
    S.y[i] = (double)hi[1] + (double)lo[1];
    S.z[i] = (double)hi[2] + (double)lo[2];
    S.vx[i] = (double)hi[3] + (double)lo[3];
    S.vy[i] = (double)hi[4] + (double)lo[4];
    S.vz[i] = (double)hi[5] + (double)lo[5];
    S.flags[i] = static_cast<uint8_t>((active ? 1 : 0) | (born ? 2 : 0));
    S.death[i] = death;
    S.arrival[i] = arrival;
    S.ncoll[i] = nc;
}

template <int INTEG, int FIELD, int COLL, bool SUB>
__global__ void __launch_bounds__(256) step_f32_kernel(const StepParams P, const IonPtrs S) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t pushed = 0, ncoll_launch = 0;
    if (i < P.n_ions) f32_ion<INTEG, FIELD, COLL, SUB, SUB>(P, S, P.order ? P.order[i] : i, pushed, ncoll_launch);
    add_counters(P, pushed, ncoll_launch);
}

// ======================= FP32 + EHSS surrogate ==============================
//
// EHSS with the scattering normal drawn by the surrogate MLP instead of the
// geometry ray test.  The collision test is the reference's (neutral from the
// Maxwellian, P = 1 - exp(-n sigma_eff |v_rel| dt), EHSSCollisionHandler.cpp:222-246);
// a colliding ion draws (u, psi), the MLP maps (u, cos psi, sin psi, features)
// to the contact normal in the collision frame, and the relative velocity is
// reflected about it (offline-table branch, EHSSCollisionHandler.cpp:253-277).
// mlp_eval(step, coll, in, out) evaluates the MLP for the colliding lanes:
// mlp_group_eval (the single-cloud kernel: the workgroup's colliding ions
// gathered into 32-ion blocks through LDS, so the matrix cores evaluate about
// as many rows as there are collisions) or mlp_wave_eval_any (the batch
// kernel: per wavefront, no barriers).  Every lane stays in the step loop
// (dead lanes are masked, not exited) so that barriers and the wave-wide matrix
// instructions see every lane they need.  One ion per lane over P.n_steps
// steps; with mlp_group_eval every lane of the workgroup calls it with the same
// P.n_steps (lanes with i >= P.n_ions are carried along masked).
template <int INTEG, int FIELD, bool AHEAD, class MlpEval>
__device__ __forceinline__ void surr_ion(const StepParams& P, const IonPtrs& S, uint32_t i,
                                         MlpEval&& mlp_eval, uint32_t& pushed, uint32_t& ncoll_launch) {
    const bool valid = i < P.n_ions;
    const uint32_t ii = valid ? i : 0;
    const FastConst& C = P.fc;
    const double X[6] = {S.x[ii], S.y[ii], S.z[ii], S.vx[ii], S.vy[ii], S.vz[ii]};
    float hi[6], lo[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        hi[c] = (float)X[c];
        lo[c] = (float)(X[c] - (double)hi[c]);
    }
    const double md = S.mass[ii];
    const double qd = S.charge[ii];
    const SpeciesDev sp = P.species[S.species[ii]];
    const float sigma = (float)sp.sigma_ehss;
    const float qm = (float)(qd / md);
    const float m = (float)md;
    const float inv_m_plus = (float)(1.0 / (md + P.m_gas));
    const uint8_t flags = S.flags[ii];
    const bool active = flags & 1, born = (flags >> 1) & 1;
    // 0: done, 1: stepping, 2: unborn, 3: stepping, position not yet known to
    // be inside.  Birth, death and arrival times stay in memory until their
    // event: registers decide this kernel's occupancy.
    uint32_t state = !valid ? 0u : !born ? 2u : active ? 3u : 0u;
    uint32_t nc = 0;
    const float dt = (float)P.dt;
    const float half_dt = 0.5f * dt;
    const float h6 = dt * (1.0f / 6.0f);
    CellF32 cell;
    // AHEAD: the next step's table entry is loaded one step ahead
    StepEntry te_next{};
    if (AHEAD && P.n_steps) te_next = P.table[0];
    for (uint32_t k = 0; k < P.n_steps; ++k) {
        StepEntry te;
        if constexpr (AHEAD) {
            te = te_next;
            if (k + 1 < P.n_steps) te_next = P.table[k + 1];
        } else {
            te = P.table[k];
        }
        const double t = te.t;
        if (__ballot(state > 1u) != 0ull) {   // before an ion's first step only
            if (state == 2u && (!S.birth || t >= S.birth[here(ii)])) state = 3u;
            if (state == 3u) {
                state = 1u;
                if (!contains_f32<FIELD == FIELD_ARRAY_X>(P, C, hi[0], hi[1], hi[2])) {
                    state = 0u;
                    S.death[here(ii)] = t;
                }
            }
        }
        const bool live = state == 1u;
        bool coll = false;
        float in[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        f3 vn{0.f, 0.f, 0.f}, vrel{0.f, 0.f, 0.f};
        float vm = 0.f;
        float z_before = hi[2], z_before_lo = lo[2];
        if (live) {
            const f3 p0{hi[0], hi[1], hi[2]};
            const f3 v0{hi[3], hi[4], hi[5]};
            f3 dpos, dvel;
            push_f32<INTEG, FIELD, COLL_NONE>(P, C, te, p0, v0, qm, 0.f, dt, half_dt, cell, dpos, dvel);
            apply_push_f32<INTEG>(hi, lo, dpos, dvel, dt, h6);
            ++pushed;
            if (sigma > 0.0f) {
                PhiloxStream rng(P.seed, i, P.step0 + k);
                const float u1 = rng.uniform_f32(), u2 = rng.uniform_f32();
                const float u3 = rng.uniform_f32(), u4 = rng.uniform_f32();
                const float r1 = C.sigma_neutral * fast_sqrt(-2.0f * fast_ln(u1));
                const float r2 = C.sigma_neutral * fast_sqrt(-2.0f * fast_ln(u3));
                vn = f3{fmaf(r1, fast_cos_rev(u2), C.u_gas[0]), fmaf(r1, fast_sin_rev(u2), C.u_gas[1]),
                        fmaf(r2, fast_cos_rev(u4), C.u_gas[2])};
                const f3 v{hi[3], hi[4], hi[5]};
                vrel = v - vn;
                vm = fast_sqrt(speed2_f32<INTEG>(vrel));
                if (vm >= (float)kMinRelativeVelocity) {
                    // n dt of the step (the density ratio of a pressure waveform)
                    const float x = C.n_dt * te.nrelf * sigma * vm;
                    const float Pc = collision_probability_f32(x);
                    if (rng.uniform_f32() < Pc) {
                        coll = true;
                        const float uq = rng.uniform_f32();
                        const float psi = rng.uniform_f32();  // revolutions
                        in[0] = uq;
                        in[1] = fast_cos_rev(psi);
                        in[2] = fast_sin_rev(psi);
                        in[3] = sp.feat[0];
                        in[4] = sp.feat[1];
                        in[5] = sp.feat[2];
                    }
                }
            }
        }
        float out[3];
        if (mlp_eval(k, coll, in, out)) {
            if (coll) {
                const f3 o{out[0], out[1], out[2]};
                const float nrm = fast_sqrt(dot(o, o));
                float mu = nrm > 0.f ? -out[2] / nrm : 0.f;
                mu = fminf(1.f, fmaxf(0.f, mu));
                const float st = fast_sqrt(fmaxf(0.f, fmaf(-mu, mu, 1.f)));
                const float inv = 1.0f / vm;
                const f3 ax{vrel.x * inv, vrel.y * inv, vrel.z * inv};
                const f3 a = fabsf(ax.x) < 0.9f ? f3{1.f, 0.f, 0.f} : f3{0.f, 1.f, 0.f};
                f3 t1 = cross(ax, a);
                t1 = t1 * (1.0f / fast_sqrt(dot(t1, t1)));
                f3 t2 = cross(ax, t1);
                t2 = t2 * (1.0f / fast_sqrt(dot(t2, t2)));
                const f3 nvec = fma3(ax, -mu, fma3(t1, st * in[1], t2 * (st * in[2])));
                const f3 vr = fma3(nvec, -2.0f * dot(vrel, nvec), vrel);
                const f3 v{hi[3], hi[4], hi[5]};
                // centre of mass velocity + relative velocity times the neutral's share
                const f3 vnew = fma3(fma3(v, m, vn * C.m_gas), inv_m_plus, vr * (C.m_gas * inv_m_plus));
                hi[3] = vnew.x; hi[4] = vnew.y; hi[5] = vnew.z;
                lo[3] = 0.f; lo[4] = 0.f; lo[5] = 0.f;
                ++nc;
                ++ncoll_launch;
            }
        }
        if (live) {
            if (P.detect) {
                keep_branch<FIELD == FIELD_ARRAY_X>();
                const double zb = (double)z_before + (double)z_before_lo;
                const double za = (double)hi[2] + (double)lo[2];
                if (zb < P.det_z && za >= P.det_z) {
                    double& arrival = S.arrival[here(ii)];
                    if (isnan(arrival)) arrival = t + P.dt * (P.det_z - zb) / (za - zb);
                }
            }
            if (!(contains_f32<FIELD == FIELD_ARRAY_X>(P, C, hi[0], hi[1], hi[2]) & isfinite(hi[0]) & isfinite(hi[1]) & isfinite(hi[2]) &
                  isfinite(hi[3]) & isfinite(hi[4]) & isfinite(hi[5]))) {
                state = 0u;
                S.death[here(ii)] = t;
            }
        }
    }
    if (valid) {
        S.x[i] = (double)hi[0] + (double)lo[0];
        S.y[i] = (double)hi[1] + (double)lo[1];
        S.z[i] = (double)hi[2] + (double)lo[2];
        S.vx[i] = (double)hi[3] + (double)lo[3];
        S.vy[i] = (double)hi[4] + (double)lo[4];
        S.vz[i] = (double)hi[5] + (double)lo[5];
        if (state != 2u) S.flags[i] = static_cast<uint8_t>((state != 0u ? 1 : 0) | 2);
        S.ncoll[i] += nc;
    }
}

// OCC: wavefronts per SIMD.  Four (128 registers and 4 spilled ones, 40 KB of LDS
// per workgroup) run a large cloud faster, three a small one, whose one or two
// wavefronts per SIMD gain from the registers instead (surrogate_large): 1M ions x
// 4000 steps 151.8 and 134 ms, 3001 x 2000 6.9 and 7.8 ms (three and four).
template <int INTEG, int FIELD, int OCC>
__global__ void __launch_bounds__(kSurrogateBlock, OCC) step_surrogate_kernel(const StepParams P, const IonPtrs S) {
    __shared__ uint4 mlp_lds[kPackBytes / 16];
    __shared__ MlpExchange<kSurrogateBlock / 64> xch;
    mlp_exchange_init(xch);
    mlp_stage(P.mlp_blob, mlp_lds);
    const unsigned char* lds = reinterpret_cast<const unsigned char*>(mlp_lds);
    uint32_t pushed = 0, nc = 0;
    // lanes below ions_per_wave own an ion each; the others take part in the MLP
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t first = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * P.ions_per_wave;
    surr_ion<INTEG, FIELD, OCC == 3>(P, S, lane < P.ions_per_wave ? first + lane : 0xFFFFFFFFu,
                           [&](uint32_t k, bool coll, const float* in, float* out) {
                               return mlp_group_eval(lds, xch, k, coll, in, out, k + blockIdx.x);
                           },
                           pushed, nc);
    add_counters(P, pushed, nc);
}

// ======================= batched clouds (persistent) ========================
//
// A fixed pool of workgroups pulls tiles from a queue until it is empty; the
// host orders the tiles longest first, so the long clouds start first and the
// short ones fill in at the end.  Every workgroup leaves the loop once the
// queue index passes the tile count.  Each tile runs the per-ion body of the
// single-cloud kernels (f64_ion, f32_ion): a cloud's ions take the same course as
// on a handle of their own, to rounding, where the compiler fuses other products,
// or where the handle runs four lanes per ion (step_f64_quad_kernel).

template <int PREC, bool SUB, int I, int F, int Cc>
__device__ __forceinline__ void batch_ion(const StepParams& P, const IonPtrs& S, uint32_t i,
                                          uint32_t& pushed, uint32_t& nc) {
    if constexpr (PREC == 1) {
        f32_ion<I, F, Cc, SUB>(P, S, i, pushed, nc);
    } else {
        f64_ion<I, F, Cc, SUB>(P, S, i, pushed, nc);
    }
}

// MIX: the kernel also holds the gas-mixture kinds (12-15), in FP64 the
// geometry EHSS kinds (16-19), and the uniform-grid field-array kinds (20-25),
// and its FP32 bodies run collision substeps (clouds with more than one
// collision stage per step run in this variant).
// Their bodies need more registers, so a batch without such clouds runs the
// variant without them (FP32: 90 VGPRs, 5 waves per SIMD).
template <int PREC, bool MIX>
__device__ __forceinline__ void batch_dispatch(uint32_t kind, const StepParams& P, const IonPtrs& S,
                                               uint32_t i, uint32_t& pushed, uint32_t& nc) {
    switch (kind) {
        case 0: batch_ion<PREC, MIX, 0, FIELD_LINEAR, COLL_NONE>(P, S, i, pushed, nc); break;
        case 1: batch_ion<PREC, MIX, 1, FIELD_LINEAR, COLL_NONE>(P, S, i, pushed, nc); break;
        case 2: batch_ion<PREC, MIX, 0, FIELD_ORBITRAP, COLL_NONE>(P, S, i, pushed, nc); break;
        case 3: batch_ion<PREC, MIX, 1, FIELD_ORBITRAP, COLL_NONE>(P, S, i, pushed, nc); break;
        case 4: batch_ion<PREC, MIX, 0, FIELD_LINEAR, COLL_HSS>(P, S, i, pushed, nc); break;
        case 5: batch_ion<PREC, MIX, 1, FIELD_LINEAR, COLL_HSS>(P, S, i, pushed, nc); break;
        case 6: batch_ion<PREC, MIX, 0, FIELD_ORBITRAP, COLL_HSS>(P, S, i, pushed, nc); break;
        case 7: batch_ion<PREC, MIX, 1, FIELD_ORBITRAP, COLL_HSS>(P, S, i, pushed, nc); break;
        case 8: batch_ion<PREC, MIX, 0, FIELD_LINEAR, COLL_DAMPING>(P, S, i, pushed, nc); break;
        case 9: batch_ion<PREC, MIX, 1, FIELD_LINEAR, COLL_DAMPING>(P, S, i, pushed, nc); break;
        case 10: batch_ion<PREC, MIX, 0, FIELD_ORBITRAP, COLL_DAMPING>(P, S, i, pushed, nc); break;
        case 11: batch_ion<PREC, MIX, 1, FIELD_ORBITRAP, COLL_DAMPING>(P, S, i, pushed, nc); break;
        default:
            if constexpr (MIX) {
                switch (kind) {
                    case 12: batch_ion<PREC, MIX, 0, FIELD_LINEAR, COLL_HSS_MIX>(P, S, i, pushed, nc); break;
                    case 13: batch_ion<PREC, MIX, 1, FIELD_LINEAR, COLL_HSS_MIX>(P, S, i, pushed, nc); break;
                    case 14: batch_ion<PREC, MIX, 0, FIELD_ORBITRAP, COLL_HSS_MIX>(P, S, i, pushed, nc); break;
                    case 15: batch_ion<PREC, MIX, 1, FIELD_ORBITRAP, COLL_HSS_MIX>(P, S, i, pushed, nc); break;
                    case 20: batch_ion<PREC, MIX, 0, FIELD_ARRAY, COLL_NONE>(P, S, i, pushed, nc); break;
                    case 21: batch_ion<PREC, MIX, 1, FIELD_ARRAY, COLL_NONE>(P, S, i, pushed, nc); break;
                    case 22: batch_ion<PREC, MIX, 0, FIELD_ARRAY, COLL_HSS>(P, S, i, pushed, nc); break;
                    case 23: batch_ion<PREC, MIX, 1, FIELD_ARRAY, COLL_HSS>(P, S, i, pushed, nc); break;
                    case 24: batch_ion<PREC, MIX, 0, FIELD_ARRAY, COLL_DAMPING>(P, S, i, pushed, nc); break;
                    case 25: batch_ion<PREC, MIX, 1, FIELD_ARRAY, COLL_DAMPING>(P, S, i, pushed, nc); break;
                    default:
                        if constexpr (PREC == 0) {
                            switch (kind) {
                                case 16: batch_ion<0, MIX, 0, FIELD_LINEAR, COLL_EHSS>(P, S, i, pushed, nc); break;
                                case 17: batch_ion<0, MIX, 1, FIELD_LINEAR, COLL_EHSS>(P, S, i, pushed, nc); break;
                                case 18: batch_ion<0, MIX, 0, FIELD_ORBITRAP, COLL_EHSS>(P, S, i, pushed, nc); break;
                                case 19: batch_ion<0, MIX, 1, FIELD_ORBITRAP, COLL_EHSS>(P, S, i, pushed, nc); break;
                                default: break;
                            }
                        }
                        break;
                }
            }
            break;
    }
}

// Persistent tile loop shared by the batch kernels: take tiles from the queue
// until it is empty, run `body(cloud, first ion)` on each, stamp the cloud's
// completion clock after the tile.  Queue and clock updates are made by wave 0
// under a wave-uniform branch (all its lanes, one combined increment): a
// lane-divergent region on each side of the loop's back edge could be merged
// by the compiler into a divergent loop in which lanes 1..63 pass the barriers
// again before lane 0 has taken the next tile.
template <typename Body>
__device__ __forceinline__ void batch_queue_loop(const BatchTile* __restrict__ tiles, uint32_t n_tiles,
                                                 uint32_t* queue, unsigned long long* done,
                                                 unsigned long long* start, Body&& body) {
    __shared__ uint32_t s_tile;
    const bool wave0 = __builtin_amdgcn_readfirstlane(threadIdx.x) == 0;
    const uint32_t lane = threadIdx.x & 63;
    if (wave0) atomicMin(start, static_cast<unsigned long long>(__builtin_amdgcn_s_memrealtime()));
    uint32_t prev = 0xFFFFFFFFu;
    for (;;) {
        if (wave0) {
            if (prev != 0xFFFFFFFFu)
                atomicMax(&done[prev], static_cast<unsigned long long>(__builtin_amdgcn_s_memrealtime()));
            const uint32_t got = atomicAdd(queue, lane == 0 ? 1u : 0u);
            s_tile = __builtin_amdgcn_readfirstlane(got);
        }
        __syncthreads();
        const uint32_t tile = __builtin_amdgcn_readfirstlane(s_tile);
        __syncthreads();
        if (tile >= n_tiles) break;
        const uint32_t c = __builtin_amdgcn_readfirstlane(tiles[tile].cloud);
        const uint32_t first = __builtin_amdgcn_readfirstlane(tiles[tile].first);
        body(c, first);
        __syncthreads();   // the whole tile is done before its cloud's clock is stamped
        prev = c;
    }
}

// The per-cloud tables come in as separate read-only, non-aliased arguments so
// that the wave-uniform parameter loads stay scalar.
template <int PREC, bool MIX>
__global__ void __launch_bounds__(256) batch_kernel(const StepParams* __restrict__ params,
                                                    const IonPtrs* __restrict__ ions,
                                                    const uint32_t* __restrict__ kinds,
                                                    const BatchTile* __restrict__ tiles, uint32_t n_tiles,
                                                    uint32_t* queue, unsigned long long* done,
                                                    unsigned long long* start) {
    batch_queue_loop(tiles, n_tiles, queue, done, start, [&](uint32_t c, uint32_t first) {
        const StepParams& P = params[c];
        const IonPtrs S = ions[c];
        const uint32_t kind = __builtin_amdgcn_readfirstlane(kinds[c]);
        const uint32_t i = first + threadIdx.x;
        uint32_t pushed = 0, nc = 0;
        if (i < P.n_ions) batch_dispatch<PREC, MIX>(kind, P, S, i, pushed, nc);
        add_counters(P, pushed, nc);
    });
}

// FP32 + EHSS surrogate clouds: the packed MLP weights are staged into LDS once
// per persistent workgroup and serve every tile it takes.  kind = integrator
// (0 RK4, 1 Boris) + 2 * (Orbitrap field).  The MLP runs per wavefront, both
// halves together (mlp_wave_eval_any, two waves per SIMD): in this kernel the
// workgroup-wide batches and the one-block-at-a-time core of the single-cloud
// kernel measured slower (2.53e10 against 2.88e10 ion-steps/s on 256 EHSS
// clouds).  A wavefront whose 64 ions all lie beyond the cloud's end skips the
// tile.
__global__ void __launch_bounds__(256, 2) batch_surrogate_kernel(const StepParams* __restrict__ params,
                                                                 const IonPtrs* __restrict__ ions,
                                                                 const uint32_t* __restrict__ kinds,
                                                                 const BatchTile* __restrict__ tiles,
                                                                 uint32_t n_tiles, uint32_t* queue,
                                                                 unsigned long long* done,
                                                                 unsigned long long* start,
                                                                 const uint4* __restrict__ blob) {
    __shared__ uint4 mlp_lds[kPackBytes / 16];
    mlp_stage(blob, mlp_lds);
    const unsigned char* lds = reinterpret_cast<const unsigned char*>(mlp_lds);
    const auto eval = [&](uint32_t, bool coll, const float* in, float* out) {
        return mlp_wave_eval_any(lds, coll, in, out);
    };
    batch_queue_loop(tiles, n_tiles, queue, done, start, [&](uint32_t c, uint32_t first) {
        const StepParams& P = params[c];
        const IonPtrs S = ions[c];
        const uint32_t kind = __builtin_amdgcn_readfirstlane(kinds[c]);
        const uint32_t wave_first = first + __builtin_amdgcn_readfirstlane(threadIdx.x & ~63u);
        uint32_t pushed = 0, nc = 0;
        if (wave_first < P.n_ions) {
            const uint32_t i = first + threadIdx.x;
            switch (kind) {
                case 0: surr_ion<0, FIELD_LINEAR, true>(P, S, i, eval, pushed, nc); break;
                case 1: surr_ion<1, FIELD_LINEAR, true>(P, S, i, eval, pushed, nc); break;
                case 2: surr_ion<0, FIELD_ORBITRAP, true>(P, S, i, eval, pushed, nc); break;
                case 3: surr_ion<1, FIELD_ORBITRAP, true>(P, S, i, eval, pushed, nc); break;
                default: break;
            }
        }
        add_counters(P, pushed, nc);
    });
}

__global__ void batch_reset_kernel(uint32_t* queue, unsigned long long* done, unsigned long long* start,
                                   unsigned long long* counters, uint32_t n_clouds) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kBatchClasses) queue[i] = 0u;
    if (i == 0) *start = ~0ull;
    if (i < n_clouds) {
        done[i] = 0ull;
        counters[4 * i + 0] = 0ull; counters[4 * i + 1] = 0ull;
        counters[4 * i + 2] = 0ull; counters[4 * i + 3] = 0ull;
    }
}

// Reset the queue/clock/counter records, then the persistent kernel of each
// class present (FP64, FP32, FP32 + surrogate; a class with n_tiles == 0 is
// skipped).  The first class present runs on `s`, the others on the side
// streams, forked from and joined back into `s`, so that the classes overlap.
hipError_t launch_batch(const BatchParams* B, const uint32_t* block, const uint32_t* grid,
                        const uint4* blob, uint32_t n_clouds, unsigned long long* counters, hipStream_t s,
                        const hipStream_t* side, hipEvent_t fork, const hipEvent_t* join) {
    hipLaunchKernelGGL(batch_reset_kernel, dim3((n_clouds + 255) / 256 + 1), dim3(256), 0, s, B[0].queue,
                       B[0].done, B[0].start, counters, n_clouds);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    int present[kBatchClasses], n_present = 0;
    for (int c = 0; c < kBatchClasses; ++c)
        if (B[c].n_tiles) present[n_present++] = c;
    if (n_present > 1 && (e = hipEventRecord(fork, s)) != hipSuccess) return e;
    for (int k = 0; k < n_present; ++k) {
        const int c = present[k];
        hipStream_t st = k == 0 ? s : side[k - 1];
        if (k > 0 && (e = hipStreamWaitEvent(st, fork, 0)) != hipSuccess) return e;
        const BatchParams& b = B[c];
        if (c == 0 && b.with_mix)
            hipLaunchKernelGGL((batch_kernel<0, true>), dim3(grid[c]), dim3(block[c]), 0, st, b.params, b.ions,
                               b.kinds, b.tiles, b.n_tiles, b.queue, b.done, b.start);
        else if (c == 0)
            hipLaunchKernelGGL((batch_kernel<0, false>), dim3(grid[c]), dim3(block[c]), 0, st, b.params, b.ions,
                               b.kinds, b.tiles, b.n_tiles, b.queue, b.done, b.start);
        else if (c == 1 && b.with_mix)
            hipLaunchKernelGGL((batch_kernel<1, true>), dim3(grid[c]), dim3(block[c]), 0, st, b.params, b.ions,
                               b.kinds, b.tiles, b.n_tiles, b.queue, b.done, b.start);
        else if (c == 1)
            hipLaunchKernelGGL((batch_kernel<1, false>), dim3(grid[c]), dim3(block[c]), 0, st, b.params, b.ions,
                               b.kinds, b.tiles, b.n_tiles, b.queue, b.done, b.start);
        else
            hipLaunchKernelGGL(batch_surrogate_kernel, dim3(grid[c]), dim3(256), 0, st, b.params, b.ions,
                               b.kinds, b.tiles, b.n_tiles, b.queue, b.done, b.start, blob);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    for (int k = 1; k < n_present; ++k) {
        if ((e = hipEventRecord(join[k - 1], side[k - 1])) != hipSuccess) return e;
        if ((e = hipStreamWaitEvent(s, join[k - 1], 0)) != hipSuccess) return e;
    }
    return hipSuccess;
}

// ======================= trajectory snapshots ================================
//
// One pass over the SoA state per snapshot:
//   * the full snapshot in OutputManager's layout (positions and velocities
//     interleaved [n][3] in FP64, species, domain index, flags) into a
//     device staging slot;
//   * the records of the ions that may have changed since the previous
//     snapshot: those active now, or whose flags changed (died or were born
//     since).  Unborn and dead ions do not move, so the others hold the values
//     the previous snapshot gave them.  Records are compacted per workgroup
//     (wave ballots + one atomic per workgroup); their order across workgroups
//     is arbitrary and each carries its ion index.
// prev[] keeps every ion's flags at the last snapshot; full = 1 selects every ion.
struct SnapRecord {
    double p[3];
    double v[3];
    uint32_t idx;
    uint8_t flags;
    int8_t domain;
    uint16_t pad;
};
static_assert(sizeof(SnapRecord) == 56, "snapshot record layout");

// 1024 threads per workgroup: the records of its 16 waves take one atomic.  No
// thread leaves before the barriers (lanes past n carry sel = false).
constexpr int kPackThreads = 1024;

__global__ void __launch_bounds__(kPackThreads) pack_snapshot_kernel(const IonPtrs S, uint32_t n, int full,
                                                                     double* __restrict__ pos, double* __restrict__ vel,
                                                                     uint32_t* __restrict__ spec,
                                                                     int32_t* __restrict__ dom,
                                                                     uint8_t* __restrict__ flags,
                                                                     uint8_t* __restrict__ prev,
                                                                     SnapRecord* __restrict__ rec,
                                                                     uint32_t* __restrict__ count) {
    __shared__ uint32_t wave_base[kPackThreads / 64];
    __shared__ uint32_t block_base;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool in = i < n;
    bool sel = false;
    double x = 0, y = 0, z = 0, vx = 0, vy = 0, vz = 0;
    uint8_t f = 0;
    int32_t d = 0;
    if (in) {
        x = S.x[i]; y = S.y[i]; z = S.z[i];
        vx = S.vx[i]; vy = S.vy[i]; vz = S.vz[i];
        f = S.flags[i];
        d = S.domain ? S.domain[i] : 0;
        const size_t o = 3ull * i;
        pos[o] = x; pos[o + 1] = y; pos[o + 2] = z;
        vel[o] = vx; vel[o + 1] = vy; vel[o + 2] = vz;
        spec[i] = S.species[i];
        dom[i] = d;
        flags[i] = f;
        sel = full || (f & 1) || f != prev[i];
        prev[i] = f;
    }
    const unsigned long long m = __ballot(sel);
    const int lane = static_cast<int>(threadIdx.x & 63);
    const int wave = static_cast<int>(threadIdx.x >> 6);
    if (lane == 0) wave_base[wave] = static_cast<uint32_t>(__popcll(m));
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t total = 0;
        const int n_waves = static_cast<int>(blockDim.x >> 6);
        for (int w = 0; w < n_waves; ++w) {
            const uint32_t c = wave_base[w];
            wave_base[w] = total;
            total += c;
        }
        block_base = total ? atomicAdd(count, total) : 0u;
    }
    __syncthreads();
    if (sel) {
        const uint32_t k = block_base + wave_base[wave] +
                           static_cast<uint32_t>(__popcll(m & ((1ull << lane) - 1ull)));
        SnapRecord r;
        r.p[0] = x; r.p[1] = y; r.p[2] = z;
        r.v[0] = vx; r.v[1] = vy; r.v[2] = vz;
        r.idx = i;
        r.flags = f;
        r.domain = static_cast<int8_t>(d);
        r.pad = 0;
        rec[k] = r;
    }
}

// After a pack: its record count to pinned host memory (a vector store, read by
// the host once the stream has passed this kernel), and the counter of the
// next pack cleared.
__global__ void publish_count_kernel(const uint32_t* count, uint32_t* host_count, uint32_t* next_count) {
    if (threadIdx.x == 0) {
        host_count[0] = count[0];
        next_count[0] = 0u;
        __threadfence_system();
    }
}

__global__ void zero_u32_kernel(uint32_t* p) {
    if (threadIdx.x == 0) p[0] = 0u;
}

hipError_t launch_zero_u32(uint32_t* p, hipStream_t s) {
    hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(64), 0, s, p);
    return hipGetLastError();
}

// count must be zero on entry (launch_zero_u32 before the first pack; each
// publish clears next_count for the pack after it).
hipError_t launch_pack_snapshot(const IonPtrs& S, uint32_t n, int full, double* pos, double* vel, uint32_t* spec,
                                int32_t* dom, uint8_t* flags, uint8_t* prev, void* rec, uint32_t* count,
                                uint32_t* host_count, uint32_t* next_count, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(pack_snapshot_kernel, dim3((n + kPackThreads - 1) / kPackThreads), dim3(kPackThreads), 0, s,
                       S, n, full, pos, vel, spec, dom, flags, prev, static_cast<SnapRecord*>(rec), count);
    hipLaunchKernelGGL(publish_count_kernel, dim3(1), dim3(64), 0, s, count, host_count, next_count);
    return hipGetLastError();
}

// ---- launch dispatch --------------------------------------------------------

using KernelFn = void (*)(const StepParams, const IonPtrs);

// sub: more than one collision stage per step (the FP32 kernels have an
// instantiation of their own for it; the FP64 bodies loop at run time)
template <int I, int F, int Cc>
KernelFn pick_prec(int precision, bool sub) {
    if constexpr (Cc != COLL_NONE) {
        if (sub) return precision == 1 ? step_f32_kernel<I, F, Cc, true> : step_f64_kernel<I, F, Cc, true>;
    }
    return precision == 1 ? step_f32_kernel<I, F, Cc, false> : step_f64_kernel<I, F, Cc, false>;
}

template <int I, int F, int Cc>
KernelFn pick_f64(bool sub) {
    return sub ? step_f64_kernel<I, F, Cc, true> : step_f64_kernel<I, F, Cc, false>;
}

template <int I, int F>
KernelFn pick_coll(int coll, int precision, bool sub) {
    switch (coll) {
        case COLL_HSS: return pick_prec<I, F, COLL_HSS>(precision, sub);
        case COLL_HSS_MIX: return pick_prec<I, F, COLL_HSS_MIX>(precision, sub);
        case COLL_EHSS: return precision == 1 ? nullptr : step_f64_ehss_kernel<I, F>;
        case COLL_EHSS_TAB: return precision == 1 ? nullptr : pick_f64<I, F, COLL_EHSS_TAB>(sub);
        case COLL_EHSS_MIX: return precision == 1 ? nullptr : pick_f64<I, F, COLL_EHSS_MIX>(sub);
        case COLL_DAMPING: return pick_prec<I, F, COLL_DAMPING>(precision, sub);
        default: return pick_prec<I, F, COLL_NONE>(precision, sub);
    }
}

template <int I>
KernelFn pick_field(int field, int coll, int precision, bool sub) {
    switch (field) {
        case FIELD_ORBITRAP: return pick_coll<I, FIELD_ORBITRAP>(coll, precision, sub);
        case FIELD_ARRAY: return pick_coll<I, FIELD_ARRAY>(coll, precision, sub);
        case FIELD_ARRAY_X: return pick_coll<I, FIELD_ARRAY_X>(coll, precision, sub);
        default: return pick_coll<I, FIELD_LINEAR>(coll, precision, sub);
    }
}

// large: four wavefronts per SIMD; the field-array kernels, which keep a cell's
// corners in registers, have three for every cloud.
template <int I>
KernelFn pick_surrogate(int field, bool large) {
    switch (field) {
        case FIELD_ORBITRAP:
            return large ? step_surrogate_kernel<I, FIELD_ORBITRAP, 4> : step_surrogate_kernel<I, FIELD_ORBITRAP, 3>;
        case FIELD_ARRAY: return step_surrogate_kernel<I, FIELD_ARRAY, 3>;
        case FIELD_ARRAY_X: return step_surrogate_kernel<I, FIELD_ARRAY_X, 3>;
        default: return large ? step_surrogate_kernel<I, FIELD_LINEAR, 4> : step_surrogate_kernel<I, FIELD_LINEAR, 3>;
    }
}

// The four-lanes-per-ion kernel of a combination, or null.
KernelFn pick_quad(int integrator, int field, int coll) {
    if (field != FIELD_LINEAR) return nullptr;
    switch (coll) {
        case COLL_NONE: return integrator == 1 ? step_f64_quad_kernel<1, COLL_NONE> : step_f64_quad_kernel<0, COLL_NONE>;
        case COLL_HSS: return integrator == 1 ? step_f64_quad_kernel<1, COLL_HSS> : step_f64_quad_kernel<0, COLL_HSS>;
        case COLL_DAMPING:
            return integrator == 1 ? step_f64_quad_kernel<1, COLL_DAMPING> : step_f64_quad_kernel<0, COLL_DAMPING>;
        default: return nullptr;
    }
}

hipError_t launch_quad(KernelFn fn, const StepParams& P, const IonPtrs& S, hipStream_t stream) {
    const uint32_t per_block = 256 / 4;
    hipLaunchKernelGGL(fn, dim3((P.n_ions + per_block - 1) / per_block), dim3(256), 0, stream, P, S);
    return hipGetLastError();
}

// Returns hipSuccess, or hipErrorInvalidValue when the combination has no
// kernel (the host maps that to ICARION_ERR_UNSUPPORTED).
hipError_t launch_step(int integrator, int field, int coll, int precision, int surrogate,
                       const StepParams& params, const IonPtrs& S, uint32_t block, hipStream_t stream) {
    StepParams P = params;
    KernelFn fn;
    if (surrogate) {
        const bool large = surrogate_large(P.n_ions);
        fn = integrator == 1 ? pick_surrogate<1>(field, large) : pick_surrogate<0>(field, large);
    } else {
        // the extended instantiation: collision substeps or a parabolic flow
        const bool ext = P.n_sub > 1 || P.flow_parabolic;
        fn = integrator == 1 ? pick_field<1>(field, coll, precision, ext) : pick_field<0>(field, coll, precision, ext);
        if (KernelFn quad = pick_quad(integrator, field, coll); quad && precision == 0 && !ext && !P.magnetic &&
                                                                !P.order && P.n_ions <= kQuadMaxIons)
            return launch_quad(quad, P, S, stream);
    }
    if (!fn) return hipErrorInvalidValue;
    // the EHSS kernels run their own workgroup size (the handle's block size
    // does not change any result)
    static_assert(kSurrogateBlock == 256, "four wavefronts per workgroup");
    uint32_t grid = (P.n_ions + block - 1) / block;
    if (surrogate || coll == COLL_EHSS) {
        P.ions_per_wave = surrogate ? surrogate_ions_per_wave(P.n_ions)
                                    : ehss_ions_per_wave(P.n_ions, ehss_waves_per_simd(integrator, field == FIELD_ARRAY,
                                                                                       field == FIELD_ARRAY_X));
        block = 256;
        const uint32_t per_block = 4 * P.ions_per_wave;
        grid = (P.n_ions + per_block - 1) / per_block;
    }
    hipLaunchKernelGGL(fn, dim3(grid), dim3(block), 0, stream, P, S);
    return hipGetLastError();
}

}  // namespace icarion
