// Fused per-axis pass of the compressible RHS on gfx950.
//
// One workgroup owns a segment of P neighbouring pencils along the pass axis
// D and walks it in tiles of T cells (em_faces.h).  Phases of a tile
// (LDS-staged, one barrier between each):
//   1. load: coalesced SoA loads of the 5 conserved variables of the tile's
//      cells and, in the first tile, its halo of 10 (ghost cells are produced
//      from the boundary condition of the pencil itself), conversion to
//      primitives into LDS (plus the hybrid sensor ln rho, ln(p + p_inf));
//   2. hybrid only: blend weight theta of every face;
//   3. WCNS midpoints: each of the T+5 midpoints of a pencil is computed
//      once (characteristic WENO5-Z interpolation + HLLC) into LDS;
//   4. faces: S6 midpoint-to-node combination, KEEP-PE central flux and the
//      theta blend, Hu-Adams-Shu positivity limiter;
//   5. cells: divergence -(F_{i+1/2} - F_{i-1/2})/dx accumulated in the
//      reference's axis order; on the last active axis fused with the
//      SSP-RK3 combination and the CFL max-rate of the updated state.
// Reference: fluid/crates/compressible/src/scheme.rs:132-281 (line_fluxes),
// 286-333 (midpoint_flux), 395-464 (positivity_limit);
// fluid/crates/compressible/src/solver.rs:97-137 (rk_combine), 351-475 (rhs),
// 259-348 (ghosts), 478-523 (dt_cfl).
//
// This file is compiled once per (variant, flux mode): EM_VARIANT=precise
// with -ffp-contract=off (reproduces the reference CPU arithmetic) or
// EM_VARIANT=fast with FMA contraction; EM_MODE = 0 hybrid, 1 weno,
// 2 central.  Kernels ask for 4 waves per SIMD (<= 128 VGPRs).
//
// Bound by FP64 instruction issue (VALU 85 to 86% busy).  256^3 Weno, x, y and
// z pass of a step: 1.41 to 1.45 and 1.57 to 1.65 ms (z) with independent
// 59-cell tiles and general divisions (2,544, 2,551 and 2,768 VALU
// instructions per cell), 1.03, 1.05, 1.23 ms now (1,857, 1,881 and 2,256).  Code size counts: a version that inlined the
// boundary images three times (59 KB) ran 20% slower than this one.
#include <hip/hip_runtime.h>

#include "em_pass.h"
#include "em_types.h"

#ifndef EM_VARIANT
#error "EM_VARIANT must name the arithmetic variant"
#endif
#ifndef EM_MODE
#error "EM_MODE must name the flux mode instantiated by this translation unit"
#endif
#if EM_MODE == 0
#define EM_LAUNCHER launch_pass_hybrid
#define EM_LAUNCHER32 launch_pass32_hybrid
#define EM_AMR_LAUNCHER launch_amr_hybrid
#define EM_AMR_LAUNCHER32 launch_amr32_hybrid
#define EM_AMR_MULTI_LAUNCHER launch_amr_multi_hybrid
#define EM_ENS_LAUNCHER launch_ens_hybrid
#elif EM_MODE == 1
#define EM_LAUNCHER launch_pass_weno
#define EM_LAUNCHER32 launch_pass32_weno
#define EM_AMR_LAUNCHER launch_amr_weno
#define EM_AMR_LAUNCHER32 launch_amr32_weno
#define EM_AMR_MULTI_LAUNCHER launch_amr_multi_weno
#define EM_ENS_LAUNCHER launch_ens_weno
#else
#define EM_LAUNCHER launch_pass_central
#define EM_LAUNCHER32 launch_pass32_central
#define EM_AMR_LAUNCHER launch_amr_central
#define EM_AMR_LAUNCHER32 launch_amr32_central
#define EM_AMR_MULTI_LAUNCHER launch_amr_multi_central
#define EM_ENS_LAUNCHER launch_ens_central
#endif
#ifndef EM_WAVES_PER_EU
#define EM_WAVES_PER_EU 4
#endif

#include "em_faces.h"
#include "em_amr_pass.h"

namespace em {
namespace EM_VARIANT {

// Conserved state of the virtual ghost cell at pencil coordinate g (outside
// [0, n)) of the pencil starting at cell `pen`.
template <int D, class Real>
__device__ __forceinline__ void ghost_state(const PassArgsT<Real>& a, long long pen, int g, Real u[5]) {
    const long long sD = a.stride[D];
    auto ld = [&](int x, Real* o) {
#pragma unroll
        for (int k = 0; k < 5; ++k) o[k] = a.U[k * a.ncell + pen + (long long)x * sD];
    };
    bc_ghost<D>(a.eos, a.n[D], g, a.bc_kind, a.bc_state, ld, u);
}

// LDS of a pass (declared by the kernels, passed to axis_segment)
template <class Real, int MODE, int T, int P, bool CF, int NT>
struct PassLds : Tile<Real, MODE, T, P, CF, true> {
    double sred[NT / 64 + 1];  // per-wave CFL rate (in double for the slot max)
    unsigned int scnt[3];
};

// Segment `bid` of one axis pass described by `a`: a.seg cells of P
// neighbouring pencils, walked in tiles of T cells (every thread of the
// workgroup calls it; it returns uniformly).
template <class Real, int D, int MODE, int T, int P, bool CF, int NT>
__device__ __forceinline__ void axis_segment(const PassArgsT<Real>& a, int bid, PassLds<Real, MODE, T, P, CF, NT>& L) {
    using TL = Tile<Real, MODE, T, P, CF, true>;
    constexpr bool HYB = MODE == MODE_HYBRID;
    auto& sw = L.sw;
    auto& sm = L.sm;
    auto& sred = L.sred;
    auto& scnt = L.scnt;

    const int tid = threadIdx.x;
    const int sg = bid % a.nseg;
    const int rest = bid / a.nseg;
    const int gF = rest % a.ngroup;
    const int sI = rest / a.ngroup;
    const int nD = a.n[D];
    const int nF = a.n_fast;
    const int s0 = sg * a.seg, s1 = min(s0 + a.seg, nD);
    const int p0 = gF * P;
    const int Pv = min(P, nF - p0);
    const long long sD = a.stride[D];
    const long long sF = a.s_fast;
    const long long base = (long long)sI * a.s_slow + (long long)p0 * sF;
    const long long nc = a.ncell;
    const EosT<Real> e = a.eos;
    if (tid < 3) scnt[tid] = 0;
    if (HYB && tid < P) L.late[tid] = 0;
    // read together and tested behind the first tile's loads: one round trip
    const int active = a.sc->active;
    const double dt_d = wave_uniform(a.sc->dt);
    double lam_d = 0.0;
    if (a.ndim_pos > 0.0) lam_d = a.ndim_pos * (a.stage_dt_host ? a.stage_dt : dt_d) / a.dx_d;  // solver.rs:393
    const Real lam = Real(wave_uniform(lam_d));
    const Real dt = Real(dt_d);
    unsigned int n_shock = 0;
    double rate = 0.0;

#pragma unroll 1
    for (int c0 = s0; c0 < s1; c0 += T) {
        // opaque in every turn: addresses are formed where they are used
        // (hoisted out of the loop they fill the registers and spill)
        const int tid = opaque(threadIdx.x);
        const bool first = HYB || c0 == s0;
        const int Tv = min(T, s1 - c0);
        // ---- 1. load + primitives
#pragma unroll 1
        for (int it = tid - (first ? TL::HC * P : 0); it < T * P; it += NT) {
            int c, p;
            TL::template item<TL::HC>(it, c, p);
            const int g = c0 - 5 + c;
            if (p >= Pv || c >= Tv + TL::HC || g >= nD + 5) continue;
            const long long pen = base + (long long)p * sF;
            Real u[5], w[5];
            if (g >= 0 && g < nD) {
                const long long idx = pen + (long long)g * sD;
#pragma unroll
                for (int k = 0; k < 5; ++k) u[k] = a.U[k * nc + idx];
            } else {
                ghost_state<D>(a, pen, g, u);
            }
            Real v;
            to_prim_v(e, u, w, v);
            const int q = TL::at(c, p);
#pragma unroll
            for (int k = 0; k < 5; ++k) sw[k][q] = w[k];
            L.sre[q] = eos_rho_e_v(e, w[0], w[4], v);
            if constexpr (HYB) {
                // Euler::sensor, system.rs:409-413
                L.ss[0][q] = log(fmax(w[0], Real(1e-300)));
                L.ss[1][q] = log(fmax(w[4] + e.p_inf, Real(1e-300)));
            }
        }
        if (active == 0) return;
        // the midpoints and the face flux taken over from the last tile
        if (!first) {
            if (tid < TL::HM * P) {
                const int m = CF ? tid % TL::HM : tid / P, p = CF ? tid / TL::HM : tid % P;
#pragma unroll
                for (int k = 0; k < 5; ++k) {
                    const Real x = sm[k][TL::mt(T + m, p)];
                    if (m == 0) L.sf[k][p] = sm[k][TL::mt(T - 1, p)];
                    sm[k][TL::mt(m, p)] = x;
                }
            }
        }
        __syncthreads();

        int c, p;
        TL::template item<0>(tid, c, p);
        const bool mine = tid < T * P && p < Pv && c < Tv;
        const long long idx = base + (long long)p * sF + (long long)(c0 + c) * sD;
        Real r[5], u0[5], us[5];
        tile_faces<D, MODE, NT>(L, tid, first, Tv, Pv, c0, s0, s1, nD, e, lam, a.tol, !a.active[(D + 1) % 3],
                                !a.active[(D + 2) % 3], n_shock, scnt, [&] {
#pragma unroll
                                    for (int k = 0; k < 5; ++k) {
                                        r[k] = a.first || !mine ? Real(0.0) : a.R[k * nc + idx];
                                        u0[k] = a.rk_stage == 0 || !mine ? Real(0.0) : a.U0[k * nc + idx];
                                        // stage 1: the stage input is U^n itself
                                        us[k] = a.rk_stage < 2 || !mine ? Real(0.0) : a.U[k * nc + idx];
                                    }
                                });

        // ---- 5. divergence, fused RK stage and CFL rate
        if (mine) {
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                const Real fl = c == 0 ? L.sf[k][p] : sm[k][TL::mt(c - 1, p)];
                r[k] = r[k] - (sm[k][TL::mt(c, p)] - fl) * a.inv_dx;
            }
            if (a.rk_stage == 0) {
#pragma unroll
                for (int k = 0; k < 5; ++k) a.R[k * nc + idx] = r[k];
            } else {
                Real uo[5];
#pragma unroll
                for (int k = 0; k < 5; ++k) {
                    Real o;
                    if (a.rk_stage == 1)
                        o = u0[k] + dt * r[k];
                    else if (a.rk_stage == 2)
                        o = Real(0.75) * u0[k] + Real(0.25) * (us[k] + dt * r[k]);
                    else
                        o = u0[k] / Real(3.0) + Real(2.0) / Real(3.0) * (us[k] + dt * r[k]);
                    uo[k] = o;
                    a.Uout[k * nc + idx] = o;
                }
                if (a.want_rate) {
                    Real w[5], v;
                    to_prim_v(e, uo, w, v);
                    const Real cs = sound_speed(e, w[0], w[4]);
                    Real ac = Real(-0.0);
#pragma unroll
                    for (int d = 0; d < 3; ++d)
                        if (a.active[d]) ac += (fabs(w[1 + d]) + cs) / a.dx_all[d];
                    rate = fmax(rate, (double)ac);
                }
            }
        }
        if constexpr (HYB) {
            late_fallbacks(L, tid, a.tol, scnt, [&](int p, int h, int k) {
                Real u[5], w[5];
                const long long i = base + (long long)p * sF + (long long)(c0 - 7 + h) * sD;
#pragma unroll
                for (int q = 0; q < 5; ++q) u[q] = a.U[q * nc + i];
                to_prim(e, u, w);
                return log(fmax(k ? w[4] + e.p_inf : w[0], Real(1e-300)));
            });
            break;  // one tile (cut_segments)
        }
        // the cells the next tile takes over
        if (c0 + T < s1) {
            for (int it = tid; it < TL::HC * P; it += NT) {
                const int h = CF ? it % TL::HC : it / P, hp = CF ? it / TL::HC : it % P;
                const int q = TL::at(h, hp), o = TL::at(h + T, hp);
#pragma unroll
                for (int k = 0; k < 5; ++k) sw[k][q] = sw[k][o];
                L.sre[q] = L.sre[o];
            }
            __syncthreads();
        }
    }

    // ---- counters (per wave) and rate: one atomic per workgroup
    if (a.want_rate) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) rate = fmax(rate, __shfl_xor(rate, off));
    }
    const int lane = tid & 63, wid = tid >> 6;
    if (lane == 0) {
        if (n_shock) atomicAdd(&scnt[0], n_shock);
        sred[wid] = rate;
    }
    __syncthreads();
    if (tid == 0) {
        const int slot = bid % kSlots;
        if (scnt[0]) atomicAdd(&a.sc->counters[0][slot][0], (unsigned long long)scnt[0]);
        if (scnt[1]) atomicAdd(&a.sc->counters[1][slot][0], (unsigned long long)scnt[1]);
        if (scnt[2]) atomicAdd(&a.sc->counters[2][slot][0], (unsigned long long)scnt[2]);
        if (a.want_rate) {
            double rm = 0.0;
            for (int w = 0; w < (NT + 63) / 64; ++w) rm = fmax(rm, sred[w]);
            rm = rm > 0.0 ? rm : 0.0;  // IEEE bits of +x order like x (no -0.0)
            atomicMax(&a.sc->rate[slot][0], (unsigned long long)__double_as_longlong(rm));
        }
    }
}

template <int D, int MODE, int T, int P, bool CF, int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(EM_WAVES_PER_EU))) void axis_pass(PassArgs a) {
    __shared__ PassLds<double, MODE, T, P, CF, NT> L;
    axis_segment<double, D, MODE, T, P, CF, NT>(a, xcd_major((int)blockIdx.x, (int)gridDim.x), L);
}

// The FP32 variant of the same pass (the reference's GpuSolver<f32>): state,
// residual and arithmetic in float.
template <int D, int MODE, int T, int P, bool CF, int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(EM_WAVES_PER_EU))) void axis_pass_f32(
    PassArgsT<float> a) {
    __shared__ PassLds<float, MODE, T, P, CF, NT> L;
    axis_segment<float, D, MODE, T, P, CF, NT>(a, xcd_major((int)blockIdx.x, (int)gridDim.x), L);
}

// Ensemble pass: the segments of every instance in one persistent launch.  Work
// item w belongs to the instance i = owner[w] and is its segment
// w - prefix[i]; each instance brings its own arrays, extents,
// boundary conditions and device scalars (dt, CFL rate, counters).
template <int D, int MODE, int T, int P, bool CF, int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(EM_WAVES_PER_EU))) void ens_pass(EnsPassArgs e) {
    __shared__ PassLds<double, MODE, T, P, CF, NT> L;
    const XcdStride xs = xcd_stride();
    for (long long t = xs.first;; t += xs.step) {
        const long long w = xs.item(t);
        if (w >= e.total) break;
        const int i = __builtin_amdgcn_readfirstlane(scalar_copy(e.owner + w));
        const PassArgs a = scalar_copy(e.args + i);
        axis_segment<double, D, MODE, T, P, CF, NT>(a, (int)(w - scalar_copy(e.prefix + i)), L);
        __syncthreads();
    }
}

// One launch of tile shape (T, P): the layout of the LDS tile follows
// whether the pass axis is contiguous (the last axis always is).
template <int D, int MODE, int T, int P, int NT>
static hipError_t launch_one(const PassArgs& a, hipStream_t s) {
    const long long blocks = (long long)a.nseg * a.ngroup * a.n[a.slow_axis];
    if (blocks * NT > kMaxLaunchThreads) return hipErrorInvalidValue;
    const dim3 grid((unsigned)blocks);
    if (D == 2 || a.dfast)
        hipLaunchKernelGGL((axis_pass<D, MODE, T, P, true, NT>), grid, dim3(NT), 0, s, a);
    else
        hipLaunchKernelGGL((axis_pass<D, MODE, T, P, D == 2, NT>), grid, dim3(NT), 0, s, a);
    return hipGetLastError();
}
template <int D, int MODE, int T, int P, int NT>
static hipError_t launch_one(const PassArgsT<float>& a, hipStream_t s) {
    const long long blocks = (long long)a.nseg * a.ngroup * a.n[a.slow_axis];
    if (blocks * NT > kMaxLaunchThreads) return hipErrorInvalidValue;
    const dim3 grid((unsigned)blocks);
    if (D == 2 || a.dfast)
        hipLaunchKernelGGL((axis_pass_f32<D, MODE, T, P, true, NT>), grid, dim3(NT), 0, s, a);
    else
        hipLaunchKernelGGL((axis_pass_f32<D, MODE, T, P, D == 2, NT>), grid, dim3(NT), 0, s, a);
    return hipGetLastError();
}

template <int D, int MODE, int T, int P, int NT>
static hipError_t launch_ens_one(const EnsPassArgs& e, unsigned grid, hipStream_t s) {
    if (D == 2 || e.dfast)
        hipLaunchKernelGGL((ens_pass<D, MODE, T, P, true, NT>), dim3(grid), dim3(NT), 0, s, e);
    else
        hipLaunchKernelGGL((ens_pass<D, MODE, T, P, D == 2, NT>), dim3(grid), dim3(NT), 0, s, e);
    return hipGetLastError();
}

// Tile table: must list the shapes of kTileCfgs (em_pass.h) in order.
#define EM_FOR_TILE(CALL)                  \
    switch (cfg) {                         \
        case 0: return CALL(32, 8, 256);  \
        case 1: return CALL(64, 8, 512);  \
        case 2: return CALL(59, 1, 64);  \
        case 3: return CALL(27, 2, 64);  \
        case 4: return CALL(27, 8, 256);  \
        case 5: return CALL(59, 4, 256);  \
        case 6: return CALL(27, 4, 128);  \
        case 7: return CALL(16, 16, 256);  \
        case 8: return CALL(123, 4, 512);  \
        case 9: return CALL(16, 4, 64);  \
        default: return hipErrorInvalidValue; \
    }
template <int D, int MODE, class Args>
static hipError_t launch_cfg(int cfg, const Args& a, hipStream_t s) {
#define EM_CALL(T, P, NT) launch_one<D, MODE, T, P, NT>(a, s)
    EM_FOR_TILE(EM_CALL)
#undef EM_CALL
}

template <int D, int MODE>
static hipError_t launch_ens_cfg(int cfg, const EnsPassArgs& e, unsigned grid, hipStream_t s) {
#define EM_CALL(T, P, NT) launch_ens_one<D, MODE, T, P, NT>(e, grid, s)
    EM_FOR_TILE(EM_CALL)
#undef EM_CALL
}

// This translation unit instantiates one flux mode (EM_MODE).
hipError_t EM_LAUNCHER(int d, int cfg, const PassArgs& a, hipStream_t s) {
    switch (d) {
        case 0: return launch_cfg<0, EM_MODE>(cfg, a, s);
        case 1: return launch_cfg<1, EM_MODE>(cfg, a, s);
        case 2: return launch_cfg<2, EM_MODE>(cfg, a, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t EM_LAUNCHER32(int d, int cfg, const PassArgsT<float>& a, hipStream_t s) {
    switch (d) {
        case 0: return launch_cfg<0, EM_MODE>(cfg, a, s);
        case 1: return launch_cfg<1, EM_MODE>(cfg, a, s);
        case 2: return launch_cfg<2, EM_MODE>(cfg, a, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t EM_ENS_LAUNCHER(int d, int cfg, const EnsPassArgs& e, unsigned grid, hipStream_t s) {
    switch (d) {
        case 0: return launch_ens_cfg<0, EM_MODE>(cfg, e, grid, s);
        case 1: return launch_ens_cfg<1, EM_MODE>(cfg, e, grid, s);
        case 2: return launch_ens_cfg<2, EM_MODE>(cfg, e, grid, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t EM_AMR_MULTI_LAUNCHER(int d, const AmrMultiArgs& m, unsigned grid, hipStream_t s) {
    switch (d) {
        case 0: return launch_amr_multi_d<0, EM_MODE>(m, grid, s);
        case 1: return launch_amr_multi_d<1, EM_MODE>(m, grid, s);
        case 2: return launch_amr_multi_d<2, EM_MODE>(m, grid, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t EM_AMR_LAUNCHER(int d, int b, int shape, const AmrPassArgs& pa, unsigned grid, hipStream_t s) {
    switch (d) {
        case 0: return launch_amr_b<0, EM_MODE>(b, shape, pa, grid, s);
        case 1: return launch_amr_b<1, EM_MODE>(b, shape, pa, grid, s);
        case 2: return launch_amr_b<2, EM_MODE>(b, shape, pa, grid, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t EM_AMR_LAUNCHER32(int d, int b, int shape, const AmrPassArgsT<float>& pa, unsigned grid, hipStream_t s) {
    switch (d) {
        case 0: return launch_amr_b<0, EM_MODE>(b, shape, pa, grid, s);
        case 1: return launch_amr_b<1, EM_MODE>(b, shape, pa, grid, s);
        case 2: return launch_amr_b<2, EM_MODE>(b, shape, pa, grid, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace EM_VARIANT
}  // namespace em
