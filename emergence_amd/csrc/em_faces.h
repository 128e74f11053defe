// Face fluxes of a tile of P pencils held in LDS: the hybrid blend weight
// (scheme.rs:171-183), the WCNS midpoints (scheme.rs:286-333, each computed
// once), the S6 midpoint-to-node combination with the KEEP-PE central flux
// and theta blend (scheme.rs:188-276), and the positivity limiter
// (scheme.rs:395-464).  Shared by the uniform-grid axis pass and the batched
// AMR pass so both evaluate identical arithmetic.
//
// A pass walks a segment [s0, s1) of its pencils tile by tile (T cells each,
// from c0), and a tile takes over what its left neighbour left in LDS: the
// cells, midpoints and the face flux at its left end.  So the
// 5 midpoints and 10 cells that neighbouring tiles share are evaluated once
// per segment, where independent tiles evaluate them twice (a 256-cell pencil
// in 59-cell tiles fills 320 midpoint slots, in 64-cell tiles of one segment
// 261).
//
// Slots of a tile: cell c is the pencil's cell c0 - 5 + c, midpoint m sits
// between cells m + 2 and m + 3, face f between cells f + 4 and f + 5 and
// combines midpoints f .. f + 4.  In hybrid mode a midpoint is evaluated only
// if one of its faces m - 4 .. m has theta > 0; the weights of the faces
// behind the tile would cost four more cells and their logarithms, and tiles
// at a shock cost several times the others, so there a segment is one tile.
// The midpoints 0 .. 4 of such a tile belong to the tile before it too, and
// either may evaluate one that the other does not need.  So that a fallback
// there is counted once whatever the tiles, the left tile counts what it
// evaluates, and this one what the left one does not; the weights of the faces
// -4 .. -1 that this takes are evaluated for such a fallback only, behind the
// other phases (with every tile's other weights they cost 3% of a Hybrid
// residual, this way 1.5%).
#pragma once
#include "em_device.h"
#include "em_types.h"

namespace em {
namespace EM_VARIANT {

// LDS of one tile.  CF (cells fast): the pass axis is contiguous in memory;
// lanes then run along the cells and the rows of a pencil are contiguous
// (with the pencils fast, as on strided axes, the loads along the axis would
// hit the same banks 8 ways).
// CUT: pencils may be cut into several segments.
template <class Real, int MODE, int T_, int P_, bool CF, bool CUT_>
struct Tile {
    static constexpr int T = T_, P = P_;
    static constexpr bool CUT = CUT_;
    static constexpr bool HYB = MODE == MODE_HYBRID;
    static constexpr int HC = 10, HM = 5;  // slots taken over: cells, midpoints
    static constexpr int C = T + HC, M = T + HM, TH = T + 1;
    // a work item's slot and pencil: items [0, T P) are the tile's own slots
    // H .. H + T - 1, items [-H P, 0) the H slots before them
    template <int H>
    __device__ static __forceinline__ void item(int it, int& c, int& p) {
        constexpr int N = H > 0 ? H : 1;
        if (H == 0 || it >= 0) {
            c = H + (CF ? it % T : it / P);
            p = CF ? it / T : it % P;
        } else {
            it += H * P;
            c = CF ? it % N : it / P;
            p = CF ? it / N : it % P;
        }
    }
    __device__ static __forceinline__ int at(int c, int p) { return CF ? p * C + c : c * P + p; }
    __device__ static __forceinline__ int mt(int m, int p) { return CF ? p * M + m : m * P + p; }
    __device__ static __forceinline__ int tt(int f, int p) { return CF ? p * TH + f : f * P + p; }
    Real sw[5][C * P];  // primitives
    Real sre[C * P];    // rho_e of each cell
    Real sm[5][M * P];  // midpoint fluxes; then the flux of face f in slot f - 1
    Real sf[5][P];      // flux of face 0
    Real ss[2][HYB ? C * P : 1];
    Real sth[HYB ? TH * P : 1];
    unsigned late[HYB && CUT ? P : 1];  // fallbacks of the midpoints 0 .. 3 that late_fallbacks decides on
};

// lanes of the wave that satisfy c (called where the wave is whole)
__device__ __forceinline__ unsigned wave_count(bool c) { return (unsigned)__popcll(__ballot(c)); }

// Blend weight of a face from the sensors k of the six cells around it, read
// through ld(j, k)
template <class R, class LD>
__device__ __forceinline__ R blend_weight(R tol, LD&& ld) {
    R r = R(0.0);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        R q[6];
#pragma unroll
        for (int j = 0; j < 6; ++j) q[j] = ld(j, k);
        r = fmax(fmax(r, d4(q[0], q[1], q[2], q[3], q[4])), d4(q[1], q[2], q[3], q[4], q[5]));
    }
    R x = (r / tol - R(0.5)) / R(0.5);
    if (x < R(0.0)) x = R(0.0);
    if (x > R(1.0)) x = R(1.0);
    return isfinite(r) ? x * x * (R(3.0) - R(2.0) * x) : R(1.0);
}

// Counts the fallbacks in L.late that the tile before did not: those whose
// faces -4 .. -1 all have weight zero.  left_sensor(p, h, k) is sensor k of the
// cell h - 2 before pencil p's tile.  (Every thread calls it, after
// tile_faces; apart from the midpoints, whose loop it would slow down.)
template <class R, class TL, class SEN>
__device__ __forceinline__ void late_fallbacks(TL& L, int tid, R tol, unsigned (&scnt)[3], SEN&& left_sensor) {
    const unsigned late = tid < TL::P ? L.late[tid] : 0;
    if (late == 0) return;
    R x[2][2] = {};
#pragma unroll 1
    for (int i = 0; i < 4; ++i) {
        const R y = left_sensor(tid, i & 1, i >> 1);
        x[0][0] = i == 0 ? y : x[0][0];
        x[1][0] = i == 1 ? y : x[1][0];
        x[0][1] = i == 2 ? y : x[0][1];
        x[1][1] = y;
    }
    unsigned n = 0;
    bool zero = true;  // the weights of the faces f .. -1
#pragma unroll 1
    for (int f = -1; f >= -4; --f) {
        zero = zero && !(blend_weight(tol, [&](int j, int k) {
                             const int c = f + 2 + j;
                             return c == -2 ? x[0][k] : c == -1 ? x[1][k] : L.ss[k][TL::at(c, tid)];
                         }) > R(0.0));
        // midpoint m = f + 4 reaches down to face f
        n += zero && (late >> (f + 4) & 1) ? 1 : 0;
    }
    if (n) atomicAdd(&scnt[1], n);
}

// On entry (after a barrier): the tile's cells are in sw, sre and ss.  On
// exit (after a barrier): the flux of face f = 1 .. Tv is sm[k][mt(f - 1, p)],
// of face 0 sf[k][p].  first: nothing was taken over.  Counters of midpoints
// and faces owned by the segment (segments of one pencil share an end):
// shock-path faces are counted per wave (a scalar register), fallbacks and
// limited faces, which are few, in scnt[1] and scnt[2].  before_last() is
// called once the faces are in registers, ahead of the last two barriers: the
// place to issue the loads of the phase that follows.  zero1, zero2: the axes of the transverse velocities (D+1) % 3 and (D+2) % 3
// are inactive (see midpoint_flux_mid).
template <int D, int MODE, int NT, class R, class TL, class PRE>
__device__ __forceinline__ void tile_faces(TL& L, int tid, bool first, int Tv, int Pv, int c0, int s0, int s1, int nD,
                                           const EosT<R>& e, R lam, R tol, bool zero1, bool zero2,
                                           unsigned& n_shock, unsigned (&scnt)[3], PRE&& before_last) {
    constexpr int T = TL::T, P = TL::P;
    constexpr bool HYB = MODE == MODE_HYBRID;
    constexpr bool CEN = MODE == MODE_CENTRAL;
    static_assert(T * P <= NT, "one item per thread");
    auto& sw = L.sw;
    auto& sre = L.sre;
    auto& sm = L.sm;
    // ---- 2. hybrid blend weights (scheme.rs:171-183)
    if constexpr (HYB) {
        for (int it = tid - P; it < T * P; it += NT) {
            int f, p;
            TL::template item<1>(it, f, p);
            if (p >= Pv || f > Tv) continue;
            L.sth[TL::tt(f, p)] =
                blend_weight(tol, [&](int j, int k) { return L.ss[k][TL::at(f + 2 + j, p)]; });
        }
        __syncthreads();
    }

    // ---- 3. WCNS midpoints (midpoint m sits between cells c0-3+m and c0-2+m)
    if constexpr (!CEN) {
#pragma unroll 1
        for (int it = tid - (first ? TL::HM * P : 0); it < T * P; it += NT) {
            int m, p;
            TL::template item<TL::HM>(it, m, p);
            if (p >= Pv || m >= Tv + 5) continue;
            if constexpr (HYB) {
                bool need = false;
                const int flo = max(0, m - 4), fhi = min(Tv, m);
                for (int f = flo; f <= fhi; ++f) need = need || L.sth[TL::tt(f, p)] > R(0.0);
                if (!need) continue;
            }
            R f[5];
            bool fb = false, done = false;
            if constexpr (sizeof(R) == 8)
                done = midpoint_flux_mid<D>(e, zero1, zero2, [&](int j, int k) { return sw[k][TL::at(m + j, p)]; }, f);
            if (!done) {
                // read again from LDS: kept from above, the stencil would spill
                const int mo = sizeof(R) == 8 ? opaque(m) : m;
                fb = midpoint_flux<D, sizeof(R) == 8>(e, [&](int j, int k) { return sw[k][TL::at(mo + j, p)]; }, f);
            }
#pragma unroll
            for (int k = 0; k < 5; ++k) sm[k][TL::mt(m, p)] = f[k];
            if (fb) {
                // counted by one segment of the pencil
                const int j = c0 - 3 + m;  // global midpoint index
                bool own = (s0 == 0 || j >= s0) && (s1 == nD || j < s1);
                if constexpr (HYB && TL::CUT) {
                    // with a weight at face 0 the left tile has evaluated it
                    own = s0 == 0 || m >= 4 || L.sth[TL::tt(0, p)] > R(0.0);
                    if (!own) atomicOr(&L.late[p], 1u << m);
                    own = own && (s0 == 0 || m > 4 || !(L.sth[TL::tt(0, p)] > R(0.0)));
                }
                if (own) atomicAdd(&scnt[1], 1u);
            }
        }
        __syncthreads();
    }

    // ---- 4. face fluxes (face f between cells c0+f-1 and c0+f).  Face 0 of a
    // segment's first tile goes with the others if the threads suffice, else
    // before them; its flux has a place of its own, so only the tile's own
    // faces wait for the last midpoint read.
    constexpr bool ONE = (T + 1) * P <= NT;
    R fo[5];
    int ff = 0, fp = 0;
    bool mine = false;
    int n_own = 0;
#pragma unroll 1
    for (int pass = first && !ONE ? 0 : 1; pass < 2; ++pass) {
        const int it = pass == 0 || (first && ONE) ? tid - P : tid;
        if (it >= (pass == 0 ? 0 : T * P)) continue;
        int f, p;
        TL::template item<1>(it, f, p);
        if (p >= Pv || f > Tv) continue;
        // a face shared by two segments is counted by the one on its right
        const bool own_face = c0 + f < s1 || s1 == nD;
        R theta;
        if constexpr (MODE == MODE_WENO)
            theta = R(1.0);
        else if constexpr (CEN)
            theta = R(0.0);
        else
            theta = L.sth[TL::tt(f, p)];
        R cen[5] = {R(0.0), R(0.0), R(0.0), R(0.0), R(0.0)};
        if (theta < R(1.0)) {
            // KEEP-PE 6th-order central flux, scheme.rs:188-214
            const R a6[3] = {R(A6_0), R(A6_1), R(A6_2)};
#pragma unroll
            for (int li = 0; li < 3; ++li) {
                const int lag = li + 1;
#pragma unroll
                for (int mm = 0; mm < lag; ++mm) {
                    R wa[5], wb[5], ft[5];
#pragma unroll
                    for (int k = 0; k < 5; ++k) {
                        wa[k] = sw[k][TL::at(f + 4 - mm, p)];
                        wb[k] = sw[k][TL::at(f + 4 - mm + lag, p)];
                    }
                    split_flux_re<D>(wa, wb, sre[TL::at(f + 4 - mm, p)], sre[TL::at(f + 4 - mm + lag, p)], ft);
#pragma unroll
                    for (int k = 0; k < 5; ++k) cen[k] += R(2.0) * a6[li] * ft[k];
                }
            }
        }
        if (theta == R(0.0)) {
#pragma unroll
            for (int k = 0; k < 5; ++k) fo[k] = cen[k];
        } else {
            n_own += own_face ? 1 : 0;
            // F = sum_s S6[s] (F_{i+s} + F_{i-s}), order s=0, i+1, i-1, i+2, i-2
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                R v = R(0.0);
                v += R(S6_0) * sm[k][TL::mt(f + 2, p)];
                v += R(S6_1) * sm[k][TL::mt(f + 3, p)];
                v += R(S6_1) * sm[k][TL::mt(f + 1, p)];
                v += R(S6_2) * sm[k][TL::mt(f + 4, p)];
                v += R(S6_2) * sm[k][TL::mt(f, p)];
                fo[k] = v;
            }
            if (theta < R(1.0)) {
#pragma unroll
                for (int k = 0; k < 5; ++k) fo[k] = theta * fo[k] + (R(1.0) - theta) * cen[k];
            }
        }
        if (lam > R(0.0)) {
            // positivity limiter, scheme.rs:401-444
            R wl[5], wr[5], ul[5], ur[5], fl[5], fr[5];
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                wl[k] = sw[k][TL::at(f + 4, p)];
                wr[k] = sw[k][TL::at(f + 5, p)];
            }
            to_cons_re(wl, sre[TL::at(f + 4, p)], ul);
            to_cons_re(wr, sre[TL::at(f + 5, p)], ur);
            phys_flux<D>(wl, ul, fl);
            phys_flux<D>(wr, ur, fr);
            const R tl = R(2.0) * lam;
            R qa[5], qb[5];
            auto test_states = [&](const R* fx) {
#pragma unroll
                for (int k = 0; k < 5; ++k) {
                    qa[k] = ul[k] - tl * (fx[k] - fl[k]);
                    qb[k] = ur[k] + tl * (fx[k] - fr[k]);
                }
            };
            auto ok = [&](const R* fx) {
                R pa[5], pb[5];
                test_states(fx);
                to_prim(e, qa, pa);
                to_prim(e, qb, pb);
                return admissible(e, pa[0], pa[4]) && admissible(e, pb[0], pb[4]);
            };
            // almost every face is admissible by a wide margin, which needs
            // no division to see (a non-finite flux never passes)
            test_states(fo);
            bool pass = clearly_admissible(e, qa) && clearly_admissible(e, qb);
            if (!pass) {
                pass = true;
#pragma unroll
                for (int k = 0; k < 5; ++k) pass = pass && isfinite(fo[k]);
                pass = pass && ok(fo);
            }
            if (!pass) {
                constexpr int un = 1 + D;
                const R al = fmax(fabs(wl[un]) + sound_speed(e, wl[0], wl[4]),
                                       fabs(wr[un]) + sound_speed(e, wr[0], wr[4]));
                R flf[5], fh[5];
#pragma unroll
                for (int k = 0; k < 5; ++k) {
                    flf[k] = R(0.5) * (fl[k] + fr[k]) - R(0.5) * al * (ur[k] - ul[k]);
                    fh[k] = fo[k];
                }
                if (own_face) atomicAdd(&scnt[2], 1u);
                R lo = R(0.0), hi = R(1.0);
                for (int itb = 0; itb < 30; ++itb) {
                    const R mid = R(0.5) * (lo + hi);
                    R bl[5];
#pragma unroll
                    for (int k = 0; k < 5; ++k) bl[k] = isfinite(fh[k]) ? mid * fh[k] + (R(1.0) - mid) * flf[k] : flf[k];
                    if (ok(bl))
                        lo = mid;
                    else
                        hi = mid;
                }
#pragma unroll
                for (int k = 0; k < 5; ++k) fo[k] = isfinite(fh[k]) ? lo * fh[k] + (R(1.0) - lo) * flf[k] : flf[k];
            }
        }
        if (f == 0) {
#pragma unroll
            for (int k = 0; k < 5; ++k) L.sf[k][p] = fo[k];
        } else {
            mine = true;
            ff = f;
            fp = p;
        }
    }
    before_last();
    n_shock += wave_count(n_own & 1) + 2 * wave_count(n_own & 2);
    __syncthreads();  // every midpoint read is done: reuse sm for face fluxes
    // the midpoints T .. T + 4 that the next tile takes over stay
    if (mine) {
#pragma unroll
        for (int k = 0; k < 5; ++k) sm[k][TL::mt(ff - 1, fp)] = fo[k];
    }
    __syncthreads();
}

}  // namespace EM_VARIANT
}  // namespace em
