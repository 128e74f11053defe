// Launchers of the fused axis pass, one per arithmetic variant.
#pragma once
#include <hip/hip_runtime.h>

#include "em_amr_types.h"
#include "em_types.h"

namespace em {

// Tile shapes (cells along the axis x pencils, threads); index = cfg id, part
// of the interface (em_solver_set_tiles: a program may have stored one, so a
// changed table keeps the surviving shapes' indices and puts under the others
// shapes that are no slower than what stood there).  A strided pass reads P
// neighbouring cells of the innermost axis.  One thread per cell (T P == NT)
// suits segments of many tiles, one per midpoint ((T + 5) P == NT) those of
// one tile.
constexpr TileCfg kTileCfgs[] = {{32, 8, 256}, {64, 8, 512}, {59, 1, 64}, {27, 2, 64}, {27, 8, 256},
                                 {59, 4, 256}, {27, 4, 128}, {16, 16, 256}, {123, 4, 512}, {16, 4, 64}};
enum : int { TILE_32x8 = 0, TILE_59x1 = 2, TILE_27x2 = 3, TILE_27x8 = 4, TILE_59x4 = 5 };
constexpr int kNumTileCfgs = 10;
// a launch of more threads runs a part of them and reports no error
constexpr long long kMaxLaunchThreads = 0xffffffffll;

#define EM_DECLARE_LAUNCHERS                                                               \
    hipError_t launch_pass_hybrid(int d, int cfg, const PassArgs& a, hipStream_t s);      \
    hipError_t launch_pass_weno(int d, int cfg, const PassArgs& a, hipStream_t s);        \
    hipError_t launch_pass_central(int d, int cfg, const PassArgs& a, hipStream_t s);     \
    hipError_t launch_amr_hybrid(int d, int b, int shape, const AmrPassArgs& pa, unsigned grid, hipStream_t s); \
    hipError_t launch_amr_weno(int d, int b, int shape, const AmrPassArgs& pa, unsigned grid, hipStream_t s);   \
    hipError_t launch_amr_central(int d, int b, int shape, const AmrPassArgs& pa, unsigned grid, hipStream_t s); \
    inline hipError_t launch_amr_pass(int d, int mode, int b, int shape, const AmrPassArgs& pa,       \
                                      unsigned grid, hipStream_t s) {                                \
        switch (mode) {                                                                    \
            case MODE_HYBRID: return launch_amr_hybrid(d, b, shape, pa, grid, s);          \
            case MODE_WENO: return launch_amr_weno(d, b, shape, pa, grid, s);              \
            case MODE_CENTRAL: return launch_amr_central(d, b, shape, pa, grid, s);        \
            default: return hipErrorInvalidValue;                                          \
        }                                                                                  \
    }                                                                                      \
    hipError_t launch_amr32_hybrid(int d, int b, int shape, const AmrPassArgsT<float>& pa, unsigned grid,  \
                                   hipStream_t s);                                                          \
    hipError_t launch_amr32_weno(int d, int b, int shape, const AmrPassArgsT<float>& pa, unsigned grid,    \
                                 hipStream_t s);                                                            \
    hipError_t launch_amr32_central(int d, int b, int shape, const AmrPassArgsT<float>& pa, unsigned grid, \
                                    hipStream_t s);                                                         \
    inline hipError_t launch_amr_pass(int d, int mode, int b, int shape, const AmrPassArgsT<float>& pa,    \
                                      unsigned grid, hipStream_t s) {                                      \
        switch (mode) {                                                                    \
            case MODE_HYBRID: return launch_amr32_hybrid(d, b, shape, pa, grid, s);        \
            case MODE_WENO: return launch_amr32_weno(d, b, shape, pa, grid, s);            \
            case MODE_CENTRAL: return launch_amr32_central(d, b, shape, pa, grid, s);      \
            default: return hipErrorInvalidValue;                                          \
        }                                                                                  \
    }                                                                                      \
    hipError_t launch_amr_multi_hybrid(int d, const AmrMultiArgs& m, unsigned grid, hipStream_t s);   \
    hipError_t launch_amr_multi_weno(int d, const AmrMultiArgs& m, unsigned grid, hipStream_t s);     \
    hipError_t launch_amr_multi_central(int d, const AmrMultiArgs& m, unsigned grid, hipStream_t s);  \
    inline hipError_t launch_amr_multi(int d, int mode, const AmrMultiArgs& m, unsigned grid, hipStream_t s) { \
        switch (mode) {                                                                    \
            case MODE_HYBRID: return launch_amr_multi_hybrid(d, m, grid, s);               \
            case MODE_WENO: return launch_amr_multi_weno(d, m, grid, s);                   \
            case MODE_CENTRAL: return launch_amr_multi_central(d, m, grid, s);             \
            default: return hipErrorInvalidValue;                                          \
        }                                                                                  \
    }                                                                                      \
    hipError_t launch_ens_hybrid(int d, int cfg, const EnsPassArgs& e, unsigned grid, hipStream_t s); \
    hipError_t launch_ens_weno(int d, int cfg, const EnsPassArgs& e, unsigned grid, hipStream_t s);   \
    hipError_t launch_ens_central(int d, int cfg, const EnsPassArgs& e, unsigned grid, hipStream_t s); \
    inline hipError_t launch_ens_pass(int d, int mode, int cfg, const EnsPassArgs& e, unsigned grid,  \
                                      hipStream_t s) {                                               \
        switch (mode) {                                                                    \
            case MODE_HYBRID: return launch_ens_hybrid(d, cfg, e, grid, s);                \
            case MODE_WENO: return launch_ens_weno(d, cfg, e, grid, s);                    \
            case MODE_CENTRAL: return launch_ens_central(d, cfg, e, grid, s);              \
            default: return hipErrorInvalidValue;                                          \
        }                                                                                  \
    }                                                                                      \
    inline hipError_t launch_pass(int d, int mode, int cfg, const PassArgs& a, hipStream_t s) { \
        switch (mode) {                                                                    \
            case MODE_HYBRID: return launch_pass_hybrid(d, cfg, a, s);                     \
            case MODE_WENO: return launch_pass_weno(d, cfg, a, s);                         \
            case MODE_CENTRAL: return launch_pass_central(d, cfg, a, s);                   \
            default: return hipErrorInvalidValue;                                          \
        }                                                                                  \
    }                                                                                      \
    hipError_t launch_pass32_hybrid(int d, int cfg, const PassArgsT<float>& a, hipStream_t s); \
    hipError_t launch_pass32_weno(int d, int cfg, const PassArgsT<float>& a, hipStream_t s);   \
    hipError_t launch_pass32_central(int d, int cfg, const PassArgsT<float>& a, hipStream_t s); \
    inline hipError_t launch_pass(int d, int mode, int cfg, const PassArgsT<float>& a, hipStream_t s) { \
        switch (mode) {                                                                    \
            case MODE_HYBRID: return launch_pass32_hybrid(d, cfg, a, s);                   \
            case MODE_WENO: return launch_pass32_weno(d, cfg, a, s);                       \
            case MODE_CENTRAL: return launch_pass32_central(d, cfg, a, s);                 \
            default: return hipErrorInvalidValue;                                          \
        }                                                                                  \
    }

namespace precise {
EM_DECLARE_LAUNCHERS
}
namespace fast {
EM_DECLARE_LAUNCHERS
}

}  // namespace em
