// Stand-in for <hip/hip_runtime.h> that lets a plain C++ compiler build the
// device headers for the CPU, so that their arithmetic and their host-side
// paths are tested without a GPU.  One lane per wave.  The hardware's
// approximate reciprocals are modelled by the exact ones cut to 26 bits, but
// for operands a few ulps from a power of two: two Newton steps from a cut
// value can end an ulp off there, which the hardware's division was measured
// not to do.
#pragma once
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <cstring>

#define __device__
#define __host__
#define __global__
#define __shared__
#define __forceinline__ inline
#define __launch_bounds__(...)
using std::isfinite;

inline double stub_cut(double x) {
    std::uint64_t b;
    std::memcpy(&b, &x, 8);
    b &= ~((std::uint64_t(1) << 27) - 1);
    std::memcpy(&x, &b, 8);
    return x;
}
inline double stub_rcp(double x) {
    std::uint64_t b;
    std::memcpy(&b, &x, 8);
    b += 8;
    return (b & ((std::uint64_t(1) << 52) - 1)) < 16 ? 1.0 / x : stub_cut(1.0 / x);
}
inline double stub_rsq(double x) { return stub_cut(1.0 / std::sqrt(x)); }
// v_div_fixup_f64: the special cases of den and num, else q with their sign;
// a NaN quotient of ordinary operands is taken for an overflow
inline double stub_fixup(double q, double den, double num) {
    const double s = std::copysign(1.0, den) * std::copysign(1.0, num);
    if (std::isnan(den) || std::isnan(num)) return NAN;
    if ((den == 0.0 && num == 0.0) || (std::isinf(den) && std::isinf(num))) return NAN;
    if (den == 0.0 || std::isinf(num)) return std::copysign(INFINITY, s);
    if (num == 0.0 || std::isinf(den)) return std::copysign(0.0, s);
    return std::copysign(std::isnan(q) ? INFINITY : std::fabs(q), s);
}
#define __builtin_amdgcn_rcp stub_rcp
#define __builtin_amdgcn_rsq stub_rsq
#define __builtin_amdgcn_div_fixup stub_fixup
#define __builtin_amdgcn_readfirstlane(x) (x)
inline int __double2hiint(double x) {
    std::uint64_t b;
    std::memcpy(&b, &x, 8);
    return (int)(b >> 32);
}
inline int __double2loint(double x) {
    std::uint64_t b;
    std::memcpy(&b, &x, 8);
    return (int)(b & 0xffffffffu);
}
inline double __hiloint2double(int hi, int lo) {
    const std::uint64_t b = (std::uint64_t)(std::uint32_t)hi << 32 | (std::uint32_t)lo;
    double x;
    std::memcpy(&x, &b, 8);
    return x;
}
inline long long __double_as_longlong(double x) {
    long long b;
    std::memcpy(&b, &x, 8);
    return b;
}
inline int __any(unsigned x) { return x != 0; }
template <class T>
inline T max(T a, T b) {
    return a > b ? a : b;
}
template <class T>
inline T min(T a, T b) {
    return a < b ? a : b;
}

// ---- the runtime calls of em_hostio.h: device memory is host memory, a
// kernel launch runs its threads in turn
typedef int hipError_t;
typedef void* hipStream_t;
constexpr hipError_t hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999;
enum { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
struct dim3 {
    unsigned x;
    explicit dim3(unsigned v) : x(v) {}
};
inline dim3 blockIdx(0), threadIdx(0);
// what the tests watch and force
struct StubState {
    size_t malloc_limit = (size_t)-1;  // larger requests fail
    int fail_copy = -1;                // the copy of this index fails
    int copies = 0, mallocs = 0, frees = 0;
    bool pending = false;              // work queued since the last synchronisation
    size_t bytes = 0;                  // copied
};
inline StubState stub;
template <class T>
inline hipError_t hipMalloc(T** p, size_t n) {
    if (n > stub.malloc_limit) return hipErrorOutOfMemory;
    stub.mallocs++;
    *p = (T*)std::malloc(n);
    return hipSuccess;
}
inline hipError_t hipFree(void* p) {
    stub.frees++;
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) {
    if (stub.copies++ == stub.fail_copy) return hipErrorUnknown;
    std::memcpy(d, s, n);
    stub.bytes += n;
    stub.pending = true;
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) {
    stub.pending = false;
    return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
template <class K, class... A>
inline void stub_launch(K k, dim3 grid, dim3 block, A... a) {
    for (blockIdx.x = 0; blockIdx.x < grid.x; ++blockIdx.x)
        for (threadIdx.x = 0; threadIdx.x < block.x; ++threadIdx.x) k(a...);
    stub.pending = true;
}
#define hipLaunchKernelGGL(k, grid, block, lds, stream, ...) stub_launch(k, grid, block, __VA_ARGS__)
