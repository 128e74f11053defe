// Conversion between a solver's device layout (interior cells, variable-major
// planes of ncell values) and the host layout of the C ABI (ghost-padded
// cells, NV doubles each), on the device: the host copies bytes only.
//
// Bound by the host link (17 to 28 GB/s for pageable memory here; the kernels
// run at several TB/s).  The strided single-thread loops this replaces took
// about 25 ms each way for a 128^3 state (110 MB in the host layout), against
// 4 to 7 ms of copying.  Large arrays go through a buffer of at most
// kHostIoBytes in pieces, so the extra device memory is bounded.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

namespace em {

constexpr size_t kHostIoBytes = 256u << 20;

// Padded extents and ghost offsets of a mesh (int: a padded plane index fits)
struct HostLayout {
    long long n0, n1, n2;  // interior extents
    int m1, m2;            // padded extents of the inner axes
    int g0, g1, g2;        // ghost offsets
    long long ncell, len;  // interior and padded cells
    // interior index of padded cell q, or -1
    __device__ __forceinline__ long long interior(long long q) const {
        const long long i = q / ((long long)m1 * m2) - g0, j = (q / m2) % m1 - g1, k = q % m2 - g2;
        return i >= 0 && i < n0 && j >= 0 && j < n1 && k >= 0 && k < n2 ? (i * n1 + j) * n2 + k : -1;
    }
};

// padded cells [q0, q0 + cnt): host layout in io -> interior planes of dev
template <int NV, class Real>
__global__ __launch_bounds__(256) void k_host_in(const double* __restrict__ io, HostLayout h, long long q0,
                                                 long long cnt, Real* __restrict__ dev) {
    const long long t = blockIdx.x * 256ll + threadIdx.x;
    if (t >= cnt) return;
    const long long c = h.interior(q0 + t);
    if (c < 0) return;
#pragma unroll
    for (int v = 0; v < NV; ++v) dev[v * h.ncell + c] = Real(io[t * NV + v]);
}

// the reverse; padded: dev holds padded planes (len values each), else
// interior planes and the ghosts are written as zero
template <int NV, class Real>
__global__ __launch_bounds__(256) void k_host_out(const Real* __restrict__ dev, HostLayout h, int padded, long long q0,
                                                  long long cnt, double* __restrict__ io) {
    const long long t = blockIdx.x * 256ll + threadIdx.x;
    if (t >= cnt) return;
    const long long c = padded ? q0 + t : h.interior(q0 + t);
    const long long plane = padded ? h.len : h.ncell;
#pragma unroll
    for (int v = 0; v < NV; ++v) io[t * NV + v] = c < 0 ? 0.0 : (double)dev[v * plane + c];
}

// The buffer and the two transfers of one solver (not thread-safe, like its
// handle).  Both leave the stream idle, also on an error: the host array is
// free on return.
template <int NV>
struct HostIo {
    double* buf = nullptr;
    long long cells = 0;           // capacity
    size_t limit = kHostIoBytes;  // of the buffer

    HostIo() = default;
    HostIo(const HostIo&) = delete;
    ~HostIo() {
        if (buf) (void)hipFree(buf);
    }
    hipError_t reserve(const HostLayout& h) {
        const long long want = std::min<long long>(h.len, (long long)(limit / (8 * NV)));
        if (cells >= want) return hipSuccess;
        const hipError_t e = hipMalloc(&buf, sizeof(double) * NV * want);
        if (e == hipSuccess) cells = want;
        return e;
    }
    static hipError_t finish(hipError_t e, hipStream_t s) {
        const hipError_t f = hipStreamSynchronize(s);
        return e == hipSuccess ? f : e;
    }
    template <class Real>
    hipError_t in(const HostLayout& h, const double* host, Real* dev, hipStream_t s) {
        hipError_t e = reserve(h);
        for (long long q0 = 0; e == hipSuccess && q0 < h.len; q0 += cells) {
            const long long cnt = std::min(cells, h.len - q0);
            e = hipMemcpyAsync(buf, host + q0 * NV, sizeof(double) * NV * cnt, hipMemcpyHostToDevice, s);
            if (e != hipSuccess) break;
            hipLaunchKernelGGL((k_host_in<NV, Real>), dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, s, buf, h, q0, cnt,
                               dev);
            e = hipGetLastError();
        }
        return finish(e, s);
    }
    template <class Real>
    hipError_t out(const HostLayout& h, const Real* dev, bool padded, double* host, hipStream_t s) {
        hipError_t e = reserve(h);
        for (long long q0 = 0; e == hipSuccess && q0 < h.len; q0 += cells) {
            const long long cnt = std::min(cells, h.len - q0);
            hipLaunchKernelGGL((k_host_out<NV, Real>), dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, s, dev, h,
                               padded ? 1 : 0, q0, cnt, buf);
            e = hipGetLastError();
            if (e == hipSuccess)
                e = hipMemcpyAsync(host + q0 * NV, buf, sizeof(double) * NV * cnt, hipMemcpyDeviceToHost, s);
        }
        return finish(e, s);
    }
};

}  // namespace em
