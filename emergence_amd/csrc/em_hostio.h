// Conversion between a solver's device layout (interior cells, variable-major
// planes of ncell values) and the host layout of the C ABI (ghost-padded
// cells, NV doubles each).
//
// Large states are converted on the device, so that the host copies bytes
// only: bound by the host link (17 to 28 GB/s for pageable memory here; the
// kernels run at several TB/s).  The strided single-thread loops took about
// 25 ms each way for a 128^3 state (110 MB in the host layout), the copies
// take 4 to 7 ms.  Large arrays go through a buffer of at most kHostIoBytes in
// pieces, so the extra device memory is bounded.
//
// The device path moves the ghosts over the link too and needs a kernel more.
// States that fit the host's caches are converted in a loop on the host where
// that is faster (HostIo::..._on_host): small ones, and thin meshes, whose
// padded array is many times the interior.  It also serves where the buffer
// cannot be had.  In microseconds, host loop / device:
//   in:  33x47 15/27, 64x64 23/31, 16^3 19/53, 1000x4x4 61/310,
//        2x200x300 328/1291, 4x40000 515/727, 512^2 833/339
//   out (seven variables): 64x48 25/36, 40x30x20 179/242, 1000x4x4 180/832
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <vector>

namespace em {

constexpr size_t kHostIoBytes = 256u << 20;
// interior bytes up to which the host loops stay in the caches (12 to 17 GB/s;
// 3.5 GB/s at 40 MB)
constexpr double kHostLoopBytes = 8e6;

// Padded extents and ghost offsets of a mesh (int: a padded plane index fits)
struct HostLayout {
    long long n0, n1, n2;  // interior extents
    int m1, m2;            // padded extents of the inner axes
    int g0, g1, g2;        // ghost offsets
    long long ncell, len;  // interior and padded cells
    // f(padded index, interior index) of the first cell of every interior row
    template <class F>
    void for_rows(F&& f) const {
        for (long long i = 0; i < n0; ++i)
            for (long long j = 0; j < n1; ++j) f(((i + g0) * m1 + (j + g1)) * m2 + g2, (i * n1 + j) * n2);
    }
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

// The buffer and the two transfers of one solver, or of an ensemble's instances
// (whose transfers may come from several threads).  Both leave the stream idle, also on an error: the host array is
// free on return.
template <int NV>
struct HostIo {
    std::mutex lock;  // of the buffer
    double* buf = nullptr;
    long long cells = 0;           // capacity
    size_t limit = kHostIoBytes;  // of the buffer

    HostIo() = default;
    HostIo(const HostIo&) = delete;
    ~HostIo() {
        if (buf) (void)hipFree(buf);
    }
    static hipError_t finish(hipError_t e, hipStream_t s) {
        const hipError_t f = hipStreamSynchronize(s);
        return e == hipSuccess ? f : e;
    }
    // false: no memory for the buffer
    bool reserve(const HostLayout& h) {
        const long long want = std::min<long long>(h.len, (long long)(limit / (8 * NV)));
        if (cells >= want) return true;
        if (buf) (void)hipFree(buf);
        buf = nullptr;
        cells = 0;
        if (hipMalloc(&buf, sizeof(double) * NV * want) != hipSuccess) {
            (void)hipGetLastError();
            buf = nullptr;
            return false;
        }
        cells = want;
        return true;
    }
    // Which side converts, by the time of either (microseconds, bytes per
    // microsecond).  in: a loop over the interior at 16 GB/s (23 in float, half
    // the bytes to write and copy) against the whole padded array at 30 GB/s
    // and a kernel.  The loop's staging array is new memory for each call where
    // it is large: page faults at 16 GB/s (with them left out of the rule,
    // 20 steps of a 65x99x27 state between upload and download took 6.7
    // against 6.2 ms)
    static double faults(double staged) { return std::max(0.0, staged - 1e6) / 16e3; }
    template <class Real>
    static bool in_on_host(const HostLayout& h) {
        const double ib = 8.0 * NV * h.ncell, pb = 8.0 * NV * h.len;
        return ib <= kHostLoopBytes &&
               10.0 + ib / (sizeof(Real) == 4 ? 23e3 : 16e3) + faults(ib * sizeof(Real) / 8.0) < 20.0 + pb / 30e3;
    }
    // out: interior planes are copied at 17 GB/s and scattered (8.2 together,
    // 15 in float) into zeros, or the padded array copied at 17.5; padded
    // planes of doubles lose the transposition at 37 GB/s but save a kernel, in
    // float they are half the bytes
    template <class Real>
    static bool out_on_host(const HostLayout& h, bool padded) {
        const double ib = 8.0 * NV * h.ncell, pb = 8.0 * NV * h.len;
        const double device = pb / 17.5e3, fault = faults((padded ? pb : ib) * sizeof(Real) / 8.0);
        if (padded) return pb / (sizeof(Real) == 4 ? 27e3 : 11.9e3) + fault < 5.0 + device;
        return ib <= kHostLoopBytes &&
               10.0 + ib / (sizeof(Real) == 4 ? 15e3 : 8.2e3) + fault + pb / 200e3 < 24.0 + device;
    }
    template <class Real>
    hipError_t in_by_host(const HostLayout& h, const double* host, Real* dev, hipStream_t s) {
        // a cleared array for each call: the clearing brings its lines into the
        // caches (an uncleared or a kept one took up to twice the time)
        std::vector<Real> t(NV * h.ncell);
        Real* const p = t.data();
        const long long nc = h.ncell, n2 = h.n2;
        h.for_rows([=](long long q, long long c) {
            const double* u = host + q * NV;
            for (long long k = 0; k < n2; ++k, u += NV)
                for (int v = 0; v < NV; ++v) p[v * nc + c + k] = Real(u[v]);
        });
        return finish(hipMemcpyAsync(dev, t.data(), sizeof(Real) * NV * h.ncell, hipMemcpyHostToDevice, s), s);
    }
    template <class Real>
    hipError_t out_by_host(const HostLayout& h, const Real* dev, bool padded, double* host, hipStream_t s) {
        const long long plane = padded ? h.len : h.ncell;
        std::vector<Real> t(NV * plane);
        const hipError_t e = finish(hipMemcpyAsync(t.data(), dev, sizeof(Real) * NV * plane, hipMemcpyDeviceToHost, s), s);
        if (e != hipSuccess) return e;
        if (padded) {
            for (long long q = 0; q < h.len; ++q)
                for (int v = 0; v < NV; ++v) host[q * NV + v] = (double)t[v * plane + q];
            return e;
        }
        std::fill(host, host + NV * h.len, 0.0);
        const Real* const p = t.data();
        const long long n2 = h.n2;
        h.for_rows([=](long long q, long long c) {
            double* u = host + q * NV;
            for (long long k = 0; k < n2; ++k, u += NV)
                for (int v = 0; v < NV; ++v) u[v] = (double)p[v * plane + c + k];
        });
        return e;
    }
    template <class Real>
    hipError_t in(const HostLayout& h, const double* host, Real* dev, hipStream_t s) {
        return in_on_host<Real>(h) ? in_by_host(h, host, dev, s) : in_by_device(h, host, dev, s);
    }
    template <class Real>
    hipError_t out(const HostLayout& h, const Real* dev, bool padded, double* host, hipStream_t s) {
        return out_on_host<Real>(h, padded) ? out_by_host(h, dev, padded, host, s) : out_by_device(h, dev, padded, host, s);
    }
    template <class Real>
    hipError_t in_by_device(const HostLayout& h, const double* host, Real* dev, hipStream_t s) {
        const std::lock_guard<std::mutex> hold(lock);
        if (!reserve(h)) return in_by_host(h, host, dev, s);
        hipError_t e = hipSuccess;
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
    hipError_t out_by_device(const HostLayout& h, const Real* dev, bool padded, double* host, hipStream_t s) {
        const std::lock_guard<std::mutex> hold(lock);
        if (!reserve(h)) return out_by_host(h, dev, padded, host, s);
        hipError_t e = hipSuccess;
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
