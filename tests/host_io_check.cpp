// em_hostio.h on the CPU: transfers in pieces that split rows and leave a
// remainder, by the device and by the host loops, without memory for the
// buffer, and the stream after a failed copy.  Prints what differs; exit
// status 1 if anything does.
#include "em_hostio.h"

#include <cstdio>
#include <random>
#include <vector>

using namespace em;

static int failures = 0;
static void check(bool ok, const char* what, long long a = 0, long long b = 0) {
    if (ok) return;
    if (failures++ < 10) std::printf("%s (%lld, %lld)\n", what, a, b);
}

static HostLayout layout(int n0, int n1, int n2, int ng) {
    auto m = [&](int n) { return n > 1 ? n + 2 * ng : 1; };
    auto g = [&](int n) { return n > 1 ? ng : 0; };
    return HostLayout{n0, n1, n2, m(n1), m(n2), g(n0), g(n1), g(n2), (long long)n0 * n1 * n2, (long long)m(n0) * m(n1) * m(n2)};
}

// one mesh through every transfer: route 0 with a buffer of `limit` bytes, 1
// the host loops, 2 as the solvers call it
template <int NV, class Real>
static void round_trip(const HostLayout& h, size_t limit, int route) {
    std::mt19937_64 rng(3);
    std::uniform_real_distribution<double> uni(-2.0, 2.0);
    std::vector<double> host(NV * h.len), back(NV * h.len, 7.0);
    for (double& x : host) x = uni(rng);
    HostIo<NV> io;
    io.limit = limit;
    std::vector<Real> dev(NV * h.ncell, Real(5)), pad(NV * h.len);
    auto in = [&](const double* u, Real* d) {
        return route == 0 ? io.in_by_device(h, u, d, nullptr) : route == 1 ? io.in_by_host(h, u, d, nullptr) : io.in(h, u, d, nullptr);
    };
    auto out = [&](const Real* d, bool padded, double* u) {
        return route == 0   ? io.out_by_device(h, d, padded, u, nullptr)
               : route == 1 ? io.out_by_host(h, d, padded, u, nullptr)
                            : io.out(h, d, padded, u, nullptr);
    };
    check(in(host.data(), dev.data()) == hipSuccess && !stub.pending, "in");
    for (long long q = 0; q < h.len; ++q) {
        const long long c = h.interior(q);
        for (int v = 0; v < NV; ++v) {
            if (c >= 0) check(dev[v * h.ncell + c] == Real(host[q * NV + v]), "value in", q, v);
            pad[v * h.len + q] = Real(uni(rng));
        }
    }
    check(out(dev.data(), false, back.data()) == hipSuccess && !stub.pending, "out");
    for (long long q = 0; q < h.len; ++q) {
        const long long c = h.interior(q);
        for (int v = 0; v < NV; ++v) check(back[q * NV + v] == (c < 0 ? 0.0 : (double)dev[v * h.ncell + c]), "value out", q, v);
    }
    check(out(pad.data(), true, back.data()) == hipSuccess && !stub.pending, "out, padded");
    for (long long q = 0; q < h.len; ++q)
        for (int v = 0; v < NV; ++v) check(back[q * NV + v] == (double)pad[v * h.len + q], "value out, padded", q, v);
}

// a copy fails after others were queued: the error comes back, and nothing is
// left running on the caller's array
template <int NV>
static void failed_copies(const HostLayout& h, size_t limit) {
    std::vector<double> host(NV * h.len), dev(NV * h.ncell), pad(NV * h.len);
    for (int fail = 0; fail < 3; ++fail)
        for (int what = 0; what < 3; ++what) {
            HostIo<NV> io;
            io.limit = limit;
            stub = StubState{};
            stub.fail_copy = fail;
            const hipError_t e = what == 0   ? io.in_by_device(h, host.data(), dev.data(), nullptr)
                                 : what == 1 ? io.out_by_device(h, dev.data(), false, host.data(), nullptr)
                                             : io.out_by_device(h, pad.data(), true, host.data(), nullptr);
            check(e == (stub.copies > fail ? hipErrorUnknown : hipSuccess), "error of a failed copy", fail, what);
            check(!stub.pending, "work left on the stream after an error", fail, what);
        }
    stub = StubState{};
}

int main() {
    const int sizes[][3] = {{40, 1, 1}, {1, 1, 33}, {9, 14, 1}, {1, 7, 12}, {5, 6, 7}, {2, 3, 11}};
    for (auto& n : sizes) {
        const HostLayout h = layout(n[0], n[1], n[2], 6);
        for (size_t cells : {1u << 20, 64u, 37u, 5u}) {
            round_trip<5, double>(h, cells * 40, 0);
            round_trip<5, float>(h, cells * 40, 0);
            round_trip<7, double>(h, cells * 56, 0);
            round_trip<7, float>(h, cells * 56, 0);
        }
        for (int route : {1, 2}) {
            round_trip<5, double>(h, kHostIoBytes, route);
            round_trip<5, float>(h, kHostIoBytes, route);
            round_trip<7, double>(h, kHostIoBytes, route);
            round_trip<7, float>(h, kHostIoBytes, route);
        }
    }
    // the ghosts of thin and small meshes stay off the link and no buffer is
    // kept; a box is converted on the device, also without memory for it
    for (auto& n : {layout(1000, 4, 4, 6), layout(2, 200, 300, 6), layout(16, 16, 16, 6), layout(33, 47, 1, 6)}) {
        stub = StubState{};
        std::vector<double> host(5 * n.len), dev(5 * n.ncell);
        HostIo<5> io;
        io.in(n, host.data(), dev.data(), nullptr);
        check(stub.bytes == 40 * (size_t)n.ncell && stub.mallocs == 0, "thin or small mesh in", n.n0, n.n1);
        io.out(n, dev.data(), false, host.data(), nullptr);
        check(stub.bytes == 80 * (size_t)n.ncell && stub.mallocs == 0, "thin or small mesh out", n.n0, n.n1);
    }
    const HostLayout box = layout(96, 96, 96, 6);
    stub = StubState{};
    round_trip<5, double>(box, kHostIoBytes, 2);
    check(stub.mallocs == 1, "box by the device");
    stub = StubState{};
    stub.malloc_limit = 1000;
    round_trip<5, double>(box, kHostIoBytes, 2);
    check(stub.mallocs == 0, "box without memory");
    stub = StubState{};
    failed_copies<5>(layout(40, 30, 20, 6), 40 * 4000);
    std::printf(failures ? "%d FAILURES\n" : "ok\n", failures);
    return failures ? 1 : 0;
}
