// The mid-range forms of em_device.h on the CPU against the general
// expressions, bit for bit, over random operands and the edges of every range
// test.  Prints one line per mismatch kind; exit status 1 if there is any.
#include <cstdio>
#include <random>

#include "em_device.h"

using namespace em;

static int failures = 0;
static bool same(double a, double b) {
    return (std::isnan(a) && std::isnan(b)) || __double_as_longlong(a) == __double_as_longlong(b);
}
static void report(const char* what, const double* in, int n, double got, double want) {
    if (failures++ >= 8) return;
    std::printf("%s: got %a, want %a for", what, got, want);
    for (int i = 0; i < n; ++i) std::printf(" %a", in[i]);
    std::printf("\n");
}

static std::mt19937_64 rng(7);
static double uni(double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); }
static int pick(int n) { return (int)(rng() % n); }
// a value of the kinds the passes meet: ordinary, zero of either sign, any
// exponent, near-integer mantissas
static double value(bool wide) {
    switch (pick(wide ? 8 : 5)) {
        case 0: return 0.0;
        case 1: return -0.0;
        case 2: return uni(-2.0, 2.0);
        case 3: return std::nextafter((double)(1 + pick(4)), pick(2) ? 0.0 : 9.0);
        case 4: return uni(-2.0, 2.0) * std::exp2(pick(60) - 40);
        case 5: return uni(-2.0, 2.0) * std::exp2(pick(400) - 200);
        case 6: return uni(-2.0, 2.0) * std::exp2(pick(2000) - 1000);
        default: return uni(-1.0, 1.0) * 1e-310;
    }
}

static const Eos gases[] = {Eos{1.4, 0, 0, 0}, Eos{5.0 / 3.0, 0, 0, 0}, Eos{4.4, 0.6, 0, 0.1}, Eos{1.3, 0.2, 0.3, 0},
                            Eos{1.3, 0.2, 0.3, -0.1}};

static void check_to_prim(int n) {
    for (int i = 0; i < n; ++i) {
        const Eos e = gases[pick(5)];
        const bool wide = pick(4) == 0;
        double u[5] = {std::fabs(value(wide)), value(wide), value(wide), value(wide), value(wide)};
        if (pick(2)) u[0] = uni(0.1, 3.0), u[4] = uni(0.1, 9.0);
        double w[5], g[5], v;
        to_prim_v(e, u, w, v);
        to_prim(e, u, g);
        for (int k = 0; k < 5; ++k)
            if (!same(w[k], g[k])) report("to_prim", u, 5, w[k], g[k]);
        if (!same(v, 1.0 / u[0])) report("1 / rho", u, 1, v, 1.0 / u[0]);
        const double x = eos_rho_e_v(e, g[0], g[4], v), y = eos_rho_e(e, g[0], g[4]);
        if (!same(x, y)) report("rho_e", u, 5, x, y);
    }
}

static void pair_case(const double v[6], long long& taken) {
    double l, r;
    unsigned top = 0;
    bool ok = true;
    weno5z_pair<true>(v, l, r, top, ok);
    if (!ok || top >= top_word(Mid<double>::beta_max) || !isfinite(l + r)) return;
    ++taken;
    const double a = weno5z_interp(v[0], v[1], v[2], v[3], v[4]), b = weno5z_interp(v[5], v[4], v[3], v[2], v[1]);
    if (!same(0.125 * l, a)) report("weno left", v, 6, 0.125 * l, a);
    if (!same(0.125 * r, b)) report("weno right", v, 6, 0.125 * r, b);
}

static void check_pairs(int n) {
    long long taken = 0;
    for (int i = 0; i < n; ++i) {
        double v[6];
        const int kind = pick(5);
        const double c = uni(0.5, 2.0) * std::exp2(kind < 2 ? pick(8) - 4 : pick(500) - 250);
        for (double& x : v) {
            if (kind == 0) x = c * (1.0 + 0.1 * uni(-1, 1));
            else if (kind == 1) x = c;
            else if (kind == 2) x = uni(-2, 2) * c;
            else if (kind == 3) x = value(true);
            else x = value(false);
        }
        // one outlier beside an exactly flat stencil
        if (kind == 1) v[pick(6)] = uni(-1, 1) * c * std::exp2(pick(60) - 20);
        pair_case(v, taken);
    }
    // flat stencils with one outlier of every size, either end
    for (int ec = -300; ec <= 300; ec += 3)
        for (int ej = -300; ej <= 600; ej += 3)
            for (int pos = 0; pos < 6; ++pos) {
                double v[6];
                for (double& x : v) x = 1.25 * std::exp2(ec);
                v[pos] = 1.5 * std::exp2(ej);
                pair_case(v, taken);
            }
    std::printf("weno pairs taken in the mid range: %lld\n", taken);
    if (taken < n / 4) ++failures;
}

template <int D>
static void check_midpoints(int n) {
    long long taken = 0, refused = 0;
    for (int i = 0; i < n; ++i) {
        const Eos e = gases[pick(5)];
        double s[6][5];
        const int kind = pick(6);
        const double rho = uni(0.2, 2.0), p = uni(0.2, 2.0);
        const bool rest = pick(3) == 0;
        for (auto& w : s) {
            const double a = kind == 1 ? 0.0 : kind == 2 ? 0.9 : 0.1;
            w[0] = rho * (1.0 + a * uni(-1, 1));
            w[4] = p * (1.0 + a * uni(-1, 1));
            for (int k = 1; k < 4; ++k) w[k] = rest ? value(kind == 5) : uni(-1, 1) * (kind == 3 ? 8.0 : 1.0);
            if (kind == 4) w[0] *= std::exp2(pick(20) - 10), w[4] *= std::exp2(pick(20) - 10);
        }
        if (e.b > 0.0)
            for (auto& w : s) w[0] *= 0.5;
        auto ld = [&](int j, int k) { return s[j][k]; };
        double f[5], g[5];
        if (!midpoint_flux_mid<D>(e, false, false, ld, f)) {
            ++refused;
            continue;
        }
        ++taken;
        const bool fb = midpoint_flux<D, true>(e, ld, g);
        if (fb) report("fallback taken in the mid range", &s[0][0], 30, 1, 0);
        for (int k = 0; k < 5; ++k)
            if (!same(f[k], g[k])) report("midpoint flux", &s[0][0], 30, f[k], g[k]);
    }
    std::printf("midpoints along %d taken in the mid range: %lld, refused: %lld\n", D, taken, refused);
    if (taken < n / 4) ++failures;
}

// a transverse velocity that is flat up to one outlier far out
template <int D>
static void check_midpoint_outliers() {
    const Eos e = gases[0];
    for (int ec = -60; ec <= 90; ec += 3)
        for (int ej = 0; ej <= 330; ej += 3)
            for (int pos = 0; pos < 6; ++pos)
                for (int t = 0; t < 2; ++t) {
                    double s[6][5];
                    for (auto& w : s) {
                        w[0] = 1.0 + 0.01 * uni(-1, 1);
                        w[4] = 1.0 + 0.01 * uni(-1, 1);
                        w[1] = w[2] = w[3] = 0.25;
                    }
                    const int k = 1 + (D + 1 + t) % 3;
                    for (auto& w : s) w[k] = std::exp2(ec);
                    s[pos][k] = std::exp2(ej);
                    auto ld = [&](int j, int q) { return s[j][q]; };
                    double f[5], g[5];
                    if (!midpoint_flux_mid<D>(e, false, false, ld, f)) continue;
                    const bool fb = midpoint_flux<D, true>(e, ld, g);
                    if (fb) report("fallback taken in the mid range", &s[0][0], 30, 1, 0);
                    for (int q = 0; q < 5; ++q)
                        if (!same(f[q], g[q])) report("midpoint flux, outlier", &s[0][0], 30, f[q], g[q]);
                }
}

// the limiter's decision without divisions never contradicts the general one
template <class R>
static void check_admissible(int n) {
    long long clear = 0;
    for (int i = 0; i < n; ++i) {
        const Eos ed = gases[pick(5)];
        const EosT<R> e = eos_as<R>(ed);
        R q[5];
        q[0] = (R)(uni(0.05, 2.0) * std::exp2(pick(8) - 6));
        R k = 0;
        for (int d = 1; d < 4; ++d) {
            q[d] = (R)(q[0] * uni(-3, 3));
            k += q[d] * q[d];
        }
        // energies around the vacuum line, from far above to far below
        const double line = 0.5 * k / q[0] + q[0] * ed.q + ed.p_inf * (1.0 - q[0] * ed.b);
        q[4] = (R)(line * (1.0 + uni(-1, 1) * std::exp2(-pick(56))) + uni(-1, 1) * std::exp2(-pick(56)));
        if (!clearly_admissible(e, q)) continue;
        ++clear;
        R w[5];
        to_prim(e, q, w);
        if (!admissible(e, w[0], w[4])) {
            double in[5] = {(double)q[0], (double)q[1], (double)q[2], (double)q[3], (double)q[4]};
            report(sizeof(R) == 4 ? "clearly admissible f32" : "clearly admissible", in, 5, 1, 0);
        }
    }
    std::printf("clearly admissible: %lld\n", clear);
    if (clear < n / 20) ++failures;
}

int main() {
    check_to_prim(400000);
    check_pairs(400000);
    check_midpoints<0>(150000);
    check_midpoints<1>(150000);
    check_midpoints<2>(150000);
    check_midpoint_outliers<0>();
    check_admissible<double>(1000000);
    check_admissible<float>(1000000);
    std::printf(failures ? "%d MISMATCHES\n" : "ok\n", failures);
    return failures ? 1 : 0;
}
