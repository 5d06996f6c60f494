// The FP64 samplers' FP32 accept estimates (tm_device.h) as they are compiled, with the
// hardware's logarithm and reciprocal as far off as an ulp either way: a trial that an
// estimate settles has the outcome of the FP64 test it stands for.  Half of the trials lie
// close to equality, where the margins decide.
#include <random>

#include "tm_device.h"

using namespace tmk;

static std::mt19937_64 rng(11);
static double uniform() { return ((double)(uint32_t)rng() + 0.5) * 0x1p-32; }
static int bad = 0;

// FP64 sides of the tests, as gamma_d_try and poisson_d form them
static double gamma_rhs(double x2, double v, double d) { return 0.5 * x2 + d * (1.0 - v + dlog(v)); }
static double ptrs_rhs(double z, double kd) { return -z + kd * dlog(z) - logfact((int64_t)kd); }
static double ptrs_lhs(const PtrsD& p, double us, double V)
{
    return dlog(V) + dlog(1.1239 + 1.1328 / (p.b - 3.4)) - dlog(p.a / (us * us) + p.b);
}

static void gamma_trials(double d, int n, double settled)
{
    std::normal_distribution<double> normal;
    const double c = 1.0 / dsqrt(9.0 * d);
    int total = 0, called = 0, wrong = 0;
    for (int i = 0; i < n; ++i) {
        const double x = normal(rng) * (i % 3 == 0 ? 2.0 : 1.0), y = c * x;
        double v = 1.0 + y;
        if (v <= 0.0) continue;
        v = v * v * v;
        const double x2 = x * x, rhs = gamma_rhs(x2, v, d);
        double u = uniform();
        const bool close = i % 2 == 0;
        if (close) u = std::exp(rhs + (uniform() - 0.5) * 6e-3);
        if (!(u > 0x1p-34 && u < 1.0)) continue;
        const bool accepts = dlog(u) < rhs;
        cpu_hip_ulp = i / 2 % 3 - 1;
        const int est = gamma_estimate(u, x2, y, v, d);
        if (est != 0 && (est > 0) != accepts) ++wrong;
        if (!close) ++total, called += est != 0;
    }
    if (wrong || called < settled * total) {
        fprintf(stderr, "gamma d = %g: %d of %d settled, %d wrong\n", d, called, total, wrong);
        ++bad;
    }
}

static void ptrs_trials(double z, int n)
{
    const PtrsD p = ptrs_setup_d(z);
    int offered = 0, called = 0, wrong = 0;
    for (int i = 0; i < n; ++i) {
        const double U = uniform() - 0.5, us = 0.5 - std::fabs(U);
        const double kd = ptrs_k_d(p, z, U, us);
        double V = uniform();
        if (kd < 0.0) continue;
        const double rhs = ptrs_rhs(z, kd);
        const bool close = i % 2 == 0;
        if (close) V = std::exp(rhs - ptrs_lhs(p, us, 1.0) + (uniform() - 0.5) * 6e-3);
        if (!(V > 0x1p-34 && V < 1.0) || (us < 0.013 && V > us)) continue;
        const bool accepts = ptrs_lhs(p, us, V) <= rhs;
        cpu_hip_ulp = i / 2 % 3 - 1;
        const int est = ptrs_estimate(p, z, kd, us, V);
        if (est != 0 && (est > 0) != accepts) ++wrong;
        const bool domain = kd >= 5.0 && z < 1e9 && (std::fabs(kd - z) < 0.1 * (kd + z) || kd < 1000.0);
        if (!close && domain) ++offered, called += est != 0;
    }
    if (wrong || called < 0.97 * offered) {
        fprintf(stderr, "PTRS z = %g: %d of %d settled, %d wrong\n", z, called, offered, wrong);
        ++bad;
    }
}

int main()
{
    const int n = 300000;
    // large shapes, where the FP64 test's rounding grows past any fixed margin
    for (double d : {2.0 / 3.0, 0.8, 1.5, 4.0, 30.0, 454.0, 456.0, 7e4, 1e7, 9.9e8}) gamma_trials(d, n, 0.98);
    for (double d = 1e9; d < 1e45; d *= 30.0) gamma_trials(d, n, 0.0);
    for (double z : {12.0, 13.7, 40.0, 300.0, 900.0, 1100.0, 1.6e3, 1.4e5, 2e7, 9.9e8, 1e9, 1e12, 1e16}) ptrs_trials(z, n);
    if (bad) return 1;
    puts("ok");
    return 0;
}
