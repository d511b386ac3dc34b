// Errors of byteqc_amd/csrc/bqc_math.h on the host, in units of 2^-53
// (relative): "name max rms" per line.  The reference of the Rys functions is
// the table's Chebyshev sum in long double.
#include <cmath>
#include <cstdio>
#include <random>
#define BQC_RYS_QUAL static
#include "../../byteqc_amd/csrc/rys_table.inc"
#include "../../byteqc_amd/csrc/bqc_math.h"
using namespace bqc;

static const double U = std::ldexp(1.0, -53);
struct Err {
    double max = 0, sq = 0;
    long n = 0;
    void add(double got, long double want) {
        const double e = std::fabs((double)((got - want) / want)) / U;
        if (!(e <= max)) max = e;
        sq += e * e;
        ++n;
    }
    void print(const char *name, int k) const {
        std::printf("%s%d %.6f %.6f\n", name, k, max, std::sqrt(sq / n));
    }
};

template <class T> static T clenshaw(const double *c, double y) {
    T b1 = 0, b2 = 0;
    for (int j = BQC_RYS_DEG; j >= 1; --j) {
        const T t = std::fma((T)(2 * y), b1, c[j] - b2);
        b2 = b1;
        b1 = t;
    }
    return std::fma((T)y, b1, c[0] - b2);
}

template <int N> static void rys(std::mt19937_64 &gen) {
    std::uniform_real_distribution<double> unif(0.0, 1.0);
    constexpr int D1 = BQC_RYS_DEG + 1;
    Err got[2], ref[2];
    for (int it = 0; it < rys_xbig(N); ++it) {
        const double *c = BQC_RYS_COEF + rys_offset(N) + it * 2 * N * D1;
        alignas(16) double row[rys_lds_stride(N)];
        for (int r = 0; r < N; ++r) rys_stage_root<N>(c, row, r);
        for (int s = 0; s < 400; ++s) {
            const double x = s == 0 ? it : std::nextafter(it + unif(gen), (double)it);
            const double y = 2 * (x - it) - 1;
            double out[2][N];
            rys_from_row<N>(y, (const rys_pair *)row, out[0], out[1]);
            for (int f = 0; f < 2 * N; ++f) {
                const long double want = clenshaw<long double>(c + f * D1, y);
                got[f / N].add(out[f / N][f % N], want);
                ref[f / N].add(clenshaw<double>(c + f * D1, y), want);
            }
        }
    }
    got[0].print("u", N);
    ref[0].print("clenshaw_u", N);
    got[1].print("w", N);
    ref[1].print("clenshaw_w", N);
}

int main() {
    std::mt19937_64 gen(7);
    std::uniform_real_distribution<double> lg(-30.0, 30.0), unif(0.5, 1.0);
    Err rcp, div, rsq, a0, a0_ref, fac, fac_ref;
    for (int i = 0; i < 2000000; ++i) {
        const double a = std::exp2(lg(gen)), b = std::exp2(lg(gen));
        rcp.add(fast_rcp(b), 1.0L / b);
        div.add(fast_div(a, b), (long double)a / b);
        rsq.add(fast_rsqrt(b), 1.0L / std::sqrt((long double)b));
    }
    // a0 = p q / (p + q) and 1 / (p q sqrt(p + q)) of the primitive quartets,
    // as the kernels form them and with quotients and square roots
    for (int i = 0; i < 2000000; ++i) {
        const double p = std::exp2(lg(gen) / 2), q = std::exp2(lg(gen) / 2), pq = p + q, a1 = p * q;
        const double f = unif(gen);
        const QuartetScale s(a1, pq);
        const long double sum = (long double)p + q, prod = (long double)p * q;
        a0.add(s.a0, prod / sum);
        a0_ref.add(a1 / pq, prod / sum);
        fac.add(f * s.scale, f / (prod * std::sqrt(sum)));
        fac_ref.add(f / (std::sqrt(pq) * a1), f / (prod * std::sqrt(sum)));
    }
    a0.print("a", 0);
    a0_ref.print("quotient_a", 0);
    fac.print("fac", 0);
    fac_ref.print("quotient_fac", 0);
    rcp.print("rcp", 0);
    div.print("div", 0);
    rsq.print("rsqrt", 0);
    rys<1>(gen);
    rys<2>(gen);
    rys<3>(gen);
    rys<4>(gen);
}
