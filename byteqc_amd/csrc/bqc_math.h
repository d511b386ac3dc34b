// Scalar arithmetic of the integral kernels: reciprocals and square roots
// from the hardware estimates, and the Rys interpolation polynomials as the
// row kernels keep them in LDS.  Host code compiles it too (with estimates of
// the hardware's precision), so that the errors are measured without a GPU.
// The includer includes rys_table.inc first.
#pragma once
#ifdef __HIPCC__
#define BQC_HD __host__ __device__ __forceinline__
#else
#define BQC_HD inline
#endif

namespace bqc {

// Estimates with a relative error of about 2^-24.
BQC_HD double rcp_estimate(double x) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_rcp(x);
#else
    return (double)(float)(1.0 / x);
#endif
}
BQC_HD double rsqrt_estimate(double x) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_rsq(x);
#else
    return (double)(float)(1.0 / __builtin_sqrt(x));
#endif
}

// 1/x, a/b and 1/sqrt(x) for positive normal x and b, rounded as the exact
// value is but for cases within 2^-40 of a tie: 4, 6 and 8 instructions.  The
// compiler's division takes 11 and its square root 14, mostly for denormals
// and infinities.  Each ends in an addition of a small correction to a value
// that is already right to 46 bits or more, so that its rounding is the only
// error left: in fast_div the correction comes from the remainder a - b q, in
// fast_rsqrt the product x r is kept in two parts.
BQC_HD double fast_rcp(double x) {
    const double r = rcp_estimate(x);
    const double e = __builtin_fma(-x, r, 1.0);
    return __builtin_fma(r, __builtin_fma(e, e, e), r);
}
BQC_HD double fast_div(double a, double b) {
    const double r0 = rcp_estimate(b);
    const double r = __builtin_fma(__builtin_fma(-b, r0, 1.0), r0, r0);
    const double q = a * r;
    return __builtin_fma(__builtin_fma(-b, q, a), r, q);
}
BQC_HD double fast_rsqrt(double x) {
    const double r = rsqrt_estimate(x);
    const double p = x * r;
    const double e = __builtin_fma(-p, r, 1.0) - __builtin_fma(x, r, -p) * r;
    return __builtin_fma(r * e, __builtin_fma(e, 0.375, 0.5), r);
}

// a0 = a1 / a and scale = 1 / (a1 sqrt(a)) of a primitive quartet, from a1 =
// the product and a = the sum of its two exponents: one inverse square root
// for both, where a quotient each would take two estimates.  a0 gets the
// remainder's correction; the roundings of a1^2 a count half in scale.
struct QuartetScale {
    double a0, scale;
    BQC_HD QuartetScale(double a1, double a) {
        scale = fast_rsqrt(a1 * (a1 * a));
        const double s = a1 * scale, ri = s * s, q = a1 * ri;
        a0 = __builtin_fma(__builtin_fma(-a, q, a1), ri, q);
    }
};

// Number of doubles of the interpolation table of N roots is
// rys_xbig(N) * 2 N (BQC_RYS_DEG + 1).
constexpr int rys_xbig(int n) { return 36 + 8 * n; }
constexpr int rys_offset(int n) {
    int off = 0;
    for (int m = 1; m < n; ++m) off += rys_xbig(m) * 2 * m * (BQC_RYS_DEG + 1);
    return off;
}

// Row of one interval in LDS: the 2 N functions of the N-root table in powers
// of y instead of Chebyshev polynomials (one FMA per term where Clenshaw's
// rule takes two operations), then the remainders of their constant terms
// (below): 2 N doubles for one and two roots, a 32-bit word per root for three
// and four, whose tables leave less room; then padding.  The lanes of a
// wavefront read 16 bytes each from rows of different intervals; an odd number
// of 16-byte units makes rows start in all 16 groups of LDS banks (rows of 24
// N doubles start in four groups for one root, in two for two).
constexpr bool rys_lds_wide(int n) { return n <= 2; }
constexpr int rys_lds_stride(int n) {
    return 2 * n * (BQC_RYS_DEG + 1) + (n == 2 ? 6 : 2);
}
constexpr int rys_lds_size(int n) { return rys_xbig(n) * rys_lds_stride(n); }

// Coefficient of y^k in the Chebyshev polynomial T_n(y): t[n][k].
struct ChebTable {
    double t[BQC_RYS_DEG + 1][BQC_RYS_DEG + 1];
    constexpr ChebTable() : t() {
        for (int n = 0; n <= BQC_RYS_DEG; ++n)
            for (int k = 0; k <= BQC_RYS_DEG; ++k)
                t[n][k] = n < 2 ? (n == k ? 1.0 : 0.0)
                                : (k > 0 ? 2.0 * t[n - 1][k - 1] : 0.0) - t[n - 2][k];
    }
};

// Coefficients m of the powers of y of the polynomial with Chebyshev
// coefficients c; returns what rounding took from m[0].
BQC_HD double rys_to_powers(const double *c, double *m) {
    constexpr ChebTable ch{};
    double v[BQC_RYS_DEG + 1];
#pragma unroll
    for (int n = 0; n <= BQC_RYS_DEG; ++n) v[n] = c[n];
    double m0 = 0.0, lo = 0.0;
#pragma unroll
    for (int k = 0; k <= BQC_RYS_DEG; ++k) {
        double s = 0.0;
#pragma unroll
        for (int n = BQC_RYS_DEG; n >= (k > 0 ? k : 1); --n)
            if ((n - k) % 2 == 0) s = __builtin_fma(ch.t[n][k], v[n], s);
        if (k == 0) {
            m0 = v[0] + s;  // |s| < |v[0]|
            lo = s - (m0 - v[0]);
            s = m0;
        }
        m[k] = s;
    }
    return lo;
}

// Row of the interval whose 2 N Chebyshev rows start at c, root r (u and w).
template <int N>
BQC_HD void rys_stage_root(const double *c, double *row, int r) {
    static_assert(N <= 4, "two doubles have room for the remainders of 4 roots");
    constexpr int D1 = BQC_RYS_DEG + 1;
    const double lo[2] = {rys_to_powers(c + r * D1, row + r * D1),
                          rys_to_powers(c + (N + r) * D1, row + (N + r) * D1)};
    double *const tail = row + 2 * N * D1;
    if constexpr (rys_lds_wide(N)) {
        tail[2 * r] = lo[0];
        tail[2 * r + 1] = lo[1];
    } else {
        // upper halves of both: 8 significant bits of a remainder are enough
        const unsigned word = (__builtin_bit_cast(unsigned, (float)lo[0]) & 0xffff0000u) |
                              __builtin_bit_cast(unsigned, (float)lo[1]) >> 16;
        __builtin_memcpy((char *)tail + 4 * r, &word, 4);
    }
}

// u_r, w_r (r < N) at y in [-1, 1] from a row.  Even and odd powers of all
// functions run side by side, 4 N chains of 4 dependent operations, and the
// last three steps are in the order of their size: with s = m1 + m2 y + ...
// the value is m0 + (y s + lo), lo being what rounding took from m0, so that
// the last addition is nearly the only error.  Largest (root mean square)
// relative error against the table's exact value, 1 to 4 roots, in 1e-16: 1.9
// (0.48); Clenshaw's rule 2.2 (0.67), even and odd sums joined by one FMA 3.3
// (0.83).  The remainders here and in QuartetScale cost 12 molecules def2-SVP
// 142.8 -> 148.2 ms, 64 waters cc-pVDZ 68.3 -> 68.8; without them the
// integrals are less precise than with Clenshaw's rule and divisions.
typedef double rys_pair __attribute__((vector_size(16)));
template <int N, typename Row>
BQC_HD void rys_from_row(double y, Row c, double *u, double *w) {
    constexpr int H = (BQC_RYS_DEG + 1) / 2;
    static_assert(BQC_RYS_DEG % 2 == 1, "coefficients are read in pairs");
    const double y2 = y * y;
    rys_pair v[2 * N];
#pragma unroll
    for (int f = 0; f < 2 * N; ++f) v[f] = c[f * H + H - 1];
#pragma unroll
    for (int j = H - 2; j >= 1; --j)
#pragma unroll
        for (int f = 0; f < 2 * N; ++f) {
            const rys_pair p = c[f * H + j];
            v[f][0] = __builtin_fma(y2, v[f][0], p[0]);
            v[f][1] = __builtin_fma(y2, v[f][1], p[1]);
        }
#pragma unroll
    for (int r = 0; r < N; ++r) {
        double lo[2];
        const rys_pair l = c[2 * N * H + (rys_lds_wide(N) ? r : 0)];
        if constexpr (rys_lds_wide(N)) {
            lo[0] = l[0];
            lo[1] = l[1];
        } else {
            const auto bits = __builtin_bit_cast(unsigned long long, (double)l[r / 2]);
            const unsigned word = (unsigned)(r % 2 ? bits >> 32 : bits);
            // the lower half adds less than 2^-7 to the remainder of u
            lo[0] = __builtin_bit_cast(float, word);
            lo[1] = __builtin_bit_cast(float, word << 16);
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int f = k * N + r;
            const rys_pair p = c[f * H];
            const double s =
                __builtin_fma(y, v[f][0], __builtin_fma(y2, v[f][1], p[1]));
            (k ? w : u)[r] = p[0] + __builtin_fma(y, s, lo[k]);
        }
    }
}

}  // namespace bqc
