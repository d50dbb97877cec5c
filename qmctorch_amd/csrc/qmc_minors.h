// Determinants and inverse columns of small matrices by minors (FP64).
//
// Branch-free and without any exchange between lanes: the kernels give every
// lane the rows of its group and let it expand the determinant along its own
// row, which also yields its column of the inverse.
#pragma once
#include <type_traits>
#include <utility>

#ifndef QMC_MINORS_FN  // a host compiler checks the expansion with this set to `inline`
#define QMC_MINORS_FN __device__ __forceinline__
#endif

namespace qmc {

// Largest matrix expanded by minors: 75 operations for N = 5, 186 for 6, 441
// for 7; at N = 8 (about 1000) an elimination does less work.
//
// Accuracy.  Near a node the determinant is a small difference of large terms,
// and N expansions along N rows round it differently: lanes that combine their
// inverse columns must divide their cofactors by one common determinant.  Then
// (2 x 2 minors to full precision) the kinetic trace of 65536 H2O walkers is
// off from an 80-bit elimination by 6.1e-15 / 1.2e-12 (99 % / 99.99 % quantile,
// relative to E_L) where a pivoted FP64 elimination is off by 9.6e-15 /
// 3.0e-12; N2: 1.2e-14 / 3.5e-12 against 1.5e-14 / 8.6e-12.  With each lane's
// own determinant it was 2.8e-14 / 6.8e-12 and 6.9e-14 / 5.8e-11.  A block with
// several small singular values (walkers far outside the molecule) loses more
// than an elimination does, so FP64 blocks whose determinant, of rows scaled to
// a largest entry of 1/2 to 1, is below kWeakDet are eliminated instead: 1e-5
// of the groups above, and the quantiles stay at or below the elimination's
// for walkers spread two and four times as far.  FP32 rows are not scaled, and
// their own rounding is larger than either way's.
constexpr int kMaxMinors = 7;

constexpr double kWeakDet = 1e-6;

template <int I, int E, typename F>
QMC_MINORS_FN void static_for(F&& f) {
    if constexpr (I < E) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, E>(f);
    }
}

// index of the columns i < j among the pairs of n columns
constexpr int pair_at(int n, int i, int j) { return i * n - i * (i + 1) / 2 + (j - i - 1); }

constexpr int popcount(int m) {
    int c = 0;
    for (; m; m &= m - 1) ++c;
    return c;
}

// the t-th column of the set m
constexpr int column_of(int m, int t) {
    for (int c = 0;; ++c)
        if ((m >> c) & 1)
            if (t-- == 0) return c;
}

// Laplace sign of the columns `top` for the upper rows among n columns without
// k, times (-1)^k of the expansion along the first row
constexpr bool laplace_negative(int n, int k, int top) {
    int s = k, pos = 0, cnt = 0;
    for (int c = 0; c < n; ++c) {
        if (c == k) continue;
        if ((top >> c) & 1) s += pos - cnt++;
        ++pos;
    }
    return (s & 1) != 0;
}

// 2 x 2 minors of rows a and b.  ACC: each to 1.5 ulp of its value by the
// products' rounding errors (Kahan's difference of products), against a
// rounding of the larger product; two more operations per minor.
template <int N, bool ACC>
QMC_MINORS_FN void minors2(const double (&a)[N], const double (&b)[N], double (&m)[N * (N - 1) / 2]) {
    static_for<0, N>([&](auto ic) {
        static_for<decltype(ic)::value + 1, N>([&](auto jc) {
            constexpr int i = decltype(ic)::value, j = decltype(jc)::value, p = pair_at(N, i, j);
            const double w = a[j] * b[i];
            m[p] = __builtin_fma(a[i], b[j], -w);
            if constexpr (ACC) m[p] += __builtin_fma(-a[j], b[i], w);
        });
    });
}

// 3 x 3 minor of row a above two rows with 2 x 2 minors m, columns of the set S
template <int N, int S>
QMC_MINORS_FN double minor3(const double (&a)[N], const double (&m)[N * (N - 1) / 2]) {
    constexpr int i = column_of(S, 0), j = column_of(S, 1), l = column_of(S, 2);
    constexpr int jl = pair_at(N, j, l), il = pair_at(N, i, l), ij = pair_at(N, i, j);
    return a[i] * m[jl] - a[j] * m[il] + a[l] * m[ij];
}

// Signed cofactors of the first row of an N x N matrix whose other rows are
// R[0..N-2]: c[k] = (-1)^k det(R without column k), so that the determinant is
// sum_k a[k] c[k] for a first row a, and c[k] / det is the first column of the
// inverse.  Laplace expansion: the minors of the upper rows (N = 4: one row, 5
// and 6: two, 7: three) meet the complementary minors of the lower rows (two,
// or three) once per column k outside both.
template <int N, bool ACC>
QMC_MINORS_FN void first_row_cofactors(const double (&R)[N > 1 ? N - 1 : 1][N], double (&c)[N]) {
    static_assert(N >= 1 && N <= kMaxMinors, "matrices up to 7 x 7");
    if constexpr (N == 1) {
        c[0] = 1.0;
    } else if constexpr (N == 2) {
        c[0] = R[0][1];
        c[1] = -R[0][0];
    } else if constexpr (N == 3) {
        c[0] = R[0][1] * R[1][2] - R[0][2] * R[1][1];
        c[1] = R[0][2] * R[1][0] - R[0][0] * R[1][2];
        c[2] = R[0][0] * R[1][1] - R[0][1] * R[1][0];
    } else {
        constexpr int kUp = N == 4 ? 1 : (N == 7 ? 3 : 2), kLow = N - 1 - kUp;
        constexpr int kAll = (1 << N) - 1;
        double low2[N * (N - 1) / 2], up2[N * (N - 1) / 2], low3[kLow == 3 ? (1 << N) : 1];  // low3: by column set
        minors2<N, ACC>(R[N - 3], R[N - 2], low2);
        if constexpr (kLow == 3)
            static_for<0, (1 << N)>([&](auto sc) {
                constexpr int S = decltype(sc)::value;
                if constexpr (popcount(S) == 3) low3[S] = minor3<N, S>(R[N - 4], low2);
            });
        if constexpr (kUp >= 2) minors2<N, ACC>(R[kUp - 2], R[kUp - 1], up2);
        static_for<0, N>([&](auto kc) { c[decltype(kc)::value] = 0.0; });
        static_for<0, (1 << N)>([&](auto tc) {
            constexpr int top = decltype(tc)::value;
            if constexpr (popcount(top) == kUp) {
                double mt;
                constexpr int t0 = column_of(top, 0), tp = kUp == 2 ? pair_at(N, t0, column_of(top, kUp - 1)) : 0;
                if constexpr (kUp == 1)
                    mt = R[0][t0];
                else if constexpr (kUp == 2)
                    mt = up2[tp];
                else
                    mt = minor3<N, top>(R[0], up2);
                static_for<0, N>([&](auto kc) {
                    constexpr int k = decltype(kc)::value;
                    if constexpr (((top >> k) & 1) == 0) {
                        constexpr int rest = kAll & ~top & ~(1 << k);
                        constexpr int at = kLow == 2 ? pair_at(N, column_of(rest, 0), column_of(rest, 1)) : rest;
                        constexpr bool minus = laplace_negative(N, k, top);
                        double ml;
                        if constexpr (kLow == 2)
                            ml = low2[at];
                        else
                            ml = low3[at];
                        c[k] = __builtin_fma(minus ? -mt : mt, ml, c[k]);
                    }
                });
            }
        });
    }
}

}  // namespace qmc
