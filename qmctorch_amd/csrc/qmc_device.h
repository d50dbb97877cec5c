// Device building blocks of the VMC kernels (gfx950, wave64).
//
// Lane layout used by every kernel: a wavefront holds G = 64 / nelec walkers,
// lane l = wl * nelec + e serves electron e of walker wl.  Basis, MO and CI
// tables are identical for all lanes of a launch (scalar-cache loads); each
// lane keeps its electron's MO row in registers.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qmc_mi355x.h"

namespace qmc {

// The tables and parameters of a launch are never written while its kernels
// run: device code reads them through the constant address space, so that
// wave-uniform reads become scalar loads whether the pointer arrived as a
// kernel argument or from a job table in device memory.
#if defined(__HIP_DEVICE_COMPILE__)
#define QMC_CONST __attribute__((address_space(4)))
#define QMC_LDS __attribute__((address_space(3)))
#else
#define QMC_CONST
#define QMC_LDS
#endif

template <typename X>
__device__ __forceinline__ X ldc(const X* p, size_t i) {
    return ((const __attribute__((address_space(4))) X*)p)[i];
}

struct Tables {
    int nelec, nup, ndown, natom, nao, nprim_ref, radial;
    int ngroup, nentry, nmo, nci, nconf_up, nconf_dn, nconf_max, nsig_max;
    int use_ee, use_en, identity_conf;
    int exc_mode;  // configurations as single/double excitations (trace-trick kernels)
    double vnn;
    const QMC_CONST int* grp_atom;
    const QMC_CONST int* grp_nprim;
    const QMC_CONST int* grp_prim0;
    const QMC_CONST int* grp_prim_src;
    const QMC_CONST int* grp_ao0;
    const QMC_CONST int* grp_nao;
    const QMC_CONST int* gao_mu;
    const QMC_CONST int* gao_k;
    const QMC_CONST double* gao_K;
    const QMC_CONST double* gao_n;
    const QMC_CONST int* gao_src;
    const QMC_CONST double* atom_z;
    const QMC_CONST double* jas_atoms;
    const QMC_CONST int* conf_up;
    const QMC_CONST int* conf_dn;
    const QMC_CONST int* ci_up;
    const QMC_CONST int* ci_dn;
    const QMC_CONST int* exc_up;  // [nconf_up][6] {level, h1, h2, p1, p2, sign}, or null
    const QMC_CONST int* exc_dn;
    // shell records of the table-driven AO row (ao_shells), kRecWords words each,
    // and their contraction coefficients
    int nrec;
    const QMC_CONST int* rec;
    const QMC_CONST double* rec_K;
    const QMC_CONST float* rec_Kf;
    int nrec_K;  // their number
    // inverse maps of the adjoint slot sum (CSR): the AO entries of AO mu are
    // ao_ent[ao_ptr[mu] .. ao_ptr[mu + 1]), the exponent-term columns
    // (entry i, primitive q) -> i * QMC_MAXP + q of bas_exp index k are
    // exp_col[exp_ptr[k] .. exp_ptr[k + 1]), both ascending
    const QMC_CONST int* ao_ptr;
    const QMC_CONST int* ao_ent;
    const QMC_CONST int* exp_ptr;
    const QMC_CONST int* exp_col;
};

// ------------------------------------------------------------------ math
// exp(x) in FP32 as the hardware 2^y of y = x log2 e: relative error about
// (|x| + 1) 2^-23, of the order of the rounding already in the argument
// (x = -a r^2 in FP32 carries |x| 2^-24); a compensated y (x log2 e split into
// its rounded product and the fma residual) halves the first term for three
// more instructions per exponential, which the sweeps do not need.
__device__ __forceinline__ float fexp(float x) { return __builtin_amdgcn_exp2f(x * 1.44269502162933349609375f); }
__device__ __forceinline__ double fexp(double x) { return exp(x); }

// 1/x: the hardware reciprocal (1 ulp) in FP32, a division in FP64
__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double frcp(double x) { return 1.0 / x; }

// log(m) for m in [0.5, 1) (a frexp mantissa): with m' = m or 2m in
// [1/sqrt 2, sqrt 2), z = (m' - 1)/(m' + 1), |z| < 0.172,
// log m' = 2 atanh z = 2 (z + z^3/3 + ... + z^21/21) (truncation < 1e-19),
// log m = log m' - [m' = 2m] log 2
// A wave-uniform constant formed where it is used (scalar moves) rather than
// hoisted by the compiler over an enclosing loop into registers it then spills.
__device__ __forceinline__ double sconst(double v) {
    asm volatile("" : "+s"(v));
    return v;
}

__device__ __forceinline__ double log_mantissa(double m) {
    const bool up = m < 0.70710678118654752;
    const double mm = up ? 2.0 * m : m;
    const double z = (mm - 1.0) / (mm + 1.0);
    const double s = z * z;
    double p = sconst(1.0 / 21.0);
    p = fma(p, s, sconst(1.0 / 19.0));
    p = fma(p, s, sconst(1.0 / 17.0));
    p = fma(p, s, sconst(1.0 / 15.0));
    p = fma(p, s, sconst(1.0 / 13.0));
    p = fma(p, s, sconst(1.0 / 11.0));
    p = fma(p, s, sconst(1.0 / 9.0));
    p = fma(p, s, sconst(1.0 / 7.0));
    p = fma(p, s, sconst(1.0 / 5.0));
    p = fma(p, s, sconst(1.0 / 3.0));
    p = fma(p, s, 1.0);
    return 2.0 * z * p - (up ? sconst(0.6931471805599453) : 0.0);
}
__device__ __forceinline__ float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }  // hardware, 1 ulp
__device__ __forceinline__ double fsqrt(double x) { return sqrt(x); }

template <typename T>
__device__ __forceinline__ T ipow(T x, int k) {
    // k in 0..3 (Cartesian exponents / STO r powers of the supported bases)
    T x2 = x * x;
    return k == 0 ? T(1) : (k == 1 ? x : (k == 2 ? x2 : x2 * x));
}

// Cartesian polynomial x^kx y^ky z^kz with gradient and Laplacian
// (spherical_harmonics.py:102-199, Cartesian branch).
template <typename T, bool DERIV>
__device__ __forceinline__ void cart_poly(T x, T y, T z, int kx, int ky, int kz, T& Y, T& Yx, T& Yy, T& Yz,
                                          T& Ylap) {
#pragma clang fp contract(off)
    T px = ipow(x, kx), py = ipow(y, ky), pz = ipow(z, kz);
    Y = px * py * pz;
    if (DERIV) {
        T dx = kx > 0 ? T(kx) * ipow(x, kx - 1) : T(0);
        T dy = ky > 0 ? T(ky) * ipow(y, ky - 1) : T(0);
        T dz = kz > 0 ? T(kz) * ipow(z, kz - 1) : T(0);
        Yx = dx * py * pz;
        Yy = px * dy * pz;
        Yz = px * py * dz;
        T d2x = kx > 1 ? T(kx * (kx - 1)) * ipow(x, kx - 2) : T(0);
        T d2y = ky > 1 ? T(ky * (ky - 1)) * ipow(y, ky - 2) : T(0);
        T d2z = kz > 1 ? T(kz * (kz - 1)) * ipow(z, kz - 2) : T(0);
        Ylap = d2x * py * pz + px * d2y * pz + px * py * d2z;
    }
}

// ------------------------------------------------------------ AO -> MO row
// Evaluates the AOs of one electron shell by shell and contracts them into the
// MO row on the fly (the AO row never leaves registers).  With the moments
// m_j = sum_p K_p a_p^j e_p of a shell's primitives, e_p = exp(-a_p r^2) (GTO,
// radial_functions.py:241-320) or exp(-a_p r) (STO, radial_functions.py:6-123),
//   AO = v Y,  grad AO = v grad Y + c Y r,  lap AO = Y (A + L B) + v lap Y:
//   GTO  v = m0, c = -2 m1, A = 4 r^2 m2 - 6 m1, B = -4 m1;
//   STO  R = r^n:  v = R m0, c = R (n m0 / r^2 - m1 / r),
//        A = R (n (n+1) m0 / r^2 - 2 (n+1) m1 / r + m2), B = 2 c
// (L the total Cartesian power), shared by the shell's 1, 3 or 6 entries.
//
// sink(i, ao, gx, gy, gz, lap) is called once per AO entry i; entries of one
// AO that were split across groups are delivered separately (all consumers
// are linear in the AO).

// exponents gathered in group-primitive order, in the evaluation precision
template <typename T>
__device__ __forceinline__ const T* group_exponents(const QmcParams& prm);
template <>
__device__ __forceinline__ const float* group_exponents<float>(const QmcParams& prm) {
    return prm.grp_expf;
}
template <>
__device__ __forceinline__ const double* group_exponents<double>(const QmcParams& prm) {
    return prm.grp_exp;
}

// exp(-a r^2) (or exp(-a r)) of the NP primitives of a group whose exponents
// start at p0 of the gathered exponent list
template <typename T, int RAD, int NP>
__device__ __forceinline__ void group_prims_from(const T* gexp, int p0, T r2, T r, T (&E)[NP], T (&A)[NP]) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const T a = ldc(gexp, p0 + p);
        A[p] = a;
        E[p] = (RAD == QMC_RADIAL_GTO_PURE) ? fexp(-a * r2) : fexp(-a * r);
    }
}

// ----------------------------------------------- table-driven AO row by shells
// The row of the kernels for any basis layout.  The plan describes it as
// records of up to three shells that share their primitives:
//   {atom, first exponent, first coefficient, first AO entry, shell word x 3,
//    np | nk << 8},
//   shell word: type | kx << 4 | ky << 8 | kz << 12 | r power << 16,
// each shell with np + 1 coefficients (its contraction, then the d_xy / d_xx
// normalisation ratio).  One scalar load fetches a record, one record ahead of
// its use, and the loads it leads to (exponents, coefficients, W rows) are
// issued together: walking the group and entry tables instead cost four
// dependent scalar loads per group and three per entry, and every entry
// selected its Cartesian powers at run time.  Two waters (20 electrons, 50 AOs,
// FP64), 2047 walkers x 50 steps: 1.411 -> 1.181 ms.
constexpr int kRecWords = 8;
constexpr int kRecShells = 3;  // shells per record at most
enum ShellType { kShellS = 0, kShellP = 1, kShellD = 2, kShellOne = 3 };  // D: xx xy xz yy yz zz; One: one entry

template <typename T>
__device__ __forceinline__ const QMC_CONST T* record_coeffs(const Tables& t);
template <>
__device__ __forceinline__ const QMC_CONST float* record_coeffs<float>(const Tables& t) {
    return t.rec_Kf;
}
template <>
__device__ __forceinline__ const QMC_CONST double* record_coeffs<double>(const Tables& t) {
    return t.rec_K;
}

// The pieces of a shell below say themselves where a product and a sum share
// one rounding: left to the compiler, a table-driven and a generated row would
// round differently, and near a node of the determinant FP32 rows that differ by
// one rounding differ by 1e-3 in log|psi|.

template <typename T>
__device__ __forceinline__ T norm2(T x, T y, T z) {
    return fma(z, z, fma(y, y, x * x));
}

// moments of a shell (m1 and m2 with DERIV) from its primitives' exponentials
template <typename T, bool DERIV, int NP, typename KF>
__device__ __forceinline__ void shell_moments(KF kcoef, const T (&E)[NP], const T (&A)[NP], T& m0, T& m1, T& m2) {
#pragma clang fp contract(off)
    m0 = m1 = m2 = T(0);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const T k = kcoef(p);
        m0 = fma(k, E[p], m0);
        if (DERIV) {
            const T kea = k * E[p] * A[p];
            m1 += kea;
            m2 = fma(kea, A[p], m2);
        }
    }
}

// radial part of a shell from its moments; n: STO r power
template <typename T>
struct ShellRadial {
    T v, c, A, B;
};
template <typename T, int RAD, bool DERIV>
__device__ __forceinline__ ShellRadial<T> shell_radial(T m0, T m1, T m2, int n, T r2, T r, T ir) {
#pragma clang fp contract(off)
    ShellRadial<T> s{m0, T(0), T(0), T(0)};
    if (RAD == QMC_RADIAL_GTO_PURE) {
        if (DERIV) {
            s.c = T(-2) * m1;
            s.A = fma(T(4) * r2, m2, T(-6) * m1);
            s.B = T(-4) * m1;
        }
    } else {
        const T R = ipow(r, n);
        s.v = R * m0;
        if (DERIV) {
            const T fn = T(n);
            s.c = R * fma(fn * m0 * ir, ir, -(m1 * ir));
            s.A = R * (fma(fn * (fn + T(1)) * m0 * ir, ir, T(-2) * (fn + T(1)) * m1 * ir) + m2);
            s.B = T(2) * s.c;
        }
    }
    return s;
}

// the entries of a shell from i on; f: normalisation of d_xy relative to d_xx;
// kx, ky, kz: the powers of a single entry
template <typename T, bool DERIV, int TYPE, typename Sink>
__device__ __forceinline__ void shell_entries(int i, const ShellRadial<T>& s, T x, T y, T z, T f, int kx, int ky,
                                              int kz, Sink& sink) {
#pragma clang fp contract(off)
    const T v = s.v, c = s.c;
    if (TYPE == kShellS) {
        sink(i, v, c * x, c * y, c * z, s.A);
    } else if (TYPE == kShellP) {
        const T l = s.A + s.B, cx = c * x, cy = c * y, cz = c * z;
        sink(i + 0, v * x, fma(cx, x, v), cx * y, cx * z, l * x);
        sink(i + 1, v * y, cy * x, fma(cy, y, v), cy * z, l * y);
        sink(i + 2, v * z, cz * x, cz * y, fma(cz, z, v), l * z);
    } else if (TYPE == kShellD) {
        const T l = fma(T(2), s.B, s.A), vf = v * f, cf = c * f, lf = l * f, v2 = v + v;
        const T xx = x * x, xy = x * y, xz = x * z, yy = y * y, yz = y * z, zz = z * z;
        sink(i + 0, v * xx, x * fma(c, xx, v2), c * xx * y, c * xx * z, fma(l, xx, v2));
        sink(i + 1, vf * xy, y * fma(cf, xx, vf), x * fma(cf, yy, vf), cf * xy * z, lf * xy);
        sink(i + 2, vf * xz, z * fma(cf, xx, vf), cf * xz * y, x * fma(cf, zz, vf), lf * xz);
        sink(i + 3, v * yy, c * yy * x, y * fma(c, yy, v2), c * yy * z, fma(l, yy, v2));
        sink(i + 4, vf * yz, cf * yz * x, z * fma(cf, yy, vf), y * fma(cf, zz, vf), lf * yz);
        sink(i + 5, v * zz, c * zz * x, c * zz * y, z * fma(c, zz, v2), fma(l, zz, v2));
    } else {
        T Y, Yx = 0, Yy = 0, Yz = 0, Yl = 0;
        cart_poly<T, DERIV>(x, y, z, kx, ky, kz, Y, Yx, Yy, Yz, Yl);
        const T cY = c * Y;
        sink(i, v * Y, fma(cY, x, v * Yx), fma(cY, y, v * Yy), fma(cY, z, v * Yz),
             fma(v, Yl, Y * fma(T(kx + ky + kz), s.B, s.A)));
    }
}

// moments m[shell][j] of a record's nk shells and NP primitives
template <typename T, int RAD, bool DERIV, int NP>
__device__ __forceinline__ void record_moments(const T* gexp, const QMC_CONST T* K, int nk, T r2, T r,
                                               T (&m)[kRecShells][3]) {
    T E[NP], A[NP];
    group_prims_from<T, RAD, NP>(gexp, 0, r2, r, E, A);
#pragma unroll
    for (int q = 0; q < kRecShells; ++q)
        if (q < nk)
            shell_moments<T, DERIV, NP>([&](int p) { return K[q * (NP + 1) + p]; }, E, A, m[q][0], m[q][1], m[q][2]);
}

// One dword of each 128-byte line of [p, p + bytes), four loads in flight a lane.
__device__ __forceinline__ uint32_t touch_lines(const void* p, int bytes, int lane) {
    uint32_t acc = 0;
    for (int b = lane * 128; b < bytes; b += 4 * 64 * 128) {
        uint32_t v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int o = b + k * 64 * 128;
            v[k] = o < bytes ? *(const uint32_t*)((const char*)p + o) : 0u;
        }
        acc |= (v[0] | v[1]) | (v[2] | v[3]);
    }
    return acc;
}

template <typename T, int RAD, bool DERIV, typename Sink>
__device__ __forceinline__ void ao_shells(const Tables& t, const QmcParams& prm, double ex, double ey, double ez,
                                          Sink&& sink) {
    typedef int int8v __attribute__((ext_vector_type(8)));
    const QMC_CONST int8v* rec = (const QMC_CONST int8v*)t.rec;
    int cur_atom = -1;
    T x = 0, y = 0, z = 0, r2 = 0, r = 0, ir = 0;
    int8v next = rec[0];
    for (int k = 0; k < t.nrec; ++k) {
        const int8v w = next;
        next = rec[k + 1 < t.nrec ? k + 1 : k];
        const int at = w[0], np = w[7] & 0xFF, nk = w[7] >> 8;
        if (at != cur_atom) {
            cur_atom = at;
            x = (T)(ex - ldc(prm.atom_coords, 3 * at + 0));
            y = (T)(ey - ldc(prm.atom_coords, 3 * at + 1));
            z = (T)(ez - ldc(prm.atom_coords, 3 * at + 2));
            r2 = norm2(x, y, z);
            if (RAD == QMC_RADIAL_STO) {
                r = fsqrt(r2);
                ir = T(1) / r;
            }
        }
        const T* gexp = group_exponents<T>(prm) + w[1];
        const QMC_CONST T* K = record_coeffs<T>(t) + w[2];
        T m[kRecShells][3];
        switch (np) {
#define QMC_REC_CASE(N)                                              \
    case N:                                                          \
        record_moments<T, RAD, DERIV, N>(gexp, K, nk, r2, r, m);     \
        break;
            QMC_REC_CASE(1) QMC_REC_CASE(2) QMC_REC_CASE(3) QMC_REC_CASE(4) QMC_REC_CASE(5) QMC_REC_CASE(6)
            QMC_REC_CASE(7) QMC_REC_CASE(8) QMC_REC_CASE(9) QMC_REC_CASE(10) QMC_REC_CASE(11) QMC_REC_CASE(12)
#undef QMC_REC_CASE
            default: break;
        }
        int i = w[3];
#pragma unroll 1
        for (int q = 0; q < nk; ++q) {
            const int word = q == 0 ? w[4] : (q == 1 ? w[5] : w[6]);
            const int type = word & 15;
            const T m0 = q == 0 ? m[0][0] : (q == 1 ? m[1][0] : m[2][0]);
            const T m1 = q == 0 ? m[0][1] : (q == 1 ? m[1][1] : m[2][1]);
            const T m2 = q == 0 ? m[0][2] : (q == 1 ? m[1][2] : m[2][2]);
            const ShellRadial<T> s = shell_radial<T, RAD, DERIV>(m0, m1, m2, word >> 16, r2, r, ir);
            if (type == kShellS) {
                shell_entries<T, DERIV, kShellS>(i, s, x, y, z, T(0), 0, 0, 0, sink);
                i += 1;
            } else if (type == kShellP) {
                shell_entries<T, DERIV, kShellP>(i, s, x, y, z, T(0), 0, 0, 0, sink);
                i += 3;
            } else if (type == kShellD) {
                shell_entries<T, DERIV, kShellD>(i, s, x, y, z, K[q * (np + 1) + np], 0, 0, 0, sink);
                i += 6;
            } else {
                shell_entries<T, DERIV, kShellOne>(i, s, x, y, z, T(0), (word >> 4) & 15, (word >> 8) & 15,
                                                   (word >> 12) & 15, sink);
                i += 1;
            }
        }
    }
}

// AO evaluation policies of the kernels: AoGeneric walks the shell records
// above; a generated policy (qmc_spec_*.hip) walks one basis layout with every
// shell, primitive offset and coefficient a compile-time constant, built from
// the same pieces in the same order, so both give the same values.
struct AoGeneric {
    static constexpr int kEntries = 0;    // AO entries of the row: known at run time only
    static constexpr int kRowBlocks = 4;  // 16-lane row blocks of the MFMA contraction: all
    template <typename T, int RAD, bool DERIV, typename Sink>
    static __device__ __forceinline__ void row(const Tables& t, const QmcParams& prm, double ex, double ey, double ez,
                                               Sink&& sink) {
        ao_shells<T, RAD, DERIV>(t, prm, ex, ey, ez, sink);
    }
};

template <typename T>
struct AtomGeo {
    T dx, dy, dz, r2, r, ir;
};

template <typename T, int RAD>
__device__ __forceinline__ AtomGeo<T> atom_geo(double dxd, double dyd, double dzd) {
    AtomGeo<T> g;
    g.dx = (T)dxd;
    g.dy = (T)dyd;
    g.dz = (T)dzd;
    g.r2 = norm2(g.dx, g.dy, g.dz);
    g.r = g.ir = T(0);
    if (RAD == QMC_RADIAL_STO) {
        g.r = fsqrt(g.r2);
        g.ir = T(1) / g.r;
    }
    return g;
}

// ------------------------------------------------------- lane-row elimination
// Gauss-Jordan elimination with partial pivoting on the n x n matrix whose
// row r lives in lane gbase + r (r < n), in FP64.  nmax (wave-uniform) is the
// largest n over the groups of the wave; lanes whose group is smaller simply
// idle through the extra columns.  On exit every lane of the group holds
// log|det| and sign(det); with WITH_B the augmented block b (n columns) is
// reduced to A^-1 B and the lane that pivoted column k returns in trace_part
// its entry (A^-1 B)_kk, otherwise 0.  Pivot choice: largest |a_rk| among the
// rows not used yet, first one on ties (LAPACK getrf's rule).
template <int NM, bool WITH_B>
__device__ __forceinline__ void lane_gauss_jordan(double (&a)[NM], double (&b)[NM], int n, int nmax, int myrow,
                                                  int gbase, uint64_t gmask, double& logdet, double& sgn,
                                                  double& trace_part, int& my_col) {
    bool done = false;
    my_col = -1;
    logdet = 0.0;
    sgn = 1.0;
    int inversions = 0;
    bool singular = false;
    double mant = 1.0;  // |det| = mant * 2^expo, renormalised after every pivot
    int expo = 0;
#pragma unroll
    for (int k = 0; k < NM; ++k) {
        if (k < nmax) {
            const bool colk = k < n;
            const double cand = (!done && colk && myrow < n) ? fabs(a[k]) : -1.0;
            // all candidates of the group are fetched first (independent
            // shuffles, one wait), then scanned in row order
            double c[NM];
#pragma unroll
            for (int s = 0; s < NM; ++s) c[s] = __shfl(cand, gbase + (s < n ? s : 0));
            double best = -1.0;
            int br = 0;
#pragma unroll
            for (int s = 0; s < NM; ++s) {
                if (s < n && c[s] > best) {
                    best = c[s];
                    br = s;
                }
            }
            const int plane = gbase + br;
            // rows not yet used with a smaller index than the pivot row
            const uint64_t bal = __ballot(!done && myrow < br);
            if (colk) inversions += __popcll(bal & gmask);
            const double piv = __shfl(a[k], plane);
            const bool is_piv = colk && (myrow == br);
            if (colk) {
                singular = singular || (piv == 0.0);
                int ex;
                mant = frexp(mant * fabs(piv), &ex);
                expo += ex;
                sgn *= (piv < 0.0) ? -1.0 : 1.0;
            }
            const double ip = (piv != 0.0) ? 1.0 / piv : 0.0;
            const double f = (colk && !is_piv && (WITH_B || !done)) ? a[k] * ip : 0.0;
            // pivot row broadcast: columns past nmax hold zeros and stay zero,
            // so every column is updated without a per-column branch
            double pa[NM];
#pragma unroll
            for (int j = k + 1; j < NM; ++j) pa[j] = __shfl(a[j], plane);
#pragma unroll
            // (rows already used are never read again by the determinant-only
            // elimination, so only the eliminated rows are written there)
            for (int j = k + 1; j < NM; ++j) a[j] = (WITH_B && is_piv) ? pa[j] * ip : a[j] - f * pa[j];
            if (WITH_B) {
                double pb[NM];
#pragma unroll
                for (int j = 0; j < NM; ++j) pb[j] = __shfl(b[j], plane);
#pragma unroll
                for (int j = 0; j < NM; ++j) b[j] = is_piv ? pb[j] * ip : b[j] - f * pb[j];
            }
            if (is_piv) {
                done = true;
                my_col = k;
            }
        }
    }
    if (inversions & 1) sgn = -sgn;
    logdet = singular ? -INFINITY : log_mantissa(mant) + 0.6931471805599453 * (double)expo;
    trace_part = 0.0;
    if (WITH_B) {
#pragma unroll
        for (int j = 0; j < NM; ++j)
            if (j == my_col) trace_part = b[j];
    }
}

// ------------------------------------------------------------ Philox4x32-10
// Salmon, Moraes, Dror, Shaw, "Parallel random numbers: as easy as 1, 2, 3",
// SC'11.  Round constants and Weyl key increments from that paper.
struct u4 {
    uint32_t x, y, z, w;
};

__device__ __forceinline__ u4 philox4x32_10(u4 c, uint32_t k0, uint32_t k1) {
    const uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u;
    const uint32_t W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        // one 32 x 32 -> 64-bit product per multiplier (v_mad_u64_u32) instead
        // of separate high and low multiplies
        const uint64_t p0 = (uint64_t)M0 * (uint64_t)c.x, p1 = (uint64_t)M1 * (uint64_t)c.z;
        const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
        const uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
        c = u4{hi1 ^ c.y ^ k0, lo1, hi0 ^ c.w ^ k1, lo0};
        k0 += W0;
        k1 += W1;
    }
    return c;
}

// (0,1] and [0,1) uniforms from 32 random bits
__device__ __forceinline__ double u01_open0(uint32_t v) { return ((double)v + 1.0) * 2.3283064365386963e-10; }
__device__ __forceinline__ double u01_closed0(uint32_t v) { return (double)v * 2.3283064365386963e-10; }

// Three standard normals from one Philox block, Box-Muller in FP64:
// (x, y) -> sqrt(-2 ln u) (cos 2 pi v, sin 2 pi v), (z, w) -> sqrt(-2 ln u) cos 2 pi v.
__device__ __forceinline__ void gauss3_f64(const u4 r, double& a, double& b, double& c) {
    const double r1 = sqrt(-2.0 * log(u01_open0(r.x)));
    const double r2 = sqrt(-2.0 * log(u01_open0(r.z)));
    double s1, c1;
    sincospi(2.0 * u01_closed0(r.y), &s1, &c1);
    a = r1 * c1;
    b = r1 * s1;
    c = r2 * cospi(2.0 * u01_closed0(r.w));
}

// ------------------------------------------------------------ wave-local LDS
// Orders one wavefront's LDS accesses across this point: the compiler moves no
// access over it, and the LDS performs a wavefront's requests in the order
// issued, so loads of any lane of the wavefront issued after the call see the
// stores issued before it.  No wait is needed for that: the fences have
// wavefront scope (at workgroup scope each drained the LDS counter; on its own
// worth 1 to 2 % of the benzene and two-water sweeps, nothing elsewhere).  It
// orders nothing between wavefronts and no access to global memory.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int kBlock = 256;  // threads per block of the wave-per-walker-group kernels
constexpr int kBlockWaves = kBlock / 64;

// Pivot row (group-relative) of column k for the eliminations of the large
// buckets: the candidate with the largest |v| (the first one on ties), by an
// LDS atomic maximum into a slot of the group instead of ceil(log2 n)
// dependent shuffle rounds.  Each lane's key is the high word of |v|'s FP64 bit
// pattern (exponent and top 20 mantissa bits, monotonic in |v|) with its five
// low bits replaced by 31 - row; non-candidates do not take part.  Magnitudes
// that differ beyond their top 15 mantissa bits are ordered exactly; closer
// ones count as tied and go to the first row (partial pivoting only needs a
// large pivot, not the exact maximum).  No candidate (a column past this
// group's n): row 0.
// The slot of a group is its first lane's index; columns alternate between two
// slot sets, and row 0 of each group clears the other set's slot for column
// k + 1 while column k's maxima are formed.  The LDS runs one wavefront's
// instructions in order, so that clear follows the reads of column k - 1 and
// precedes the maxima of column k + 1.  Lanes outside every walker (real =
// false, whose group may share its first lane index with a real group) only
// read.  seg_pivot_init clears set 0 before column 0.  The read of the
// maximum is issued after every maximum and after the caller's earlier LDS stores.
__device__ __forceinline__ uint32_t* seg_pivot_slots() {
    __shared__ uint32_t slots[kBlockWaves * 128];
    return slots + (threadIdx.x >> 6) * 128;
}

// Reciprocal of each group's published pivot (lane_det_lds), at the group's
// first lane index.
__device__ __forceinline__ double* det_recips() {
    __shared__ double r[kBlockWaves * 64];
    return r + (threadIdx.x >> 6) * 64;
}

__device__ __forceinline__ void seg_pivot_init(int myrow, int gbase, bool real) {
    uint32_t* S = seg_pivot_slots();
    wave_lds_sync();  // earlier eliminations' reads of the slots come first
    if (real && myrow == 0) S[gbase] = 0u;
}

// seg_pivot_post issues column k's maximum (and the next column's clear);
// seg_pivot_get reads it, after every LDS store the caller issued in between,
// and returns the pivot row.
template <int NM>
__device__ __forceinline__ void seg_pivot_post(int k, bool cand, double v, int myrow, int gbase, bool real) {
    static_assert(NM <= 32, "five bits of row index");
    uint32_t* S = seg_pivot_slots();
    const uint32_t hi = (uint32_t)((uint64_t)__double_as_longlong(fabs(v)) >> 32);
    const uint32_t key = (hi & ~31u) | (uint32_t)(31 - myrow);
    if (real && cand)
        __hip_atomic_fetch_max(S + (k & 1) * 64 + gbase, key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (real && myrow == 0) S[((k + 1) & 1) * 64 + gbase] = 0u;
}

__device__ __forceinline__ int seg_pivot_get(int k, int gbase) {
    wave_lds_sync();
    const uint32_t m = seg_pivot_slots()[(k & 1) * 64 + gbase];
    return m ? 31 - (int)(m & 31u) : 0;
}

// ------------------------------------------------- determinant-only elimination
// Determinant det 2^ex2 (det 0 or a signed mantissa) of the n x n matrix whose
// row r lives in lane gbase + r, with the row arithmetic of
// lane_gauss_jordan<NM, false> but fewer cross-lane moves per column:
//  * the pivot (largest |a_rk| among the rows not used yet, first one on ties,
//    compared through seg_pivot_post's 32-bit keys): up to 8 columns from the n
//    keys gathered into every lane by shuffles; for the larger buckets by
//    its LDS atomic maximum;
//  * the pivot row through LDS, read back as broadcast loads (two columns per
//    load) instead of one shuffle pair per column, with the pivot itself and
//    its reciprocal (det_recips()), which every candidate forms while the
//    pivot is searched (the division leaves the column's critical path): for
//    the larger buckets the pivot lane stores its remaining columns at
//    rowbuf[0..NM) once the pivot is known; up to 8 columns every candidate
//    row r stores them at rowbuf[r NM ..] during the search (n NM doubles).
// Stores happen only when may_store.
// Rows already used are never read again (f = 0 for them), so only the rows
// still to be eliminated are written.
template <int NM>
__device__ __forceinline__ void lane_det_lds(double (&a)[NM], int n, int nmax, int myrow, int gbase, int spin,
                                             uint64_t gmask, bool may_store, double* rowbuf, double& det, int& ex2) {
    if constexpr (NM > 8) seg_pivot_init(myrow, gbase, may_store);
    double* const recip = det_recips() + gbase;  // the group's pivot reciprocal
    bool done = false;
    double sgn = 1.0;
    int inversions = 0;
    bool singular = false;
    double mant = 1.0;  // |det| = mant * 2^expo, renormalised after every pivot
    int expo = 0;
#pragma unroll
    for (int k = 0; k < NM; ++k) {
        if (k < nmax) {
            const bool colk = k < n;
            if constexpr (NM > 8) {
                // the reciprocal of every candidate's pivot is formed while the
                // search runs; the pivot lane then publishes its remaining
                // columns and that reciprocal (rowbuf[0..NM) and the group's
                // det_recips() entry), which the group reads back at once
                const bool cand = !done && colk && myrow < n;
                seg_pivot_post<NM>(k, cand, a[k], myrow, gbase, may_store);
                double rk = (a[k] != 0.0) ? 1.0 / a[k] : 0.0;
                asm volatile("" : "+v"(rk));  // formed here, not sunk into the pivot lane's store
                const int br = seg_pivot_get(k, gbase);
                const uint64_t bal = __ballot(!done && myrow < br);
                if (colk) inversions += __popcll(bal & gmask);
                const bool is_piv = colk && (myrow == br);
                wave_lds_sync();  // the previous column's reads come first
                if (is_piv && may_store) {
#pragma unroll
                    for (int j = k; j < NM; ++j) rowbuf[j] = a[j];
                    *recip = rk;
                }
                wave_lds_sync();
                // past this group's n nobody stores and the row is stale: colk
                // is false there, so neither the determinant nor a uses it
                const double piv = rowbuf[k];
                const double ip = *recip;
                {
                    const double pv = colk ? piv : 1.0;
                    singular = singular || (pv == 0.0);
                    int ex;
                    mant = frexp(mant * fabs(pv), &ex);
                    expo += ex;
                    sgn *= (pv < 0.0) ? -1.0 : 1.0;
                }
                const double f = (colk && !is_piv && !done) ? a[k] * ip : 0.0;
#pragma unroll
                for (int j = k + 1; j < NM; ++j) a[j] = a[j] - f * rowbuf[j];
                if (is_piv) done = true;
            } else {
                // keys as in seg_pivot_post, gathered from the group's n lanes (reads
                // past the last row repeat it, which leaves the maximum alone);
                // meanwhile every candidate row r publishes its remaining
                // columns at rowbuf[r NM + k ..] and its pivot's reciprocal at
                // recip[r], and the group then reads the chosen row back (slots
                // of rows already used are not written again, so rows read in
                // earlier columns stay intact)
                const bool cand = !done && colk && myrow < n;
                const uint32_t hi = (uint32_t)((uint64_t)__double_as_longlong(fabs(a[k])) >> 32);
                const uint32_t key = cand ? ((hi & ~31u) | (uint32_t)(31 - myrow)) : 0u;
                if (cand && may_store) {
                    double* const slot = rowbuf + myrow * NM;
#pragma unroll
                    for (int j = k; j < NM; ++j) slot[j] = a[j];
                    recip[myrow] = (a[k] != 0.0) ? 1.0 / a[k] : 0.0;
                }
                uint32_t m = 0;
#pragma unroll
                for (int s = 0; s < NM; ++s) m = max(m, (uint32_t)__shfl((int)key, gbase + (s < n ? s : n - 1)));
                const int br = m ? 31 - (int)(m & 31u) : 0;
                const uint64_t bal = __ballot(!done && myrow < br);
                if (colk) inversions += __popcll(bal & gmask);
                const bool is_piv = colk && (myrow == br);
                wave_lds_sync();  // the candidates' stores come first
                const double* const prow = rowbuf + br * NM;
                const double piv = prow[k];
                const double ip = recip[br];
                {
                    const double pv = colk ? piv : 1.0;
                    singular = singular || (pv == 0.0);
                    int ex;
                    mant = frexp(mant * fabs(pv), &ex);
                    expo += ex;
                    sgn *= (pv < 0.0) ? -1.0 : 1.0;
                }
                const double f = (colk && !is_piv && !done) ? a[k] * ip : 0.0;
#pragma unroll
                for (int j = k + 1; j < NM; ++j) a[j] = a[j] - f * prow[j];
                if (is_piv) done = true;
            }
        }
    }
    if (inversions & 1) sgn = -sgn;
    det = singular ? 0.0 : sgn * mant;
    ex2 = expo;
}

// ------------------------------------------------------ in-place inverse (LDS)
// Gauss-Jordan inversion of the n x n matrix whose row r lives in lane
// gbase + r, in the NM registers of the row: after the step of column k with
// pivot row p, storage column k holds the inverse's column of row p.  On exit
// the lane that pivoted column k (my_col = k) holds row k of A^-1 with the
// entry of row i in storage column (my_col of row i's lane); det and ex2 as
// lane_det_lds, pivots chosen by seg_pivot_post.  NM multiply-adds per column and
// row, where eliminating [A | I] or [A | B] took up to 2 NM and twice the
// registers.  rowbuf: the group's row buffer (NM doubles used).
template <int NM>
__device__ __forceinline__ void lane_invert_lds(double (&a)[NM], int n, int nmax, int myrow, int gbase,
                                                uint64_t gmask, bool may_store, double* rowbuf, double& det,
                                                int& ex2, int& my_col) {
    seg_pivot_init(myrow, gbase, may_store);
    double* const pivot = det_recips() + gbase;  // the column's pivot
    bool done = false;
    my_col = -1;
    double sgn = 1.0;
    int inversions = 0;
    bool singular = false;
    double mant = 1.0;  // |det| = mant * 2^expo, renormalised after every pivot
    int expo = 0;
#pragma unroll
    for (int k = 0; k < NM; ++k) {
        if (k < nmax) {
            const bool colk = k < n;
            const bool cand = !done && colk && myrow < n;
            seg_pivot_post<NM>(k, cand, a[k], myrow, gbase, may_store);
            // the reciprocal of every candidate is formed while the search runs
            double rk = (a[k] != 0.0) ? 1.0 / a[k] : 0.0;
            asm volatile("" : "+v"(rk));
            const int br = seg_pivot_get(k, gbase);
            const uint64_t bal = __ballot(!done && myrow < br);
            if (colk) inversions += __popcll(bal & gmask);
            const bool is_piv = colk && (myrow == br);
            wave_lds_sync();  // the previous column's reads come first
            if (is_piv && may_store) {
                // the pivot row over its pivot, the reciprocal in its own column
#pragma unroll
                for (int j = 0; j < NM; ++j) rowbuf[j] = j == k ? rk : a[j] * rk;
                *pivot = a[k];
            }
            wave_lds_sync();
            {
                // past this group's n nobody stores: colk is false, nothing is used
                const double pv = colk ? *pivot : 1.0;
                singular = singular || (pv == 0.0);
                int ex;
                mant = frexp(mant * fabs(pv), &ex);
                expo += ex;
                sgn *= (pv < 0.0) ? -1.0 : 1.0;
            }
            const double f = colk ? a[k] : 0.0;
#pragma unroll
            for (int j = 0; j < NM; ++j) {
                const double p = rowbuf[j];
                if (j == k)
                    a[k] = is_piv ? p : (colk ? -f * p : a[k]);
                else
                    a[j] = is_piv ? p : fma(-f, p, a[j]);
            }
            if (is_piv) {
                done = true;
                my_col = k;
            }
        }
    }
    if (inversions & 1) sgn = -sgn;
    det = singular ? 0.0 : sgn * mant;
    ex2 = expo;
}

}  // namespace qmc
