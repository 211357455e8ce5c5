// eri_math.h -- contracted s/p shell-quartet ERIs by Obara-Saika vertical
// recursion and Head-Gordon-Pople horizontal recursion, FP64.
//
// Everything here is __host__ __device__ so the same code runs in the gfx950
// kernels and in the host-side check against the oracle.
//
// Numerics follow the reference's integral path where they change values at
// the 1e-10 level (src/integrals/int2e.f90, src/integrals/auxilary.f90):
//   * pi rounded to single precision (the `Pi = 3.1415926535897931` literals
//     without a D0 suffix, int2e.f90:621, auxilary.f90:169,196,711);
//   * Boys F_m(T): for T < 12 a 7-term Taylor expansion of F_Q from the
//     tabulated Ftab at Tk = NINT(10 T), Q = 3 * (sum of the four sets' max L),
//     then downward recursion (auxilary.f90:130-162); for 12 <= T < 2Q+36 the
//     asymptotic F_0 with the piecewise g(T), upward recursion
//     (auxilary.f90:167-189,265-285); beyond, the simplified upward form
//     (auxilary.f90:194-215);
//   * primitive quartets with EIJ*EGH < 1e-14 skipped (int2e.f90:257).
// The recursion itself (OS/HGP rather than McMurchie-Davidson) differs from
// the reference only at rounding level.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>

#include <cmath>
#include <vector>

#define MYQC_HD __host__ __device__ __forceinline__

namespace myqc {

// `REAL(KIND=8),PARAMETER :: Pi = 3.1415926535897931` holds the single-precision value
constexpr double PI_SP = (double)3.1415926535897931f;

constexpr int FT_NT = 121;   // Tk = 0..120  (T = 0 .. 12 step 0.1)
constexpr int FT_NM = 19;    // m  = 0..18 of the record's 23: the largest order read is Q + 6 = 18 (Q <= 12)
// The Boys tables as the kernels use them.  For T < 12 the reference expands
// F_Q about Tk and recurs downward to F_M (below), up to 12 dependent steps for
// each primitive quartet.  On the interval of one Tk that whole procedure is a
// polynomial in x = Tk/10 - T times known functions, so its value F_M is
// tabulated instead, per (M, Q / 3, Tk), as a polynomial of degree 6 (7 for
// M >= 2, the last coefficient in a float) in x, |x| <= 0.05: the series to
// degree 9, telescoped.  Against the procedure in 80 bits (400,000 T below 12 for
// each M and Q, all orders) the largest relative error grows with Q: 1.1e-16 for
// Q = 0, at most 1.4, 1.4, 1.8 and 2.2e-15 for 3, 6, 9 and 12; the recursion in
// doubles had 1.4e-16, 1.4, 2.0, 2.6 and 3.1e-15, and was in no row better.
//
// One block of FT_BLOCK per M = 0..4: FT_POLY coefficients ([Q / 3][Tk][power];
// seven, an odd stride, spread a wavefront's rows over the LDS banks), then the
// FT_TOP floats of degree 7 (Q >= 3: Q = 0 is the Taylor sum itself, degree 6).
// After the blocks, at FT_EG: e^{-k/10}, k = 0..600 (e^{-T} for T < 60, the
// largest T at which it is used, 2Q + 36 with Q <= 12, from one entry and a
// short series), then the coefficients of BoysG's g(T) = c0 + c1/T + c2/T^2 +
// c3/T^3 on its four ranges of T (12-15, 15-18, 18-24, 24 on); at FT_RAW the
// record's Boys values, which the blocks are made from.
constexpr int FT_NC = 7, FT_NQ = 5;
constexpr int FT_POLY = FT_NQ * FT_NT * FT_NC + 1;         // even
constexpr int FT_TOP = (FT_NQ - 1) * FT_NT / 2;            // in doubles
constexpr int FT_BLOCK = FT_POLY + FT_TOP;
constexpr int FT_NE = 601, FT_EGN = FT_NE + 17;            // even
constexpr int FT_EG = 5 * FT_BLOCK, FT_RAW = FT_EG + FT_EGN, FT_RAWN = FT_NT * FT_NM;
constexpr int FT_TOTAL = FT_RAW + FT_RAWN;

// The tables of one order M, wherever they lie
struct BoysTab {
    const double *poly, *eg;
    const float *top;
};
// in the full array
template <int M>
__host__ __device__ __forceinline__ BoysTab boys_tab(const double *full) {
    const double *b = full + M * FT_BLOCK;
    return {b, full + FT_EG, reinterpret_cast<const float *>(b + FT_POLY)};
}
template <int M>
__host__ __device__ __forceinline__ BoysTab boys_tab(const BoysTab &t) {
    return t;
}
// staged for a kernel: polynomials, e and g, and the degree-7 floats for M >= 2
// (four workgroups per CU)
constexpr int ft_staged(int M) { return FT_POLY + FT_EGN + (M >= 2 ? FT_TOP : 0); }
static_assert(4 * sizeof(double) * ft_staged(4) <= 160 * 1024, "LDS of four workgroups");

// Cartesian components up to l = 2: 0 s | 1 x 2 y 3 z | 4 xx 5 xy 6 xz 7 yy 8 yz 9 zz
MYQC_HD constexpr int cexp(int idx, int d) {
    // exponents (x,y,z) per component
    return (d == 0) ? (idx == 1 ? 1 : idx == 4 ? 2 : (idx == 5 || idx == 6) ? 1 : 0)
         : (d == 1) ? (idx == 2 ? 1 : idx == 7 ? 2 : (idx == 5 || idx == 8) ? 1 : 0)
                    : (idx == 3 ? 1 : idx == 9 ? 2 : (idx == 6 || idx == 8) ? 1 : 0);
}
MYQC_HD constexpr int lvl(int idx) { return idx == 0 ? 0 : idx < 4 ? 1 : 2; }
MYQC_HD constexpr int ncart(int l) { return (l + 1) * (l + 2) / 2; }
MYQC_HD constexpr int nupto(int l) { return (l + 1) * (l + 2) * (l + 3) / 6; }  // components of level <= l
MYQC_HD constexpr int first(int l) { return nupto(l - 1 < 0 ? -1 : l - 1) * (l > 0); }
// index of the component with exponents (x,y,z), total <= 2
MYQC_HD constexpr int cidx(int x, int y, int z) {
    return (x + y + z == 0) ? 0
         : (x + y + z == 1) ? (x ? 1 : y ? 2 : 3)
         : (x == 2 ? 4 : (x == 1 && y == 1) ? 5 : (x == 1 && z == 1) ? 6 : y == 2 ? 7 : (y == 1 && z == 1) ? 8 : 9);
}
// component minus one unit along d (-1 if none)
MYQC_HD constexpr int lower(int idx, int d) {
    return cexp(idx, d) == 0 ? -1
         : cidx(cexp(idx, 0) - (d == 0), cexp(idx, 1) - (d == 1), cexp(idx, 2) - (d == 2));
}
// component plus one unit along d (level <= 2 only)
MYQC_HD constexpr int raise(int idx, int d) {
    return cidx(cexp(idx, 0) + (d == 0), cexp(idx, 1) + (d == 1), cexp(idx, 2) + (d == 2));
}
// the direction used to build a component by recursion: its first nonzero axis
MYQC_HD constexpr int bdir(int idx) { return cexp(idx, 0) ? 0 : cexp(idx, 1) ? 1 : 2; }

// 1/sqrt(x) for x > 0 in the normal range: the device's reciprocal square
// root estimate y refined by one second-order step, y + y e (1/2 + 3/8 e)
// with e = 1 - x y^2 (the series of (1 - e)^(-1/2)), or the host's
// 1/sqrt.  No handling of 0, infinity or denormals: every caller passes a
// sum of Gaussian exponents or a Boys argument above 12.
MYQC_HD double rsqrt_hd(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
#else
    return 1.0 / sqrt(x);
#endif
}

// 1/x from r = rsqrt_hd(x): r^2 and one Newton-Raphson step (within about an
// ulp of the quotient), one transcendental for both.  The host divides.
MYQC_HD double recip_rsq(double x, double r) {
#if defined(__HIP_DEVICE_COMPILE__)
    const double y = r * r;
    return fma(y, fma(-x, y, 1.0), y);
#else
    return 1.0 / x;
#endif
}

// a b for 0 <= a, b < 2^24
MYQC_HD int mul24(int a, int b) {
#if defined(__HIP_DEVICE_COMPILE__)
    return (int)__umul24((unsigned)a, (unsigned)b);
#else
    return a * b;
#endif
}

// The part of the array from FT_EG on, which comes from the host: e, g and the
// record's values (Ft(Tk, m) at Tk + 121 m).
inline void boys_inputs(const double *Ftab, double *e) {
    for (int k = 0; k < FT_NE; ++k) e[k] = std::exp(-0.1 * k);
    // BoysG (auxilary.f90:271-283); beyond T = 30 the reference's g is
    // undefined and 0.49 is used (changes F_0 by at most 3e-15 |g|)
    const double gc[16] = {0.4999489092, -0.2473631686, 0.321180909, -0.3811559346,
                           0.4998436875, -0.24249438,   0.24642845,  0.0,
                           0.499093162,  -0.2152832,    0.0,         0.0,
                           0.490,        0.0,           0.0,         0.0};
    for (int k = 0; k < 16; ++k) e[FT_NE + k] = gc[k];
    e[FT_NE + 16] = 0.0;
    for (int k = 0; k < FT_RAWN; ++k) e[FT_EGN + k] = Ftab[k];
}

// Row (q = Q / 3, Tk) of every block.  a[k]: the coefficients of F_j about Tk,
// first F_Q's Taylor terms Ft(Tk, Q + k) / k! to k = 6 as the reference sums
// them (auxilary.f90:152-155), then F_j = (2 T F_{j+1} + e^{-T}) / (2j + 1)
// (:158-160) with T = Tk/10 - x and e^{-T} = e^{-Tk/10} e^x.  Orders above Q
// are never formed: their row holds F_Q.
MYQC_HD void boys_row(double *full, int q, int Tk) {
    constexpr int ND = 10;
    constexpr double h = 0.05;
    const double *F = full + FT_RAW + Tk;
    const int Q = 3 * q;
    const double T0 = Tk / 10.0, E = full[FT_EG + Tk];
    double a[ND], ek[ND];
    double f = 1.0;
#pragma unroll
    for (int k = 0; k < ND; ++k) {
        if (k > 0) f *= k;
        a[k] = k <= 6 ? F[FT_NT * (Q + k)] / f : 0.0;
        ek[k] = E / f;
    }
    for (int j = Q; j >= 0; --j) {
        if (j < Q) {
            const double d = 1.0 / (2.0 * j + 1.0);
#pragma unroll
            for (int k = ND - 1; k >= 0; --k) a[k] = (2.0 * T0 * a[k] - (k > 0 ? 2.0 * a[k > 0 ? k - 1 : 0] : 0.0) + ek[k]) * d;
        }
        if (j > 4) continue;
        double b[ND], hk = 1.0;
#pragma unroll
        for (int k = 0; k < ND; ++k) {
            b[k] = a[k] * hk;
            hk *= h;
        }
        // u^9, u^8 (and u^7) by the Chebyshev polynomials of their degree
        b[7] += b[9] * (576.0 / 256.0);
        b[5] -= b[9] * (432.0 / 256.0);
        b[3] += b[9] * (120.0 / 256.0);
        b[1] -= b[9] * (9.0 / 256.0);
        b[6] += b[8] * 2.0;
        b[4] -= b[8] * 1.25;
        b[2] += b[8] * 0.25;
        b[0] -= b[8] * (1.0 / 128.0);
        for (int M = j; M <= (j == Q ? 4 : j); ++M) {
            double c5 = b[5], c3 = b[3], c1 = b[1];
            if (M < 2 || q == 0) {
                c5 += b[7] * 1.75;
                c3 -= b[7] * 0.875;
                c1 += b[7] * (7.0 / 64.0);
            }
            double *r = full + M * FT_BLOCK + (q * FT_NT + Tk) * FT_NC;
            constexpr double ih = 20.0;
            r[0] = b[0];
            r[1] = c1 * ih;
            r[2] = b[2] * (ih * ih);
            r[3] = c3 * (ih * ih * ih);
            r[4] = b[4] * (ih * ih * ih * ih);
            r[5] = c5 * (ih * ih * ih * ih * ih);
            r[6] = b[6] * (ih * ih * ih * ih * ih * ih);
            if (q > 0)
                reinterpret_cast<float *>(full + M * FT_BLOCK + FT_POLY)[(q - 1) * FT_NT + Tk] =
                    (float)(b[7] * (ih * ih * ih * ih * ih * ih * ih));
        }
    }
}

// The whole array on the host
inline std::vector<double> build_ftT(const double *Ftab) {
    std::vector<double> full(FT_TOTAL);
    boys_inputs(Ftab, full.data() + FT_EG);
    for (int q = 0; q < FT_NQ; ++q)
        for (int Tk = 0; Tk < FT_NT; ++Tk) boys_row(full.data(), q, Tk);
    return full;
}

// Boys F_0..F_M(T) as the reference computes them at order Q (a multiple of 3,
// at most 12: sets have max L <= 1, which is checked when the system is built,
// and Q = 3 (sum of four set L's)).  ft: the array, or order M's tables.
template <int M, typename FT>
MYQC_HD void boys_ref(int Q, double T, const FT &ft, double (&F)[M + 1]) {
    const BoysTab tab = boys_tab<M>(ft);
    // Tk = NINT(10 T) (T >= 0; T clamped to 60, beyond every table use) and
    // x = Tk / 10 - T, |x| <= 0.05, with 1/10 in two doubles
    const double Tc = T < 60.0 ? T : 60.0;
    const double tkd = floor(fma(Tc, 10.0, 0.5));
    const int Tk = (int)tkd;
    const double x = fma(tkd, -0x1.999999999999ap-58, fma(tkd, 0.1, -Tc));
    // e^{-T} feeds the downward recursion below T = 12 (M > 0) and the
    // asymptotic form up to 2Q + 36; one evaluation serves both branches (the
    // lanes of a wavefront usually fall on both sides of T = 12):
    // e^{-T} = e^{-Tk/10} e^x with the Taylor series of e^x to x^7 (the next
    // term is below 1e-15 relative); to x^5 for M = 0, where it enters F_0 only
    // above T = 12, as at most 1e-6 of it
    double e = 0.0;
    if (((M > 0 && Q > 0) || T >= 12.0) && T < 2.0 * Q + 36.0) {
        double s = 1.0 / 120.0;
        if constexpr (M > 0) s = fma(fma(1.0 / 5040.0, x, 1.0 / 720.0), x, s);
        s = fma(s, x, 1.0 / 24.0);
        s = fma(s, x, 1.0 / 6.0);
        s = fma(s, x, 0.5);
        s = fma(s, x, 1.0);
        s = fma(s, x, 1.0);
        e = tab.eg[Tk] * s;
    }
    if (T < 12.0) {
        const int q = Q / 3, row = q * FT_NT + Tk;
        const double *r = tab.poly + mul24(row, FT_NC);
        double fq = r[6];
        if constexpr (M >= 2) fq = fma(q > 0 ? (double)tab.top[max(row - FT_NT, 0)] : 0.0, x, fq);
#pragma unroll
        for (int k = 5; k >= 0; --k) fq = fma(fq, x, r[k]);
        // fq holds F_top; the reference never forms F_j for j > Q, and callers
        // only read F_j for j <= Q
        const int top = M > 0 && Q < M ? Q : M;
        const double t2 = 2.0 * T;
#pragma unroll
        for (int j = M; j >= 0; --j) {
            if (j > top) F[j] = 0.0;
            else if (j == top) F[j] = fq;
            else F[j] = (t2 * F[j + 1] + e) * (1.0 / (2.0 * j + 1.0));
        }
    } else {
        const double half_sqrt_pi = 0.5 * sqrt(PI_SP);
        const double rt = rsqrt_hd(T);
        const double iT = rt * rt;
        const double it2 = 0.5 * iT;
        if (T < 2.0 * Q + 36.0) {
            // auxilary.f90:181-187 with BoysG (:271-283): g's coefficients
            // for T's range from the staged table, one polynomial for every
            // lane (no branch per range)
            const int rg = (T >= 15.0) + (T >= 18.0) + (T >= 24.0);
            const double *gc = tab.eg + FT_NE + 4 * rg;
            const double g = fma(fma(fma(gc[3], iT, gc[2]), iT, gc[1]), iT, gc[0]);
            F[0] = half_sqrt_pi * rt - e * g * iT;
#pragma unroll
            for (int j = 1; j <= M; ++j) F[j] = it2 * ((2.0 * (j - 1) + 1.0) * F[j - 1] - e);
        } else {
            F[0] = half_sqrt_pi * rt;
#pragma unroll
            for (int j = 1; j <= M; ++j) F[j] = it2 * (2.0 * (j - 1) + 1.0) * F[j - 1];
        }
    }
}

// One primitive pair of a shell pair (first shell carries the larger L).
struct PrimPair {
    double p;        // alpha + beta
    double P[3];     // Gaussian product centre
    double PA[3];    // P - A (A = centre of the first shell)
    double K;        // EIJ * c_a * c_b  (normalised contraction weights folded in)
    double EIJ;      // exp(-alpha beta |AB|^2 / p): the reference's pair screen factor
    double beta;     // exponent of the second shell's primitive (kinetic energy)
    double ip;       // 1 / p
    double KI;       // K / p
    // default construction leaves the fields unset: arrays of primitive pairs
    // are sized before they are filled
    MYQC_HD PrimPair() {}
};

// Contracted shell pair.
struct ShellPair {
    double AB[3];    // A - B
    int pp0;         // first PrimPair
    int npp;         // number of primitive pairs
    int ao_a, ao_b;  // first AO of each shell
    int la, lb;      // angular momentum of each shell (la >= lb)
    int bl;          // sum of the two shells' set max-L (Boys order Q = 3*(bl_bra+bl_ket))
    int same;        // both shells identical
    int sa, sb;      // shell indices of the first and second shell
};

// Contracted [e0|f0] for e in levels LA..LA+LB and f in LC..LC+LD, accumulated
// over all primitive quartets of the shell quartet (bra, ket).
template <int LA, int LB, int LC, int LD>
struct QuartetAcc {
    static constexpr int EB = LA + LB, EK = LC + LD, M = EB + EK;
    static constexpr int E0 = first(LA), NE = nupto(EB) - E0;
    static constexpr int F0 = first(LC), NF = nupto(EK) - F0;
    double v[NE][NF];
};

// One primitive quartet (b k) of a shell quartet added into acc: the Boys
// values, the bra vertical recursion [e0|00]^(m), the ket vertical recursion
// [e0|f0]^(m), and the targets.  Q: the Boys order rule of the shell
// quartet; c0 = 2 pi^2.5.
template <int LA, int LB, int LC, int LD, typename FT>
MYQC_HD __forceinline__ void prim_quartet(const PrimPair &b, const PrimPair &k, int Q, double c0,
                                          const FT &ftT, QuartetAcc<LA, LB, LC, LD> &acc) {
    using A = QuartetAcc<LA, LB, LC, LD>;
    constexpr int EB = A::EB, EK = A::EK, M = A::M;
    constexpr int NB = nupto(EB);
    const double p = b.p, q = k.p, pq = p + q;
    const double rsq = rsqrt_hd(pq);
    const double ipq = recip_rsq(pq, rsq);
    const double rho = p * q * ipq;
    double PQ[3], WP[3], WQ[3], QC[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        PQ[d] = b.P[d] - k.P[d];
        // W = (pP + qQ)/(p+q):  W - P = -q/(p+q) PQ,  W - Q = p/(p+q) PQ
        WP[d] = -q * ipq * PQ[d];
        WQ[d] = p * ipq * PQ[d];
        QC[d] = k.PA[d];
    }
    const double T = rho * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]);
    const double pref = c0 * k.KI * (b.KI * rsq);
    double F[M + 1];
    boys_ref<M>(Q, T, ftT, F);
    // bra vertical recursion [e0|00]^(m)
    double Vb[NB][M + 1];
#pragma unroll
    for (int m = 0; m <= M; ++m) Vb[0][m] = pref * F[m];
    if constexpr (EB > 0) {
        const double i2p = 0.5 * b.ip, rp = q * ipq;
#pragma unroll
        for (int idx = 1; idx < NB; ++idx) {
            const int d = bdir(idx), lo = lower(idx, d);
            const int am1 = cexp(lo, d);
#pragma unroll
            for (int m = 0; m <= M - lvl(idx); ++m) {
                double v = b.PA[d] * Vb[lo][m] + WP[d] * Vb[lo][m + 1];
                if (am1 > 0) {
                    const int lo2 = lower(lo, d);
                    v += am1 * i2p * (Vb[lo2][m] - rp * Vb[lo2][m + 1]);
                }
                Vb[idx][m] = v;
            }
        }
    }
    // ket vertical recursion [e0|f0]^(m), then accumulate the targets
    if constexpr (EK == 0) {
#pragma unroll
        for (int e = A::E0; e < NB; ++e) acc.v[e - A::E0][0] += Vb[e][0];
    } else {
        constexpr int NK = nupto(EK);
        const double i2q = 0.5 * k.ip, rq = p * ipq, i2pq = 0.5 * ipq;
        double W[NB][NK][M + 1];
#pragma unroll
        for (int e = 0; e < NB; ++e)
#pragma unroll
            for (int m = 0; m <= M - lvl(e); ++m) W[e][0][m] = Vb[e][m];
#pragma unroll
        for (int f = 1; f < NK; ++f) {
            const int d = bdir(f), lo = lower(f, d);
            const int cm1 = cexp(lo, d);
#pragma unroll
            for (int e = 0; e < NB; ++e) {
#pragma unroll
                for (int m = 0; m <= M - lvl(e) - lvl(f); ++m) {
                    double v = QC[d] * W[e][lo][m] + WQ[d] * W[e][lo][m + 1];
                    if (cm1 > 0) {
                        const int lo2 = lower(lo, d);
                        v += cm1 * i2q * (W[e][lo2][m] - rq * W[e][lo2][m + 1]);
                    }
                    if (cexp(e, d) > 0) {
                        const int el = lower(e, d);
                        v += cexp(e, d) * i2pq * W[el][lo][m + 1];
                    }
                    W[e][f][m] = v;
                }
            }
        }
#pragma unroll
        for (int e = A::E0; e < NB; ++e)
#pragma unroll
            for (int f = A::F0; f < NK; ++f) acc.v[e - A::E0][f - A::F0] += W[e][f][0];
    }
}

// SCREEN = false skips the reference's primitive-pair screen: used for the
// Schwarz factors, since a primitive pair dropped from (ab|ab) by
// EIJ^2 < 1e-14 can survive EIJ*EGH >= 1e-14 against a compact ket pair.
// The ket's primitive pairs come from kprim(j), j < ket.npp.
template <int LA, int LB, int LC, int LD, bool SCREEN = true, typename KF, typename FT>
MYQC_HD void quartet_prims_f(const ShellPair &bra, const ShellPair &ket, const PrimPair *__restrict__ ppb,
                             KF &&kprim, const FT &ftT, QuartetAcc<LA, LB, LC, LD> &acc) {
    using A = QuartetAcc<LA, LB, LC, LD>;
    const int Q = 3 * (bra.bl + ket.bl);
#pragma unroll
    for (int e = 0; e < A::NE; ++e)
#pragma unroll
        for (int f = 0; f < A::NF; ++f) acc.v[e][f] = 0.0;
    const double c0 = 2.0 * pow(PI_SP, 2.5);
    // ket primitives outer: a lane's own ket data is loaded once per quartet,
    // and the inner loop reads the bra's primitives, whose addresses the lanes
    // of a wavefront (one bra pair, consecutive kets) mostly share.  A pair's
    // primitives stand with the largest screen factor first (system.h), so a
    // row ends at the first one screened (int2e.f90:257), and the rows at the
    // first that starts with one: a third to a half of the primitive quartets
    // survive.  The next primitive of either side is loaded before the work on
    // the current one: where the lanes' bras differ (batch.hip), the wait for
    // each was a fifth of the time.
    const PrimPair *bp = ppb + bra.pp0;
    const PrimPair b0 = bp[0];
    PrimPair kn = kprim(0);
    for (int j = 0; j < ket.npp; ++j) {
        const PrimPair k = kn;
        if (SCREEN && b0.EIJ * k.EIJ < 1.0e-14) break;
        kn = kprim(j + 1 < ket.npp ? j + 1 : j);
        PrimPair b = b0;
        for (int i = 1; ; ++i) {
            const PrimPair bn = bp[i < bra.npp ? i : 0];
            prim_quartet<LA, LB, LC, LD>(b, k, Q, c0, ftT, acc);
            if (i >= bra.npp || (SCREEN && bn.EIJ * k.EIJ < 1.0e-14)) break;
            b = bn;
        }
    }
}

// The same sum split over SPLIT lanes: lane `sub` of the quartet's group
// takes the primitive quartets t = j npp_bra + i with t = sub (mod SPLIT);
// the group's partial sums are added afterwards (split_reduce on the device).
template <int LA, int LB, int LC, int LD, int SPLIT, bool SCREEN = true, typename KF, typename FT>
MYQC_HD void quartet_prims_split(const ShellPair &bra, const ShellPair &ket, const PrimPair *__restrict__ ppb,
                                 KF &&kprim, const FT &ftT, QuartetAcc<LA, LB, LC, LD> &acc,
                                 int sub) {
    using A = QuartetAcc<LA, LB, LC, LD>;
    const int Q = 3 * (bra.bl + ket.bl);
#pragma unroll
    for (int e = 0; e < A::NE; ++e)
#pragma unroll
        for (int f = 0; f < A::NF; ++f) acc.v[e][f] = 0.0;
    const double c0 = 2.0 * pow(PI_SP, 2.5);
    const int nbp = bra.npp, total = nbp * ket.npp;
    int j = 0, i = sub;
    while (i >= nbp && nbp > 0) {
        i -= nbp;
        ++j;
    }
    for (int t = sub; t < total; t += SPLIT) {
        const PrimPair k = kprim(j);
        const PrimPair b = ppb[bra.pp0 + i];
        if (!(SCREEN && b.EIJ * k.EIJ < 1.0e-14))
            prim_quartet<LA, LB, LC, LD>(b, k, Q, c0, ftT, acc);   // int2e.f90:257
        i += SPLIT;
        while (i >= nbp) {
            i -= nbp;
            ++j;
        }
    }
}

template <int LA, int LB, int LC, int LD, bool SCREEN = true, typename FT>
MYQC_HD void quartet_prims(const ShellPair &bra, const ShellPair &ket, const PrimPair *__restrict__ ppb,
                           const PrimPair *__restrict__ ppk, const FT &ftT, QuartetAcc<LA, LB, LC, LD> &acc) {
    quartet_prims_f<LA, LB, LC, LD, SCREEN>(bra, ket, ppb, [&](int j) { return ppk[ket.pp0 + j]; }, ftT, acc);
}

// Horizontal recursion: contracted (ab|cd) with a,b,c,d component indices
// within each shell (s: 0; p: 0,1,2 = x,y,z).  out[((a*NBb + b)*NCc + c)*NDd + d].
template <int LA, int LB, int LC, int LD>
MYQC_HD void quartet_hrr(const QuartetAcc<LA, LB, LC, LD> &acc, const double AB[3], const double CD[3],
                         double *out) {
    using A = QuartetAcc<LA, LB, LC, LD>;
    constexpr int na = ncart(LA), nb = ncart(LB), nc = ncart(LC), nd = ncart(LD);
    // ket HRR for every bra level-(LA..LA+LB) component e: I[e][c][d]
    double I[A::NE][nc][nd];
#pragma unroll
    for (int e = 0; e < A::NE; ++e)
#pragma unroll
        for (int c = 0; c < nc; ++c)
#pragma unroll
            for (int d = 0; d < nd; ++d) {
                const int ci = first(LC) + c;       // component index of c
                if constexpr (LD == 0) {
                    I[e][c][d] = acc.v[e][ci - A::F0];
                } else {
                    // (e0|c p_d) = [e0|(c+1_d)0] + CD_d [e0|c0]
                    I[e][c][d] = acc.v[e][raise(ci, d) - A::F0] + CD[d] * acc.v[e][ci - A::F0];
                }
            }
#pragma unroll
    for (int a = 0; a < na; ++a)
#pragma unroll
        for (int b = 0; b < nb; ++b)
#pragma unroll
            for (int c = 0; c < nc; ++c)
#pragma unroll
                for (int d = 0; d < nd; ++d) {
                    const int ai = first(LA) + a;
                    double v;
                    if constexpr (LB == 0) {
                        v = I[ai - A::E0][c][d];
                    } else {
                        v = I[raise(ai, b) - A::E0][c][d] + AB[b] * I[ai - A::E0][c][d];
                    }
                    out[((a * nb + b) * nc + c) * nd + d] = v;
                }
}

// Degeneracy weight of element (i,j|k,l) of a shell-quartet block so that
// every unique integral is visited once in the J/K digestion: 0 for a repeat
// within a block whose shells or pairs coincide, else 1/2 per index equality
// (i==j, k==l, (ij)==(kl)).
MYQC_HD double block_weight(int a, int b, int c, int d, int same_ab, int same_cd, int same_pair, int nb, int nd,
                            int i, int j, int k, int l) {
    if (same_ab && a > b) return 0.0;
    if (same_cd && c > d) return 0.0;
    if (same_pair && (a * nb + b) > (c * nd + d)) return 0.0;
    double w = 1.0;
    if (i == j) w *= 0.5;
    if (k == l) w *= 0.5;
    if ((i == k && j == l) || (i == l && j == k)) w *= 0.5;
    return w;
}

}  // namespace myqc
