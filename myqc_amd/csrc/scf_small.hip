// scf_small.hip -- the dense part of an RHF iteration of a small system in one
// launch of one workgroup.
//
// Up to about a hundred functions, a matrix product is a fraction of a
// microsecond of one CU's matrix cores, and the loop of scf.hip is bounded by
// its launches (about 55 per iteration at 4 us and more, 30 of them
// purification steps) and its two synchronisations.  Here the matrices live in
// LDS: one launch forms F, its orthonormal-basis form, the DIIS error and
// extrapolation, the purified projector (trace-correcting, as in sp2.hip) and
// the next density, and writes the scalars the host decides by to pinned
// memory; one synchronisation per iteration.  X = S^-1/2 (coupled
// Newton-Schulz, as in scf.hip) and the final orbitals (cyclic Jacobi) are one
// launch each.
//
// Products: v_mfma_f64_16x16x4f64 on 16 x 16 tiles, a wavefront per tile or
// two.  The step's right operands are symmetric and read by rows, so that both
// operands' fragments are 16 consecutive doubles of an LDS column; the leading
// dimension is 16 mod 32 doubles where it fits, which puts the two k's of a
// half-wavefront's read in distinct banks.  Rows and columns beyond n are
// zero.
//
// Why up to 84: from there on a purification step spread over the chip (5 to 7
// us) is no slower than one CU's matrix cores, and the library's eigenvectors
// no slower than one CU's Jacobi (n = 56: 112 us for a step of about 36
// purifications, 656 for the orbitals).  Whole solves of water clusters with
// helium, here / by the general loop, ms, in FP64 from the core guess and mixed
// from the learned one: n = 56 4.0 / 7.0 and 4.1 / 6.8; 70 7.6 / 10.1 and 5.6 / 6.9;
// 80 7.5 / 8.5 and 6.3 / 7.1; 84 9.5 / 9.8 and 7.1 / 7.2 (never the slower of
// three clusters); 86 9.3 / 9.5 and 7.3 / 7.3; 88 10.0 / 9.8 and 7.5 / 7.2; 96
// 11.6 / 11.2 and 8.3 / 7.6.  One water (n = 7) 4.04 -> 1.37.
#include <algorithm>

#include "scf_small.h"
#include "small_dense.h"

namespace myqc {

// enough wavefronts for a tile or two each
template <int NP>
using Sm = DenseLds<NP, NP <= 32 ? 4 : NP <= 48 ? 8 : 16>;

template <int NP>
__global__ __launch_bounds__(Sm<NP>::THREADS) void k_small_step(SmallStep a) {
    constexpr int LD = Sm<NP>::LD, MD = 8, MT = Sm<NP>::MT, MU = Sm<NP>::MU, TH = Sm<NP>::THREADS, WV = Sm<NP>::WAVES;
    __shared__ double sA[NP * LD], sB[NP * LD];
    __shared__ double s_red[WV], s_part[16 * WV], s_sum[WV][MD + 2], s_c[MD], s_tot[MD + 2];
    const int n = a.n, nn = n * n, t = threadIdx.x, lane = t & 63, w = t >> 6;
    d4_t acc[MT];
    // F = H + G, with the energy sums and the density change
    double e0 = 0.0, e1 = 0.0, dd = 0.0;
    for (int e = t; e < NP * NP; e += TH) {
        const int i = e % NP, j = e / NP;
        double f = 0.0;
        if (i < n && j < n) {
            const int q = i + n * j;
            const double h = a.H[q];
            f = h;
            if (!a.core) {
                f += a.g_half ? a.G[q] + a.G[j + n * i] : a.G[q];
                const double d = a.D[q];
                e0 += d * f;
                e1 += d * h;
                if (a.with_dd) dd = fmax(dd, fabs(d - a.Dprev[q]));
            }
        }
        sB[i + LD * j] = f;
    }
    load<Sm<NP>>(sA, a.X, n);
    __syncthreads();
    // Fo = X F X: W = X F (F symmetric), then W X
    product<Sm<NP>>(sA, sB, acc);
    __syncthreads();
    to_lds<Sm<NP>>(sB, acc);   // W
    __syncthreads();
    product<Sm<NP>>(sB, sA, acc);
    __syncthreads();
    to_lds<Sm<NP>>(sA, acc);   // Fo
    double err = 0.0;
    if (!a.core) {
        double *fs = a.hF + (size_t)nn * a.head, *es = a.hE + (size_t)nn * a.head;
        each<Sm<NP>>(acc, [&](int i, int j, double v) {
            if (i < n && j < n) fs[i + n * j] = v;
        });
        load<Sm<NP>>(sB, a.Do, n);
        __syncthreads();
        // the error Fo Do - Do Fo, and its products with the history
        product<Sm<NP>>(sA, sB, acc);
        __syncthreads();
        to_lds<Sm<NP>>(sB, acc);
        __syncthreads();
        double dot[MD];
#pragma unroll
        for (int q = 0; q < MD; ++q) dot[q] = 0.0;
        for (int e = t; e < nn; e += TH) {
            const int i = e % n, j = e / n;
            const double v = sB[i + LD * j] - sB[j + LD * i];
            es[e] = v;
#pragma unroll
            for (int q = 0; q < MD; ++q)
                if (q < a.hn) dot[q] += v * (q == a.head ? v : a.hE[(size_t)nn * q + e]);
        }
        // all sums at once
        const double x0 = wave_total(e0), x1 = wave_total(e1), xd = wave_largest(dd);
#pragma unroll
        for (int q = 0; q < MD; ++q) {
            const double v = wave_total(dot[q]);
            if (lane == 0) s_sum[w][q] = v;
        }
        if (lane == 0) {
            s_sum[w][MD] = x0;
            s_sum[w][MD + 1] = x1;
            s_red[w] = xd;
        }
        __syncthreads();
        if (t < MD + 2) {
            double v = 0.0;
            for (int q = 0; q < WV; ++q) v += s_sum[q][t];
            s_tot[t] = v;
            if (t < MD) {
                a.out[SO_B + t] = v;
                if (t < a.hn) {
                    a.B[a.head * MD + t] = v;
                    a.B[t * MD + a.head] = v;
                }
            } else {
                a.out[t == MD ? SO_DF : SO_DH] = v;
            }
        }
        if (t == 0) {
            double v = 0.0;
            for (int q = 0; q < WV; ++q) v = fmax(v, s_red[q]);
            a.out[SO_DD] = v;
        }
        __syncthreads();   // B's new row is written (by this workgroup)
        if (w == 0) diis_wave(a.B, a.hn, a.head, s_c);
        __syncthreads();
        err = sqrt(fabs(s_tot[a.head]));
        const double sh = err > a.shift_err ? a.shift : 0.0;
        // the extrapolated Fock matrix (with the level shift)
        for (int e = t; e < NP * NP; e += TH) {
            const int i = e % NP, j = e / NP;
            double v = 0.0;
            if (i < n && j < n) {
                const int q = i + n * j;
#pragma unroll
                for (int h = 0; h < MD; ++h)
                    if (h < a.hn) v += s_c[h] * a.hF[(size_t)nn * h + q];
                if (sh != 0.0) v += (i == j ? sh : 0.0) - sh * a.Do[q];
                a.Fx[q] = v;
            }
            sA[i + LD * j] = v;
        }
    } else {
        each<Sm<NP>>(acc, [&](int i, int j, double v) {
            if (i < n && j < n) a.Fx[i + n * j] = v;
        });
    }
    __syncthreads();
    // the projector onto the nocc lowest levels (as sp2.hip)
    int ok = 1, steps = 0;
    if (a.nocc == 0 || a.nocc == n) {
        for (int e = t; e < NP * NP; e += TH) {
            const int i = e % NP, j = e / NP;
            sA[i + LD * j] = i == j && i < n && a.nocc == n ? 1.0 : 0.0;
        }
        __syncthreads();
    } else {
        ok = purify<Sm<NP>>(sA, sB, n, a.nocc, 120, s_red, s_part, steps);
        __syncthreads();
    }
    if (t == 0) {
        a.out[SO_OK] = ok;
        a.out[SO_STEPS] = steps;
    }
    if (!ok) return;   // (uniform) the host takes the eigenvectors of Fx
    // the projector, and D = 2 X P X
    for (int e = t; e < nn; e += TH) a.Don[e] = sA[e % n + LD * (e / n)];
    load<Sm<NP>>(sB, a.X, n);
    __syncthreads();
    product<Sm<NP>>(sB, sA, acc);   // X P
    __syncthreads();
    to_lds<Sm<NP>>(sA, acc);
    __syncthreads();
    product<Sm<NP>>(sA, sB, acc);
    each<Sm<NP>>(acc, [&](int i, int j, double v) {
        if (i < n && j < n) a.Dnext[i + n * j] = 2.0 * v;
    });
}

// X = S^-1/2 and Xi = S^1/2 (small_dense.h); out[0] = 1, or 0 if they were not reached
template <int NP>
__global__ __launch_bounds__(Sm<NP>::THREADS) void k_small_inv_sqrt(int n, const double *__restrict__ S, double *X,
                                                                    double *Xi, double *Y, double *Z, double *out) {
    __shared__ double sM[2 * NP * (NP + 1)], s_red[Sm<NP>::WAVES];
    const bool ok = inv_sqrt_ns<Sm<NP>>(n, S, X, Xi, Y, Z, sM, s_red, 40);
    if (threadIdx.x == 0) out[0] = ok ? 1.0 : 0.0;
}

// Eigenvalues (ascending) and C = X U by cyclic Jacobi, round-robin pairs: the
// n / 2 rotations of a round are disjoint and each thread applies them to
// whole 2 x 2 blocks in place, two barriers per round.
template <int NP>
__global__ __launch_bounds__(Sm<NP>::THREADS) void k_small_orbitals(int n, const double *__restrict__ Fo,
                                                                    const double *__restrict__ X,
                                                                    double *__restrict__ C, double *__restrict__ eig) {
    constexpr int LD = Sm<NP>::LD, TH = Sm<NP>::THREADS, WV = Sm<NP>::WAVES;
    __shared__ double sA[NP * LD], sU[NP * LD], s_red[WV], s_cos[NP / 2], s_sin[NP / 2];
    __shared__ int s_p[NP / 2], s_q[NP / 2], s_at[NP];
    const int t = threadIdx.x;
    const int npad = n + (n & 1), half = npad >> 1;
    load<Sm<NP>>(sA, Fo, n);
    for (int e = t; e < NP * NP; e += TH) sU[e % NP + LD * (e / NP)] = e % NP == e / NP ? 1.0 : 0.0;
    __syncthreads();
    for (int sweep = 0; sweep < 40; ++sweep) {
        double off = 0.0, dia = 0.0;
        for (int e = t; e < NP * NP; e += TH) {
            const double v = sA[e % NP + LD * (e / NP)];
            if (e % NP == e / NP) dia += v * v;
            else off += v * v;
        }
        off = wg_total<Sm<NP>>(off, s_red);
        dia = wg_total<Sm<NP>>(dia, s_red);
        if (!(off > 1e-30 * dia)) break;
        for (int r = 0; r < npad - 1; ++r) {
            for (int k = t; k < half; k += TH) {
                const int x = k == 0 ? 0 : (k - 1 + r) % (npad - 1) + 1;
                const int y = (npad - 2 - k + r) % (npad - 1) + 1;
                const int p = min(x, y), q = max(x, y);
                double c = 1.0, s = 0.0;
                if (q < n) {
                    const double apq = sA[p + LD * q];
                    if (fabs(apq) > 1e-300) {
                        const double th = (sA[q * (LD + 1)] - sA[p * (LD + 1)]) / (2.0 * apq);
                        const double u = (th >= 0.0 ? 1.0 : -1.0) / (fabs(th) + sqrt(th * th + 1.0));
                        c = 1.0 / sqrt(u * u + 1.0);
                        s = u * c;
                    }
                }
                s_p[k] = p;
                s_q[k] = q;
                s_cos[k] = c;
                s_sin[k] = s;
            }
            __syncthreads();
            // A <- J^T A J on 2 x 2 blocks (rows of pair k1, columns of pair
            // k2); a row or column past n (odd n) is zero and has c = 1
            for (int b = t; b < half * half; b += TH) {
                const int k1 = b % half, k2 = b / half;
                const int p1 = s_p[k1], q1 = s_q[k1], p2 = s_p[k2], q2 = s_q[k2];
                const double c1 = s_cos[k1], s1 = s_sin[k1], c2 = s_cos[k2], s2 = s_sin[k2];
                const double m00 = sA[p1 + LD * p2], m01 = sA[p1 + LD * q2], m10 = sA[q1 + LD * p2],
                             m11 = sA[q1 + LD * q2];
                const double t00 = c1 * m00 - s1 * m10, t01 = c1 * m01 - s1 * m11;
                const double t10 = s1 * m00 + c1 * m10, t11 = s1 * m01 + c1 * m11;
                sA[p1 + LD * p2] = t00 * c2 - t01 * s2;
                sA[p1 + LD * q2] = t00 * s2 + t01 * c2;
                sA[q1 + LD * p2] = t10 * c2 - t11 * s2;
                sA[q1 + LD * q2] = t10 * s2 + t11 * c2;
            }
            for (int b = t; b < n * half; b += TH) {
                const int i = b % n, k = b / n;
                const int p = s_p[k], q = s_q[k];
                const double c = s_cos[k], s = s_sin[k];
                const double up = sU[i + LD * p], uq = sU[i + LD * q];
                sU[i + LD * p] = c * up - s * uq;
                sU[i + LD * q] = s * up + c * uq;
            }
            __syncthreads();
        }
    }
    __syncthreads();
    // ascending order
    if (t < n) {
        const double v = sA[t * (LD + 1)];
        int at = 0;
        // (not a number: after every number, so that each still has its own place)
        auto before = [](double x, double y) { return x < y || (x == x && y != y); };
        for (int j = 0; j < n; ++j) {
            const double u = sA[j * (LD + 1)];
            at += before(u, v) || (!before(v, u) && j < t);
        }
        s_at[t] = at;
        eig[at] = v;
    }
    __syncthreads();
    // C = X U, columns to their places
    load<Sm<NP>>(sA, X, n);
    __syncthreads();
    const int w = t >> 6, lane = t & 63, g = lane >> 4, c = lane & 15;
    for (int tile = w; tile < Sm<NP>::T2; tile += WV) {
        const int ti = tile % Sm<NP>::NT, tj = tile / Sm<NP>::NT;
        d4_t acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < NP; k += 4)
            acc = mfma64(sA[16 * ti + c + LD * (k + g)], sU[k + g + LD * (16 * tj + c)], acc);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = 16 * ti + g + 4 * v, j = 16 * tj + c;
            if (i < n && j < n) C[i + n * s_at[j]] = acc[v];
        }
    }
}

template <typename F>
static int with_np(myqc_ctx *ctx, int n, F f) {
    switch ((n + 15) / 16) {
        case 1: f(std::integral_constant<int, 16>{}); break;
        case 2: f(std::integral_constant<int, 32>{}); break;
        case 3: f(std::integral_constant<int, 48>{}); break;
        case 4: f(std::integral_constant<int, 64>{}); break;
        case 5: f(std::integral_constant<int, 80>{}); break;
        case 6: f(std::integral_constant<int, 96>{}); break;
        default: return set_error(ctx, MYQC_E_ARG, "scf_small: n=%d", n);
    }
    MYQC_HIP(ctx, hipGetLastError());
    return 0;
}

int small_step(myqc_ctx *ctx, const SmallStep &s) {
    return with_np(ctx, s.n, [&](auto np) {
        constexpr int NP = decltype(np)::value;
        k_small_step<NP><<<1, Sm<NP>::THREADS, 0, ctx->stream>>>(s);
    });
}

int small_inv_sqrt(myqc_ctx *ctx, int n, const double *S, double *X, double *Xi, double *Y, double *Z, double *out) {
    return with_np(ctx, n, [&](auto np) {
        constexpr int NP = decltype(np)::value;
        k_small_inv_sqrt<NP><<<1, Sm<NP>::THREADS, 0, ctx->stream>>>(n, S, X, Xi, Y, Z, out);
    });
}

int small_orbitals(myqc_ctx *ctx, int n, const double *Fo, const double *X, double *C, double *eig) {
    return with_np(ctx, n, [&](auto np) {
        constexpr int NP = decltype(np)::value;
        k_small_orbitals<NP><<<1, Sm<NP>::THREADS, 0, ctx->stream>>>(n, Fo, X, C, eig);
    });
}

}  // namespace myqc
