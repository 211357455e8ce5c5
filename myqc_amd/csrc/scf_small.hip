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
// Why up to 96: above, two matrices no longer fit, and from there on a
// purification step spread over the chip (5 to 7 us) is no slower than one
// CU's matrix cores.  Measured, one whole solve: 1 water (n = 7) 4.04 -> 1.37 ms, 8
// waters (n = 56) 9.1 -> 4.4 ms (112 us for a step of about 36 purifications).
#include <algorithm>

#include "scf_small.h"
#include "wave.h"

namespace myqc {

typedef double d4_t __attribute__((ext_vector_type(4)));

template <int NP>
struct Sm {
    static constexpr int LD = NP % 32 == 16 ? NP : NP == 96 ? NP + 1 : NP + 16;
    static constexpr int NT = NP / 16, T2 = NT * NT, TU = NT * (NT + 1) / 2;
    static constexpr int THREADS = NP <= 32 ? 256 : NP <= 48 ? 512 : 1024, WAVES = THREADS / 64;
    static constexpr int MT = (T2 + WAVES - 1) / WAVES, MU = (TU + WAVES - 1) / WAVES;
};

__device__ __forceinline__ d4_t mfma64(double a, double b, d4_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// tile (ti, tj) of A B, B symmetric
template <int NP>
__device__ __forceinline__ d4_t tile_sym(const double *A, const double *B, int ti, int tj) {
    constexpr int LD = Sm<NP>::LD;
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    const double *pa = A + 16 * ti + c + LD * g, *pb = B + 16 * tj + c + LD * g;
    d4_t acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < NP; k += 4) acc = mfma64(pa[LD * k], pb[LD * k], acc);
    return acc;
}

// the wavefront's tiles w, w + WAVES, ... of A B (B symmetric)
template <int NP>
__device__ __forceinline__ void product(const double *A, const double *B, d4_t (&acc)[Sm<NP>::MT]) {
    const int w = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < Sm<NP>::MT; ++q) {
        const int tile = w + q * Sm<NP>::WAVES;
        if (tile < Sm<NP>::T2) acc[q] = tile_sym<NP>(A, B, tile % Sm<NP>::NT, tile / Sm<NP>::NT);
    }
}

// f(row, column, value) over the wavefront's tiles
template <int NP, typename F>
__device__ __forceinline__ void each(const d4_t (&acc)[Sm<NP>::MT], F f) {
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
#pragma unroll
    for (int q = 0; q < Sm<NP>::MT; ++q) {
        const int tile = w + q * Sm<NP>::WAVES;
        if (tile >= Sm<NP>::T2) break;
#pragma unroll
        for (int v = 0; v < 4; ++v)
            f(16 * (tile % Sm<NP>::NT) + g + 4 * v, 16 * (tile / Sm<NP>::NT) + c, acc[q][v]);
    }
}

template <int NP>
__device__ __forceinline__ void to_lds(double *M, const d4_t (&acc)[Sm<NP>::MT]) {
    each<NP>(acc, [&](int i, int j, double v) { M[i + Sm<NP>::LD * j] = v; });
}

// M = scale times the n x n A, zero beyond
template <int NP>
__device__ __forceinline__ void load(double *M, const double *__restrict__ A, int n, double scale = 1.0) {
    for (int e = threadIdx.x; e < NP * NP; e += Sm<NP>::THREADS) {
        const int i = e % NP, j = e / NP;
        M[i + Sm<NP>::LD * j] = (i < n && j < n) ? scale * A[i + n * j] : 0.0;
    }
}

// sum (or maximum) over the workgroup of a value per thread; s: a double per wavefront
template <int NP>
__device__ __forceinline__ double wg_total(double v, double *s) {
    v = wave_total(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
    __syncthreads();
    return wave_total((threadIdx.x & 63) < Sm<NP>::WAVES ? s[threadIdx.x & 63] : 0.0);
}
// sum over each aligned 16 lanes
__device__ __forceinline__ double row_total(double v) {
    v = dpp_add<0xB1>(v);
    v = dpp_add<0x4E>(v);
    v = dpp_add<0x141>(v);
    return dpp_add<0x140>(v);
}
__device__ __forceinline__ double wave_largest(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
    return v;
}
template <int NP>
__device__ __forceinline__ double wg_largest(double v, double *s) {
    v = wave_largest(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
    __syncthreads();
    return wave_largest(s[(threadIdx.x & 63) % Sm<NP>::WAVES]);
}

// Gershgorin bounds of the symmetric matrix in M
template <int NP>
__device__ __forceinline__ void bounds(const double *M, int n, double *s, double &lo, double &hi) {
    // a wavefront per row
    const int lane = threadIdx.x & 63;
    double l = 1e300, h = -1e300;
    for (int i = threadIdx.x >> 6; i < n; i += Sm<NP>::WAVES) {
        double r = 0.0;
        for (int j = lane; j < n; j += 64)
            if (j != i) r += fabs(M[j + Sm<NP>::LD * i]);
        r = wave_total(r);
        const double c = M[i * (Sm<NP>::LD + 1)];
        l = fmin(l, c - r);
        h = fmax(h, c + r);
    }
    lo = -wg_largest<NP>(-l, s);
    hi = wg_largest<NP>(h, s);
}

// DIIS coefficients c_0 .. c_{m-1} of the (m + 1) system, Gauss-Jordan with
// column pivoting, by the first wavefront: lane r holds row r in registers.
// Zeros with c[head] = 1 when the system is singular or m < 2.
__device__ __forceinline__ bool diis_wave(const double *B, int m, int head, double *s_c) {
    constexpr int MD = 8, W = MD + 2;
    const int r = threadIdx.x & 63, N = m + 1;
    double row[W];
#pragma unroll
    for (int k = 0; k < W; ++k) row[k] = 0.0;
    if (r < m) {
#pragma unroll
        for (int k = 0; k < MD; ++k)
            if (k < m) row[k] = B[r * MD + k];
    }
    // columns 0 .. m - 1 the B block, MD the border, MD + 1 the right side
    if (r < m) row[MD] = -1.0;
    if (r == m) {
#pragma unroll
        for (int k = 0; k < MD; ++k)
            if (k < m) row[k] = -1.0;
        row[MD + 1] = -1.0;
    }
    bool used = false, ok = m >= 2;
    int mine = -1;   // the column this lane's row is the pivot of
#pragma unroll
    for (int col = 0; col <= MD; ++col) {
        if (col < MD && col >= m) continue;   // (uniform)
        const double v = (r < N && !used) ? fabs(row[col]) : -1.0;
        double best = v;
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) best = fmax(best, __shfl_xor(best, off, 64));
        best = lane_value(best, 0);   // (rows are lanes 0 .. 8 of the first 16)
        if (!(best >= 1e-300)) ok = false;
        const unsigned long long who = __ballot(r < 16 && v == best);
        const int p = who ? __ffsll((long long)who) - 1 : 0;
        double pr[W];
#pragma unroll
        for (int k = 0; k < W; ++k) pr[k] = lane_value(row[k], p);
        if (r == p) {
            used = true;
            mine = col;
        } else if (r < N) {
            const double f = row[col] / pr[col];
#pragma unroll
            for (int k = 0; k < W; ++k) row[k] -= f * pr[k];
            row[col] = 0.0;
        }
    }
    ok = __ballot(!ok) == 0;
    if (ok) {
#pragma unroll
        for (int k = 0; k < MD; ++k)
            if (mine == k) s_c[k] = row[MD + 1] / row[k];
    } else if (r < MD) {
        s_c[r] = r == head ? 1.0 : 0.0;
    }
    return ok;
}

template <int NP>
__global__ __launch_bounds__(Sm<NP>::THREADS) void k_small_step(SmallStep a) {
    constexpr int LD = Sm<NP>::LD, MD = 8, MT = Sm<NP>::MT, MU = Sm<NP>::MU, TH = Sm<NP>::THREADS, WV = Sm<NP>::WAVES;
    __shared__ double sA[NP * LD], sB[NP * LD];
    __shared__ double s_red[WV], s_part[2][8 * WV], s_sum[WV][MD + 2], s_c[MD], s_tot[MD + 2];
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
                f += a.G[q];
                const double d = a.D[q];
                e0 += d * f;
                e1 += d * h;
                if (a.with_dd) dd = fmax(dd, fabs(d - a.Dprev[q]));
            }
        }
        sB[i + LD * j] = f;
    }
    load<NP>(sA, a.X, n);
    __syncthreads();
    // Fo = X F X: W = X F (F symmetric), then W X
    product<NP>(sA, sB, acc);
    __syncthreads();
    to_lds<NP>(sB, acc);   // W
    __syncthreads();
    product<NP>(sB, sA, acc);
    __syncthreads();
    to_lds<NP>(sA, acc);   // Fo
    double err = 0.0;
    if (!a.core) {
        double *fs = a.hF + (size_t)nn * a.head, *es = a.hE + (size_t)nn * a.head;
        each<NP>(acc, [&](int i, int j, double v) {
            if (i < n && j < n) fs[i + n * j] = v;
        });
        load<NP>(sB, a.Do, n);
        __syncthreads();
        // the error Fo Do - Do Fo, and its products with the history
        product<NP>(sA, sB, acc);
        __syncthreads();
        to_lds<NP>(sB, acc);
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
        each<NP>(acc, [&](int i, int j, double v) {
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
        double lo, hi;
        bounds<NP>(sA, n, s_red, lo, hi);
        const double sc = 1.0 / (hi - lo);
        const int g = lane >> 4, c = lane & 15;
        // the wavefront's upper tiles of P^2
        int ti[MU], tj[MU];
#pragma unroll
        for (int q = 0; q < MU; ++q) {
            int rem = w + q * WV, col = 0;
            while (rem > col) rem -= ++col;
            ti[q] = rem;
            tj[q] = col;
        }
        // tr P and ||P||^2: each 16 lanes' sums go to LDS when P is written,
        // and every wavefront adds the partial sums up for itself
        double tr = 0.0, fr = 0.0;
        __syncthreads();
        for (int e = t; e < NP * NP; e += TH) {
            const int i = e % NP, j = e / NP;
            double v = 0.0;
            if (i < n && j < n) {
                v = ((i == j ? hi : 0.0) - sA[i + LD * j]) * sc;
                fr += v * v;
                if (i == j) tr += v;
            }
            sB[i + LD * j] = v;
        }
        const double nocc = a.nocc;
        int cs = -1;
        ok = 0;
        // P_k and P_{k+1} take turns in the two arrays: one barrier per step
        const double *P = sB;
        double *Pn = sA;
        for (int step = 0; step <= 120; ++step) {
            double *part = s_part[step & 1];
            tr = row_total(tr);
            fr = row_total(fr);
            if (c == 0) {
                part[4 * w + g] = tr;
                part[4 * WV + 4 * w + g] = fr;
            }
            __syncthreads();   // P and its sums are complete; P_{k-1} is free
            const double pt = lane < 4 * WV ? part[lane] : 0.0, pf = lane < 4 * WV ? part[4 * WV + lane] : 0.0;
            d4_t p2[MU];
#pragma unroll
            for (int q = 0; q < MU; ++q)
                if (w + q * WV < Sm<NP>::TU) p2[q] = tile_sym<NP>(P, P, ti[q], tj[q]);
            tr = wave_total(pt);
            fr = wave_total(pf);
            if (cs < 0 && step >= 8 && fabs(tr - fr) < 1e-8 && fabs(tr - nocc) < 1e-6) cs = step;
            if (cs >= 0 && step >= cs + 2) {
                ok = 1;
                steps = step;
                break;
            }
            if (step == 120) break;
            const bool square = fabs(fr - nocc) < fabs(2.0 * tr - fr - nocc);
            tr = fr = 0.0;
#pragma unroll
            for (int q = 0; q < MU; ++q) {
                if (w + q * WV >= Sm<NP>::TU) break;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int i = 16 * ti[q] + g + 4 * v, j = 16 * tj[q] + c;
                    const double nw = square ? p2[q][v] : 2.0 * P[i + LD * j] - p2[q][v];
                    Pn[i + LD * j] = nw;
                    if (ti[q] != tj[q]) Pn[j + LD * i] = nw;
                    fr += (ti[q] != tj[q] ? 2.0 : 1.0) * nw * nw;
                    if (i == j) tr += nw;
                }
            }
            double *x = const_cast<double *>(P);
            P = Pn;
            Pn = x;
        }
        if (ok && P != sA) {   // (uniform) into sA, where the rest expects it
            __syncthreads();
            for (int e = t; e < NP * LD; e += TH) sA[e] = sB[e];
        }
        __syncthreads();
    }
    if (t == 0) {
        a.out[SO_OK] = ok;
        a.out[SO_STEPS] = steps;
    }
    if (!ok) return;   // (uniform) the host takes the eigenvectors of Fx
    // the projector, and D = 2 X P X
    for (int e = t; e < nn; e += TH) a.Don[e] = sA[e % n + LD * (e / n)];
    load<NP>(sB, a.X, n);
    __syncthreads();
    product<NP>(sB, sA, acc);   // X P
    __syncthreads();
    to_lds<NP>(sA, acc);
    __syncthreads();
    product<NP>(sA, sB, acc);
    each<NP>(acc, [&](int i, int j, double v) {
        if (i < n && j < n) a.Dnext[i + n * j] = 2.0 * v;
    });
}

// X = S^-1/2 and Xi = S^1/2 by the coupled Newton-Schulz iteration of
// inv_sqrt_ns (scf.hip): A = S / c, T = (3 I - Z Y) / 2, Y <- Y T, Z <- T Z; Y and Z
// in memory, T and one of them in LDS.  The iteration is stable only with
// the products as they stand: although Y, Z and T are symmetric up to
// rounding, reading a right operand by rows (its transpose), or mirroring a
// product's upper half, diverges from condition numbers of 1e3 on.  The
// right operand is read down its columns, and the leading dimension is odd,
// which leaves a two-way bank conflict.
template <int NP>
__global__ __launch_bounds__(Sm<NP>::THREADS) void k_small_inv_sqrt(int n, const double *__restrict__ S, double *X,
                                                                    double *Xi, double *Y, double *Z, double *out) {
    constexpr int LD = NP + 1, MT = Sm<NP>::MT, TH = Sm<NP>::THREADS;
    __shared__ double sA[NP * LD], sB[NP * LD], s_red[Sm<NP>::WAVES];
    const int t = threadIdx.x, nn = n * n, w = t >> 6, lane = t & 63, g = lane >> 4, cc = lane & 15;
    auto fill = [&](double *M, const double *A) {
        for (int e = t; e < NP * NP; e += TH) {
            const int i = e % NP, j = e / NP;
            M[i + LD * j] = (i < n && j < n) ? A[i + n * j] : 0.0;
        }
    };
    d4_t acc[MT];
    auto mul = [&](const double *A, const double *B) {
#pragma unroll
        for (int q = 0; q < MT; ++q) {
            const int tile = w + q * Sm<NP>::WAVES;
            if (tile >= Sm<NP>::T2) break;
            const double *pa = A + 16 * (tile % Sm<NP>::NT) + cc + LD * g;
            const double *pb = B + LD * (16 * (tile / Sm<NP>::NT) + cc) + g;
            acc[q] = (d4_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int k = 0; k < NP; k += 4) acc[q] = mfma64(pa[LD * k], pb[k], acc[q]);
        }
    };
    // Gershgorin's upper bound
    double c = -1e300;
    for (int i = t; i < n; i += TH) {
        double r = S[i * (n + 1)];
        for (int j = 0; j < n; ++j)
            if (j != i) r += fabs(S[j + n * i]);
        c = fmax(c, r);
    }
    c = wg_largest<NP>(c, s_red);
    if (!(c > 0.0)) {
        if (t == 0) out[0] = 0.0;
        return;
    }
    for (int e = t; e < nn; e += TH) {
        Y[e] = S[e] / c;
        Z[e] = e % n == e / n ? 1.0 : 0.0;
    }
    __syncthreads();
    int extra = -1, done = 0;
    for (int k = 0; k < 40; ++k) {
        fill(sA, Z);
        fill(sB, Y);
        __syncthreads();
        mul(sA, sB);   // Z Y
        double far = 0.0;
        each<NP>(acc, [&](int i, int j, double v) {
            if (i >= n || j >= n) return;
            const double d = fabs(v - (i == j ? 1.0 : 0.0));
            far = fmax(far, d < 1e300 ? d : 1e300);   // (not a number counts as far)
        });
        far = wg_largest<NP>(far, s_red);   // (its barriers also end the reads of sA)
        if (extra == 0) {
            done = 1;
            break;
        }
        // quadratic convergence: one more step takes 1e-9 below round-off
        if (extra < 0 && far < 1e-9) extra = 1;
        each<NP>(acc, [&](int i, int j, double v) {
            sA[i + LD * j] = (i < n && j < n) ? (i == j ? 1.5 : 0.0) - 0.5 * v : 0.0;
        });
        __syncthreads();
        mul(sB, sA);   // Y T
        __syncthreads();
        each<NP>(acc, [&](int i, int j, double v) {
            if (i < n && j < n) Y[i + n * j] = v;
        });
        fill(sB, Z);
        __syncthreads();
        mul(sA, sB);   // T Z
        __syncthreads();
        each<NP>(acc, [&](int i, int j, double v) {
            if (i < n && j < n) Z[i + n * j] = v;
        });
        __syncthreads();
        if (extra > 0) --extra;
    }
    const double rc = sqrt(c);
    for (int e = t; e < nn; e += TH) {
        X[e] = Z[e] / rc;
        Xi[e] = Y[e] * rc;
    }
    if (t == 0) out[0] = done;
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
    load<NP>(sA, Fo, n);
    for (int e = t; e < NP * NP; e += TH) sU[e % NP + LD * (e / NP)] = e % NP == e / NP ? 1.0 : 0.0;
    __syncthreads();
    for (int sweep = 0; sweep < 40; ++sweep) {
        double off = 0.0, dia = 0.0;
        for (int e = t; e < NP * NP; e += TH) {
            const double v = sA[e % NP + LD * (e / NP)];
            if (e % NP == e / NP) dia += v * v;
            else off += v * v;
        }
        off = wg_total<NP>(off, s_red);
        dia = wg_total<NP>(dia, s_red);
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
        for (int j = 0; j < n; ++j) {
            const double u = sA[j * (LD + 1)];
            at += u < v || (u == v && j < t);
        }
        s_at[t] = at;
        eig[at] = v;
    }
    __syncthreads();
    // C = X U, columns to their places
    load<NP>(sA, X, n);
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
