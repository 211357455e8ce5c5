// small_dense.h -- dense algebra of matrices up to about a hundred rows, held in
// the LDS of one workgroup: products on the FP64 matrix cores, reductions, the
// DIIS system and the purification of a density.
#pragma once

#include <hip/hip_runtime.h>

#include "wave.h"

namespace myqc {

typedef double d4_t __attribute__((ext_vector_type(4)));

// n x n matrices in LDS as NP x NP (NP a multiple of 16) with leading dimension
// LD, worked by WV wavefronts
template <int NP_, int WV_>
struct DenseLds {
    static constexpr int NP = NP_, WAVES = WV_, THREADS = 64 * WV_;
    static constexpr int LD = NP % 32 == 16 ? NP : NP == 96 ? NP + 1 : NP + 16;
    static constexpr int NT = NP / 16, T2 = NT * NT, TU = NT * (NT + 1) / 2;
    static constexpr int MT = (T2 + WAVES - 1) / WAVES, MU = (TU + WAVES - 1) / WAVES;
};

__device__ __forceinline__ d4_t mfma64(double a, double b, d4_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// The thread's index, opaque to the compiler: what is computed from it stays
// inside the loop it stands in.  A long loop of many phases otherwise carries
// every phase's addresses across all of them, in registers that spill.
__device__ __forceinline__ int thread_index() {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

// tile (ti, tj) of A B, B symmetric
template <class C>
__device__ __forceinline__ d4_t tile_sym(const double *A, const double *B, int ti, int tj, int lane) {
    constexpr int LD = C::LD;
    const int g = lane >> 4, c = lane & 15;
    const double *pa = A + 16 * ti + c + LD * g, *pb = B + 16 * tj + c + LD * g;
    d4_t acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < C::NP; k += 4) acc = mfma64(pa[LD * k], pb[LD * k], acc);
    return acc;
}

// the wavefront's tiles w, w + WAVES, ... of A B (B symmetric)
template <class C>
__device__ __forceinline__ void product(const double *A, const double *B, d4_t (&acc)[C::MT]) {
    const int t = thread_index(), w = t >> 6;
#pragma unroll
    for (int q = 0; q < C::MT; ++q) {
        const int tile = w + q * C::WAVES;
        if (tile < C::T2) acc[q] = tile_sym<C>(A, B, tile % C::NT, tile / C::NT, t & 63);
    }
}

// f(row, column, value) over the wavefront's tiles
template <class C, typename F>
__device__ __forceinline__ void each(const d4_t (&acc)[C::MT], F f) {
    const int t = thread_index(), w = t >> 6, lane = t & 63, g = lane >> 4, c = lane & 15;
#pragma unroll
    for (int q = 0; q < C::MT; ++q) {
        const int tile = w + q * C::WAVES;
        if (tile >= C::T2) break;
#pragma unroll
        for (int v = 0; v < 4; ++v)
            f(16 * (tile % C::NT) + g + 4 * v, 16 * (tile / C::NT) + c, acc[q][v]);
    }
}

template <class C>
__device__ __forceinline__ void to_lds(double *M, const d4_t (&acc)[C::MT]) {
    each<C>(acc, [&](int i, int j, double v) { M[i + C::LD * j] = v; });
}

// M = scale times the n x n A, zero beyond
template <class C>
__device__ __forceinline__ void load(double *M, const double *__restrict__ A, int n, double scale = 1.0) {
    for (int e = thread_index(); e < C::NP * C::NP; e += C::THREADS) {
        const int i = e % C::NP, j = e / C::NP;
        M[i + C::LD * j] = (i < n && j < n) ? scale * A[i + n * j] : 0.0;
    }
}

// sum (or maximum) over the workgroup of a value per thread; s: a double per wavefront
template <class C>
__device__ __forceinline__ double wg_total(double v, double *s) {
    const int t = thread_index();
    v = wave_total(v);
    __syncthreads();
    if ((t & 63) == 0) s[t >> 6] = v;
    __syncthreads();
    return wave_total((t & 63) < C::WAVES ? s[t & 63] : 0.0);
}
// sum over each aligned 16 lanes
__device__ __forceinline__ double row_total(double v) {
    v = dpp_add<0xB1>(v);
    v = dpp_add<0x4E>(v);
    v = dpp_add<0x141>(v);
    return dpp_add<0x140>(v);
}
template <int CTRL>
__device__ __forceinline__ double dpp_largest(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = dpp_i<CTRL>((int)b), hi = dpp_i<CTRL>((int)(b >> 32));
    return fmax(v, __longlong_as_double(((long long)hi << 32) | (unsigned)lo));
}
// largest of each aligned 16 lanes, and of the wavefront (every lane active)
__device__ __forceinline__ double row_largest(double v) {
    v = dpp_largest<0xB1>(v);
    v = dpp_largest<0x4E>(v);
    v = dpp_largest<0x141>(v);
    return dpp_largest<0x140>(v);
}
__device__ __forceinline__ double wave_largest(double v) {
    v = row_largest(v);
    return fmax(fmax(lane_value(v, 0), lane_value(v, 16)), fmax(lane_value(v, 32), lane_value(v, 48)));
}
template <class C>
__device__ __forceinline__ double wg_largest(double v, double *s) {
    const int t = thread_index();
    v = wave_largest(v);
    __syncthreads();
    if ((t & 63) == 0) s[t >> 6] = v;
    __syncthreads();
    return wave_largest(s[(t & 63) % C::WAVES]);
}

// Gershgorin bounds of the symmetric matrix in M
template <class C>
__device__ __forceinline__ void bounds(const double *M, int n, double *s, double &lo, double &hi) {
    // a wavefront per row
    const int t = thread_index(), lane = t & 63;
    double l = 1e300, h = -1e300;
    for (int i = t >> 6; i < n; i += C::WAVES) {
        double r = 0.0;
        for (int j = lane; j < n; j += 64)
            if (j != i) r += fabs(M[j + C::LD * i]);
        r = wave_total(r);
        const double c = M[i * (C::LD + 1)];
        l = fmin(l, c - r);
        h = fmax(h, c + r);
    }
    lo = -wg_largest<C>(-l, s);
    hi = wg_largest<C>(h, s);
}

// DIIS coefficients c_0 .. c_{m-1} of the (m + 1) system, Gauss-Jordan with
// column pivoting, by the first wavefront: lane r holds row r in registers.
// Zeros with c[head] = 1 when the system is singular or m < 2.
__device__ __forceinline__ bool diis_wave(const double *B, int m, int head, double *s_c) {
    constexpr int MD = 8, W = MD + 2;
    const int r = thread_index() & 63, N = m + 1;
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
        const double best = lane_value(row_largest(v), 0);   // (rows are lanes 0 .. 8 of the first 16)
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

// The projector onto the nocc lowest levels (0 < nocc < n) of the symmetric
// matrix in sA, into sA, by trace-correcting purification (as in sp2.hip); false
// if it is not idempotent within max_steps (then sA is lost).  sB: the other
// matrix; s_red: WAVES, s_part: 16 WAVES doubles.
template <class C>
__device__ __forceinline__ bool purify(double *sA, double *sB, int n, double nocc, int max_steps, double *s_red,
                                       double *s_part, int &steps) {
    constexpr int LD = C::LD, MU = C::MU, TH = C::THREADS, WV = C::WAVES;
    const int t = thread_index(), lane = t & 63, w = t >> 6;
    double lo, hi;
    bounds<C>(sA, n, s_red, lo, hi);
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
    for (int e = t; e < C::NP * C::NP; e += TH) {
        const int i = e % C::NP, j = e / C::NP;
        double v = 0.0;
        if (i < n && j < n) {
            v = ((i == j ? hi : 0.0) - sA[i + LD * j]) * sc;
            fr += v * v;
            if (i == j) tr += v;
        }
        sB[i + LD * j] = v;
    }
    int cs = -1;
    bool ok = false;
    // P_k and P_{k+1} take turns in the two arrays: one barrier per step
    const double *P = sB;
    double *Pn = sA;
    for (int step = 0; step <= max_steps; ++step) {
        double *part = s_part + (step & 1) * 8 * WV;
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
            if (w + q * WV < C::TU) p2[q] = tile_sym<C>(P, P, ti[q], tj[q], lane);
        tr = wave_total(pt);
        fr = wave_total(pf);
        if (cs < 0 && step >= 8 && fabs(tr - fr) < 1e-8 && fabs(tr - nocc) < 1e-6) cs = step;
        if (cs >= 0 && step >= cs + 2) {
            ok = true;
            steps = step;
            break;
        }
        if (step == max_steps) break;
        const bool square = fabs(fr - nocc) < fabs(2.0 * tr - fr - nocc);
        tr = fr = 0.0;
#pragma unroll
        for (int q = 0; q < MU; ++q) {
            if (w + q * WV >= C::TU) break;
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
        for (int e = t; e < C::NP * LD; e += TH) sA[e] = sB[e];
    }
    __syncthreads();
    return ok;
}

// X = S^-1/2 and Xi = S^1/2 by the coupled Newton-Schulz iteration of
// inv_sqrt_ns (scf.hip): A = S / c, T = (3 I - Z Y) / 2, Y <- Y T, Z <- T Z; Y and Z
// in memory, T and one of them in LDS.  The iteration is stable only with
// the products as they stand: although Y, Z and T are symmetric up to
// rounding, reading a right operand by rows (its transpose), or mirroring a
// product's upper half, diverges from condition numbers of 1e3 on.  The
// right operand is read down its columns, and the leading dimension is odd,
// which leaves a two-way bank conflict.  False without
// convergence in max_steps (a step takes an eigenvalue of A at most 9/4 closer
// to one: k steps reach condition numbers of about 2.25^k).  sM: 2 NP (NP + 1), s_red: WAVES doubles.
template <class C>
__device__ __forceinline__ bool inv_sqrt_ns(int n, const double *__restrict__ S, double *X, double *Xi, double *Y,
                                            double *Z, double *sM, double *s_red, int max_steps) {
    constexpr int NP = C::NP, LD = NP + 1, MT = C::MT, TH = C::THREADS;
    double *sA = sM, *sB = sM + NP * LD;
    const int t = thread_index(), nn = n * n, w = t >> 6, lane = t & 63, g = lane >> 4, cc = lane & 15;
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
            const int tile = w + q * C::WAVES;
            if (tile >= C::T2) break;
            const double *pa = A + 16 * (tile % C::NT) + cc + LD * g;
            const double *pb = B + LD * (16 * (tile / C::NT) + cc) + g;
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
    c = wg_largest<C>(c, s_red);
    if (!(c > 0.0)) return false;
    for (int e = t; e < nn; e += TH) {
        Y[e] = S[e] / c;
        Z[e] = e % n == e / n ? 1.0 : 0.0;
    }
    __syncthreads();
    int extra = -1;
    bool done = false;
    for (int k = 0; k < max_steps; ++k) {
        fill(sA, Z);
        fill(sB, Y);
        __syncthreads();
        mul(sA, sB);   // Z Y
        double far = 0.0;
        each<C>(acc, [&](int i, int j, double v) {
            if (i >= n || j >= n) return;
            const double d = fabs(v - (i == j ? 1.0 : 0.0));
            far = fmax(far, d < 1e300 ? d : 1e300);   // (not a number counts as far)
        });
        far = wg_largest<C>(far, s_red);   // (its barriers also end the reads of sA)
        if (extra == 0) {
            done = true;
            break;
        }
        // quadratic convergence: one more step takes 1e-9 below round-off
        if (extra < 0 && far < 1e-9) extra = 1;
        each<C>(acc, [&](int i, int j, double v) {
            sA[i + LD * j] = (i < n && j < n) ? (i == j ? 1.5 : 0.0) - 0.5 * v : 0.0;
        });
        __syncthreads();
        mul(sB, sA);   // Y T
        __syncthreads();
        each<C>(acc, [&](int i, int j, double v) {
            if (i < n && j < n) Y[i + n * j] = v;
        });
        fill(sB, Z);
        __syncthreads();
        mul(sA, sB);   // T Z
        __syncthreads();
        each<C>(acc, [&](int i, int j, double v) {
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
    __syncthreads();
    return done;
}

}  // namespace myqc
