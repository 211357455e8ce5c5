// mfma_f64.hip -- the FP64 quarter transforms of ao2mo on gfx950 matrix
// cores (v_mfma_f64_16x16x4f64), replacing library GEMMs.
//
// The four quarter steps of slow_ao2mo_MP2_RHF (idx1..idx4_trans,
// src/ao2mo/ao2mo.f90:1306-1439), with orbital blocks Cp, Cq, Cr, Cs:
//   1+2  M(p,q,l,d) = sum_v [sum_u Cp(u,p) XX(u,v,l,d)] Cq(v,q)   (k_ao2mo12_f64)
//   3    N(pq,r,d)  = sum_l M(pq,l,d) Cr(l,r)                      (k_gemm_f64)
//   4    O(pq,r,s)  = sum_d N(pq,r,d) Cs(d,s)                      (k_gemm_f64)
//
// MFMA lane layout (16x16x4, checked by the GPU layout test): lane l = 16 g +
// c feeds A[c][g] of the 16x4 A and B[g][c] of the 4x16 B, and receives
// D[g + 4 v][c], v = 0..3.  Both kernels compute transposed products so that
// every store is 16 consecutive doubles, and in steps 1+2 the accumulator of
// the first product is already the B operand of the second: with
// L^T(v, p) = sum_u X^T(v, u) Cp(u, p) held as D tiles, element v of a lane's
// accumulator is L^T(v0 + 4 kb + g, p0 + c) for kb = v, which is exactly the
// B fragment of k-step kb of M^T(q, p) = sum_v Cq^T(q, v) L^T(v, p).  The o n^3
// intermediate L never leaves the registers.
#include <cstdint>

#include "dense.h"
#include "many.h"

namespace myqc {

typedef double d4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ d4_t mfma16x16x4(double a, double b, d4_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// ---------------------------------------------------------------------------
// Quarter steps 1 and 2, fused.
//
// Workgroup: 8 wavefronts, wavefront w owning the 16 orbitals p of tile
// p0 = 128 blockIdx.y + 16 w, and the 16 NAT orbitals q from 16 NAT blockIdx.z.
// Its B fragments of Cp (k-steps of u) stay in registers for the whole launch.
// The workgroup walks (l,d) blocks blockIdx.x, + gridDim.x, ... and, within
// each, v tiles of 16 columns: the tile X(:, v0..v0+15 | l,d) is 16 n
// contiguous doubles, copied into LDS (double-buffered, the next tile's loads
// in flight during this tile's MFMAs) and shared by the 8 wavefronts.  Per v
// tile a wavefront runs NKS MFMAs of step 1 (four accumulators in turn) and
// 4 NAT of step 2; after the last v tile of an (l,d) block it stores M^T and
// clears the accumulators.  Bound by the matrix cores, busy 70 % of the time:
// 24 waters, 14196 blocks, 2.53 ms, 49 TFLOP/s.  (3.04 ms with the next tile's
// loads under branches, for which the compiler waited before the first MFMA,
// and NKS in steps of 8 to 20: n = 168 ran 48 of its 42 k-steps.)
// ---------------------------------------------------------------------------
constexpr int Q12_WAVES = 8, Q12_THREADS = 64 * Q12_WAVES, Q12_NAT = 3;

template <int NKS>
__global__ __launch_bounds__(Q12_THREADS) void k_ao2mo12_f64(int np, int nq, int n, const double *__restrict__ Cp,
                                                             const double *__restrict__ Cq,
                                                             const double *__restrict__ XX, double *__restrict__ M,
                                                             int nld, const int *__restrict__ tri) {
    constexpr int LDX = 4 * NKS + 2;                           // padded column of a tile in LDS
    constexpr int XPT = (16 * 4 * NKS + Q12_THREADS - 1) / Q12_THREADS;   // tile doubles per thread
    __shared__ double sX[2][16 * LDX];
    // Cq^T of this block of q, [q][v], in LDS when it fits beside the X tiles
    constexpr bool QLDS = NKS <= 48;
    __shared__ double sQ[QLDS ? 16 * Q12_NAT * LDX : 1];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, g = lane >> 4, c = lane & 15;
    const int p0 = blockIdx.y * (16 * Q12_WAVES) + 16 * w;
    const int q0 = blockIdx.z * (16 * Q12_NAT);
    const size_t nn = (size_t)n * n;
    const int nvt = (n + 15) >> 4;
    // rows u >= n of both buffers stay zero (Cp's fragments are zero there too)
    for (int e = t; e < 2 * 16 * LDX; e += Q12_THREADS) (&sX[0][0])[e] = 0.0;
    if constexpr (QLDS)
        for (int e = t; e < 16 * Q12_NAT * LDX; e += Q12_THREADS) {
            const int ql = e / LDX, v = e - ql * LDX, q = q0 + ql;
            sQ[e] = (v < n && q < nq) ? Cq[v + (size_t)n * q] : 0.0;
        }
    // Cp fragments: B[g][c] of k-step k = Cp(4 k + g, p0 + c)
    double cf[NKS];
#pragma unroll
    for (int k = 0; k < NKS; ++k) {
        const int u = 4 * k + g;
        cf[k] = (u < n && p0 + c < np) ? Cp[u + (size_t)n * (p0 + c)] : 0.0;
    }
    // the work items of this workgroup: (ld, vt) for ld = blockIdx.x + j gridDim.x,
    // walked with counters (no divisions in the loop, nor in the copy to LDS:
    // the places of a thread's elements are the same for every tile)
    int lofs[XPT];
#pragma unroll
    for (int r = 0; r < XPT; ++r) {
        const int e = t + r * Q12_THREADS, col = e / n;
        lofs[r] = e < 16 * n ? col * LDX + (e - col * n) : -1;
    }
    double xr[XPT];
    auto load_tile = [&](int ld, int vt) {
        const double *src = XX + (size_t)ld * nn + (size_t)(16 * vt) * n;
        const int last = min(16, n - 16 * vt) * n - 1;   // of the tile's doubles inside the block
#pragma unroll
        for (int r = 0; r < XPT; ++r) xr[r] = src[min(t + r * Q12_THREADS, last)];
    };
    auto store_tile = [&](int buf, int vt) {
        const int valid = min(16, n - 16 * vt) * n;
#pragma unroll
        for (int r = 0; r < XPT; ++r)
            if (lofs[r] >= 0) sX[buf][lofs[r]] = t + r * Q12_THREADS < valid ? xr[r] : 0.0;
    };
    d4_t macc[Q12_NAT];
#pragma unroll
    for (int s = 0; s < Q12_NAT; ++s) macc[s] = (d4_t){0.0, 0.0, 0.0, 0.0};
    int ld = blockIdx.x, vt = 0;
    load_tile(min(ld, nld - 1), 0);
    __syncthreads();   // the zero fill is complete before the first tile lands
    store_tile(0, 0);
    __syncthreads();
    int cur = 0;
    while (ld < nld) {
        int ld1 = ld, vt1 = vt + 1;
        if (vt1 == nvt) {
            vt1 = 0;
            ld1 += gridDim.x;
        }
        // the next tile's loads, issued on every path (this tile's again when
        // there is no next) and without a branch, so that the wait the
        // compiler places for them is the one before their copy to LDS
        const bool more = ld1 < nld;
        load_tile(more ? ld1 : ld, more ? vt1 : vt);
        const int v0 = vt * 16;
        // step 1: L^T(v0 + ., p0 + .) over all u, four independent chains
        const double *xs = &sX[cur][c * LDX + g];
        d4_t ac[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) ac[k] = (d4_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < NKS; ++k) ac[k & 3] = mfma16x16x4(xs[4 * k], cf[k], ac[k & 3]);
        const d4_t lt = (ac[0] + ac[1]) + (ac[2] + ac[3]);
        // step 2: M^T(q, p) += sum_v Cq^T(q, v) L^T(v, p) over this tile's v
#pragma unroll
        for (int s = 0; s < Q12_NAT; ++s) {
            if constexpr (QLDS) {
                const double *qs = &sQ[(16 * s + c) * LDX + v0 + g];
#pragma unroll
                for (int kb = 0; kb < 4; ++kb) macc[s] = mfma16x16x4(qs[4 * kb], lt[kb], macc[s]);
            } else {
                const int q = q0 + 16 * s + c;
#pragma unroll
                for (int kb = 0; kb < 4; ++kb) {
                    const int v = v0 + 4 * kb + g;
                    const double qa = (v < n && q < nq) ? Cq[v + (size_t)n * q] : 0.0;
                    macc[s] = mfma16x16x4(qa, lt[kb], macc[s]);
                }
            }
        }
        if (vt == nvt - 1) {
            // M(p, q, l, d) at p + np (q + nq tri(l, d))
            const long long out = tri[ld];
#pragma unroll
            for (int s = 0; s < Q12_NAT; ++s) {
#pragma unroll
                for (int vv = 0; vv < 4; ++vv) {
                    const int q = q0 + 16 * s + g + 4 * vv, p = p0 + c;
                    if (p < np && q < nq) M[p + (size_t)np * (q + (size_t)nq * out)] = macc[s][vv];
                }
                macc[s] = (d4_t){0.0, 0.0, 0.0, 0.0};
            }
        }
        if (more) store_tile(cur ^ 1, vt1);
        __syncthreads();
        cur ^= 1;
        ld = ld1;
        vt = vt1;
    }
}

// ---------------------------------------------------------------------------
// Steps 3 and 4: C (m x nb, ldc) = A (m x k, lda) B (k x nb, ldb) for `batch`
// problems (A += bat sA, C += bat sC; B shared), all column-major FP64; with
// tri, column kk of problem bat's A is block (kk, bat) of a triangular array
// (A + lda (max (max + 1) / 2 + min)).
// A workgroup of 4 wavefronts owns 128 rows of one problem (blockIdx.x) and
// 16 NT columns (blockIdx.y), NT chosen so that the columns are covered with
// the fewest tiles (all of them up to 128: A, the large operand, is then read
// once); each wavefront 32 rows x NT column tiles, as C^T = B^T A^T so that
// lanes store 16 consecutive rows.  k goes through LDS in slices of 16,
// double-buffered, the next slice's loads in flight during this slice's
// 8 NT MFMAs.  LDS: A as [k][row], rows of 144 doubles (the two k's of a
// half-wavefront's read fall in distinct banks), B as [column][k], columns of
// 18 (its 16 columns likewise).
// Bound by the matrix cores at about half their rate, the rest the issue of
// loads and LDS traffic in between: 24 waters, step 3 (5760 x 168 x 120, 168
// problems) 0.98 ms, 40 TFLOP/s, and step 4 0.31 ms; with 16 rows per
// wavefront 1.28 and 0.34, and slices of 8 1.49; with fragments loaded
// straight from memory one k-step ahead and 48 columns per workgroup (A read
// three times) 1.56 and 0.41.
// ---------------------------------------------------------------------------
constexpr int GF_RT = 2, GF_M = 64 * GF_RT, GF_K = 16, GF_THREADS = 256, GF_NT = 8;

template <int NT>
__global__ __launch_bounds__(GF_THREADS) void k_gemm_f64(int m, int nb, int k, const double *__restrict__ A,
                                                         long long lda, long long sA, const double *__restrict__ B,
                                                         long long ldb, double *__restrict__ C, long long ldc,
                                                         long long sC, int tiles_m, int tri) {
    constexpr int LA = GF_M + 16, LB = GF_K + 2;
    __shared__ double s_a[2][GF_K * LA], s_b[2][16 * NT * LB];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, g = lane >> 4, c = lane & 15;
    const int bat = blockIdx.x / tiles_m;
    const int r0 = (int)(blockIdx.x - bat * tiles_m) * GF_M, j0 = blockIdx.y * (16 * NT);
    A += bat * sA;
    int ar[GF_RT];
#pragma unroll
    for (int x = 0; x < GF_RT; ++x) ar[x] = min(r0 + (t & 63) + 64 * x, m - 1);
    C += bat * sC;
    // the thread's share of a slice: A row t & 63 at k = (t >> 6) + 4 q;
    // B k = t & 15 of column (t >> 4) + 16 q.  Rows and columns past the end
    // repeat the last one (their results are not stored); k's past the end are
    // zero on both sides.
    const int ak = t >> 6, bk = t & 15;
    const double *pB[NT];
#pragma unroll
    for (int q = 0; q < NT; ++q) pB[q] = B + ldb * min(j0 + (t >> 4) + 16 * q, nb - 1);
    double pa[4][GF_RT], pb[NT];
    auto load = [&](int k0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int kk = min(k0 + ak + 4 * q, k - 1);
            const int hi = max(kk, bat);
            const unsigned ka = tri ? hi * (hi + 1) / 2 + min(kk, bat) : kk;
            const double *col = A + (size_t)ka * (unsigned)lda;
#pragma unroll
            for (int x = 0; x < GF_RT; ++x) {
                const double v = col[ar[x]];
                pa[q][x] = k0 + ak + 4 * q < k ? v : 0.0;
            }
        }
        const int kk = min(k0 + bk, k - 1);
#pragma unroll
        for (int q = 0; q < NT; ++q) {
            const double x = pB[q][kk];
            pb[q] = k0 + bk < k ? x : 0.0;
        }
    };
    d4_t acc[GF_RT][NT];
#pragma unroll
    for (int x = 0; x < GF_RT; ++x)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[x][j] = (d4_t){0.0, 0.0, 0.0, 0.0};
    load(0);
    int buf = 0;
    for (int k0 = 0; k0 < k; k0 += GF_K, buf ^= 1) {
#pragma unroll
        for (int q = 0; q < 4; ++q) 
#pragma unroll
            for (int x = 0; x < GF_RT; ++x) s_a[buf][((t >> 6) + 4 * q) * LA + (t & 63) + 64 * x] = pa[q][x];
#pragma unroll
        for (int q = 0; q < NT; ++q) s_b[buf][((t >> 4) + 16 * q) * LB + bk] = pb[q];
        __syncthreads();
        if (k0 + GF_K < k) load(k0 + GF_K);
#pragma unroll
        for (int ks = 0; ks < GF_K; ks += 4) {
            double fa[GF_RT];
#pragma unroll
            for (int x = 0; x < GF_RT; ++x) fa[x] = s_a[buf][(ks + g) * LA + 16 * (GF_RT * w + x) + c];
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const double fb = s_b[buf][(16 * j + c) * LB + ks + g];
#pragma unroll
                for (int x = 0; x < GF_RT; ++x) acc[x][j] = mfma16x16x4(fb, fa[x], acc[x][j]);
            }
        }
    }
#pragma unroll
    for (int x = 0; x < GF_RT; ++x) {
        const int r = r0 + 16 * (GF_RT * w + x) + c;
        if (r >= m) continue;
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int vv = 0; vv < 4; ++vv) {
                const int col = j0 + 16 * j + g + 4 * vv;
                if (col < nb) C[r + ldc * col] = acc[x][j][vv];
            }
    }
}

template <int NKS>
static void launch12(dim3 grid, hipStream_t s, const TransformJob &j, int n, const double *XX, int nld,
                     const int *tri) {
    k_ao2mo12_f64<NKS><<<grid, Q12_THREADS, 0, s>>>(j.np, j.nq, n, j.Cp, j.Cq, XX, j.M, nld, tri);
}

// Steps 1+2 in FP64 of one job over nblk blocks of XX (n^2 each), block b's
// result at M's block tri[b].
int ao2mo12_f64(myqc_ctx *ctx, const TransformJob &j, int n, const double *XX, int nblk, const int *tri) {
    if (j.np <= 0 || j.nq <= 0 || n <= 0 || nblk <= 0)
        return set_error(ctx, MYQC_E_ARG, "ao2mo12_f64: np=%d nq=%d n=%d blocks=%d", j.np, j.nq, n, nblk);
    const int nks = (n + 3) / 4;
    const int gy = (j.np + 16 * Q12_WAVES - 1) / (16 * Q12_WAVES), gz = (j.nq + 16 * Q12_NAT - 1) / (16 * Q12_NAT);
    if (gy > 65535 || gz > 65535) return set_error(ctx, MYQC_E_ARG, "ao2mo12_f64: too many orbitals");
    // one workgroup per CU and orbital block (256 CUs), each walking its (l,d) blocks
    const int gx = (int)std::min<long long>(nblk, std::max(1LL, 256LL / ((long long)gy * gz)));
    const dim3 grid((unsigned)gx, (unsigned)gy, (unsigned)gz);
    hipStream_t s = ctx->stream;
    if (nks <= 4) launch12<4>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 8) launch12<8>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 12) launch12<12>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 16) launch12<16>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 20) launch12<20>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 24) launch12<24>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 28) launch12<28>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 32) launch12<32>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 36) launch12<36>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 40) launch12<40>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 44) launch12<44>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 48) launch12<48>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 52) launch12<52>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 56) launch12<56>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 60) launch12<60>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 64) launch12<64>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 72) launch12<72>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 80) launch12<80>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 90) launch12<90>(grid, s, j, n, XX, nblk, tri);
    else if (nks <= 100) launch12<100>(grid, s, j, n, XX, nblk, tri);
    else return set_error(ctx, MYQC_E_ARG, "ao2mo12_f64: n=%d above 400", n);
    MYQC_HIP(ctx, hipGetLastError());
    return 0;
}

// C = A B (FP64), `batch` problems of A (m x k, lda, stride sA, or with tri
// column kk of problem d at block (kk, d) of a triangular array) against the
// shared B (k x nb, ldb), into C (m x nb, ldc, stride sC).
int gemm_f64(myqc_ctx *ctx, int m, int nb, int k, const double *A, long long lda, long long sA, const double *B,
             long long ldb, double *C, long long ldc, long long sC, int batch, bool tri) {
    if (m <= 0 || nb <= 0 || k <= 0 || batch <= 0) return set_error(ctx, MYQC_E_ARG, "gemm_f64: empty problem");
    const long long tiles_m = ((long long)m + GF_M - 1) / GF_M;
    const long long gx = tiles_m * batch;
    if (lda > 0xffffffffLL) return set_error(ctx, MYQC_E_ARG, "gemm_f64: leading dimension too large");
    // column tiles, in the fewest blocks of at most GF_NT, equally filled
    const int ct = (nb + 15) / 16, gy = (ct + GF_NT - 1) / GF_NT, nt = (ct + gy - 1) / gy;
    if (gx > 0x7fffffffLL || tiles_m > 0x7fffffffLL || gy > 65535)
        return set_error(ctx, MYQC_E_ARG, "gemm_f64: grid too large");
    const dim3 grid((unsigned)gx, (unsigned)gy);
    auto run = [&](auto kern) {
        kern<<<grid, GF_THREADS, 0, ctx->stream>>>(m, nb, k, A, lda, sA, B, ldb, C, ldc, sC, (int)tiles_m, tri ? 1 : 0);
    };
    switch (nt) {
        case 1: run(k_gemm_f64<1>); break;
        case 2: run(k_gemm_f64<2>); break;
        case 3: run(k_gemm_f64<3>); break;
        case 4: run(k_gemm_f64<4>); break;
        case 5: run(k_gemm_f64<5>); break;
        case 6: run(k_gemm_f64<6>); break;
        case 7: run(k_gemm_f64<7>); break;
        default: run(k_gemm_f64<8>); break;
    }
    MYQC_HIP(ctx, hipGetLastError());
    return 0;
}

// The same product for many problems in 64 x 64 output tiles: four
// wavefronts, each a 32 x 32 quarter (2 x 2 MFMA blocks); the k range goes
// through LDS in slices of 32, double-buffered (the next slice's global loads
// in flight during the current slice's MFMAs, one barrier per slice).  A is
// read down its columns (64 rows of one column contiguous), B down its
// columns too (32 k of one column contiguous), both stored [k][row or column]
// in LDS.  Workgroup b runs on XCD b mod 8; every tile of problem z runs on
// XCD z mod 8, so that its operands stay in one L2.
constexpr int GMT = 64, GMK = 32;

__global__ __launch_bounds__(256) void k_gemm_f64_many64(int m, int nb, int k, GemmMany g, double alpha, int nz,
                                                         int tm, int tn) {
    __shared__ double sA[2][GMK][GMT + 1], sB[2][GMK][GMT + 1];
    const int tiles = tm * tn;
    const int xcd = blockIdx.x & 7, jb = blockIdx.x >> 3;
    const int z = xcd + 8 * (jb / tiles), tile = jb % tiles;
    if (z >= nz) return;   // (uniform over the workgroup)
    const int ti = tile % tm, tj = tile / tm;
    const double *A = g.A[z], *B = g.B[z];
    double *C = g.C[z];
    const int row0 = ti * GMT, col0 = tj * GMT;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, r = lane & 15, kq = lane >> 4;
    const int wr = w & 1, wc = w >> 1;
    double pa[8], pb[8];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int e = t + 256 * q;
            const int ka = k0 + (e >> 6), ia = row0 + (e & 63);      // A: 64 rows of column ka
            pa[q] = (ia < m && ka < k) ? A[ia + (size_t)m * ka] : 0.0;
            const int kb = k0 + (e & 31), jc = col0 + (e >> 5);      // B: 32 k of column jc
            pb[q] = (jc < nb && kb < k) ? B[kb + (size_t)k * jc] : 0.0;
        }
    };
    d4_t acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = (d4_t){0.0, 0.0, 0.0, 0.0};
    fetch(0);
    int buf = 0;
    for (int k0 = 0; k0 < k; k0 += GMK, buf ^= 1) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int e = t + 256 * q;
            sA[buf][e >> 6][e & 63] = pa[q];
            sB[buf][e & 31][e >> 5] = pb[q];
        }
        __syncthreads();
        if (k0 + GMK < k) fetch(k0 + GMK);
#pragma unroll
        for (int ks = 0; ks < GMK; ks += 4) {
            double fa[2], fb[2];
#pragma unroll
            for (int x = 0; x < 2; ++x) fa[x] = sA[buf][ks + kq][wr * 32 + x * 16 + r];
#pragma unroll
            for (int y = 0; y < 2; ++y) fb[y] = sB[buf][ks + kq][wc * 32 + y * 16 + r];
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) acc[x][y] = mfma16x16x4(fa[x], fb[y], acc[x][y]);
        }
    }
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = row0 + wr * 32 + x * 16 + kq + 4 * v, col = col0 + wc * 32 + y * 16 + r;
                if (row < m && col < nb) C[row + (size_t)m * col] = alpha * acc[x][y][v];
            }
}

// C_z = alpha A_z B_z for nz problems (nz <= kMany), square or not:
// A_z m x k, B_z k x nb, C_z m x nb, all with their row counts as leading
// dimensions.
int gemm_f64_many(myqc_ctx *ctx, int m, int nb, int k, const GemmMany &g, int nz, double alpha) {
    if (m <= 0 || nb <= 0 || k <= 0 || nz <= 0 || nz > kMany)
        return set_error(ctx, MYQC_E_ARG, "gemm_f64_many: m=%d nb=%d k=%d problems %d", m, nb, k, nz);
    const int tm = (m + GMT - 1) / GMT, tn = (nb + GMT - 1) / GMT;
    const long long grid = 8LL * ((nz + 7) / 8) * tm * tn;
    if (grid > 0x7fffffffLL) return set_error(ctx, MYQC_E_ARG, "gemm_f64_many: grid too large");
    k_gemm_f64_many64<<<(unsigned)grid, 256, 0, ctx->stream>>>(m, nb, k, g, alpha, nz, tm, tn);
    MYQC_HIP(ctx, hipGetLastError());
    return 0;
}

}  // namespace myqc
