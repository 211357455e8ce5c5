// batch.hip -- RHF of thousands of small molecules in one persistent launch.
//
// The reference solves one molecule per run of its programs; a batch of
// 2-8 atom molecules (2-40 functions each) is far too small per molecule to
// fill a GPU, so everything here is organised around the batch:
//
//   k_batch_one_e        eight lanes per (molecule, shell pair): S and H
//   k_batch_eri<CB,CK>   one thread per (molecule, unique shell quartet) of a
//                        pair-class combination: the same OS/HGP code and
//                        reference numerics as the single-molecule path,
//                        written into the molecule's packed 8-fold-unique
//                        array (ij|kl), i>=j, k>=l, ij>=kl, halved where i = j
//                        and where ij = kl
//   k_batch_scf          persistent: each workgroup takes molecules from an
//                        atomic queue (largest first) and runs the whole SCF
//                        on-chip -- G(D) from the packed integrals streamed
//                        from HBM, products on the FP64 matrix cores, DIIS,
//                        Newton-Schulz for S^-1/2 and purification for the
//                        density (cyclic Jacobi where either does not
//                        converge) -- with no host round trip
//
// The launch shapes (threads per ERI and SCF workgroup) are chosen by timing
// the candidates on the batch itself (batch_tune), and the whole sequence is
// captured once into a hipGraph that later calls replay.
#include <algorithm>
#include <cmath>
#include <numeric>
#include <string>
#include <vector>

#include "batch_find.h"
#include "boys_dev.h"
#include "context.h"
#include "guess.h"
#include "ket_soa.h"
#include "one_e_math.h"
#include "small_dense.h"

namespace myqc {

constexpr int kBatchDiis = 8;
constexpr int kBatchMaxN = 40;

struct BMol {
    int n, nocc, nnuc, atom0;
    int cls0[3], ncls[3];    // pairs of class c: cls_ids[c][cls0[c] .. cls0[c] + ncls[c])
    long long eri0;          // packed (ij|kl) offset
    long long mat0;          // n x n blocks: offset (sum of n^2 before)
    double e_nuc;
};

template <int C> struct BPL;
template <> struct BPL<0> { static constexpr int a = 0, b = 0; };
template <> struct BPL<1> { static constexpr int a = 1, b = 0; };
template <> struct BPL<2> { static constexpr int a = 1, b = 1; };

__host__ __device__ __forceinline__ long long tri(long long a) { return a * (a + 1) / 2; }

// ---------------------------------------------------------------------------
// one-electron integrals
// ---------------------------------------------------------------------------
// kOneELanes lanes per shell pair share its nuclei and primitive pairs; the
// pairs go class by class (the lists ids, the largest work first), so that a
// wavefront's lanes run the same code, and a workgroup goes on to further pairs
// with the tables it staged.  A lane per pair, 128 in a workgroup, in the
// molecules' order took 0.53 ms for 1024 clusters of 2 to 5 waters, lanes of
// eight in that order 0.42, by class 0.21.
constexpr int kOneELanes = 8, kOneEBlocks = 1024;
__global__ __launch_bounds__(256) void k_batch_one_e(const ShellPair *__restrict__ pairs,
                                                     const PrimPair *__restrict__ prims, const double *__restrict__ ftT,
                                                     const double *__restrict__ atoms, const int *__restrict__ pair_mol,
                                                     const BMol *__restrict__ mols, const int *__restrict__ ids0,
                                                     const int *__restrict__ ids1, const int *__restrict__ ids2, int n0,
                                                     int n1, int n2, double *__restrict__ S, double *__restrict__ H) {
    __shared__ __attribute__((aligned(16))) double s_ft[ft_staged(2)];
    const BoysTab ft = stage_boys<2>(ftT, s_ft);
    const int sub = threadIdx.x % kOneELanes, per = blockDim.x / kOneELanes;
    for (int t = blockIdx.x * per + threadIdx.x / kOneELanes; t < n0 + n1 + n2; t += gridDim.x * per) {
        const int pair = t < n2 ? ids2[t] : t < n2 + n1 ? ids1[t - n2] : ids0[t - n2 - n1];
        const ShellPair sp = pairs[pair];
        const BMol mol = mols[pair_mol[pair]];
        double s[3][3], h[3][3];
        one_e_pair(sp, prims, ft, atoms + 4 * mol.atom0, mol.nnuc, s, h, sub, kOneELanes);
        const int na = sp.la ? 3 : 1, nb = sp.lb ? 3 : 1;
        const long long n = mol.n;
        double *Sm = S + mol.mat0, *Hm = H + mol.mat0;
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int b = 0; b < 3; ++b) {
                if (a >= na || b >= nb) continue;   // (the same for a pair's lanes)
                const double ss = group_sum<kOneELanes>(s[a][b]), hs = group_sum<kOneELanes>(h[a][b]);
                if (sub != 0) continue;
                const long long i = sp.ao_a + a, j = sp.ao_b + b;
                Sm[i + n * j] = ss;
                Sm[j + n * i] = ss;
                Hm[i + n * j] = hs;
                Hm[j + n * i] = hs;
            }
    }
}
// ---------------------------------------------------------------------------
// two-electron integrals into packed per-molecule storage
// ---------------------------------------------------------------------------
struct BEriArgs {
    const ShellPair *pairs;
    const PrimPair *prims;
    const double *ftT;
    const BMol *mols;
    const int *cls0, *cls1, *cls2;
    const double *ksoa;      // primitive pairs of the ket class list (ket_soa.h)
    long long nket;          // entries of the ket class list
    const long long *qcum;   // nmol + 1 prefix counts of this class combination
    const int *qfirst;       // the molecules of quartets 0, 64, 128, ... and of the last (quartet_marks)
    long long nq;
    double *eri;
};

template <int CB, int CK>
__global__ __launch_bounds__(256) void k_batch_eri(BEriArgs a) {
    constexpr int M = CB + CK;
    __shared__ __attribute__((aligned(16))) double s_ft[ft_staged(M)];
    const BoysTab ft = stage_boys<M>(a.ftT, s_ft);
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.nq) return;
    // (a search over all molecules is ten dependent loads: 5 % of the six
    // classes' time for 1024 clusters)
    const int lo = quartet_molecule(a.qcum, a.qfirst, t);
    const BMol mol = a.mols[lo];
    const long long q = t - a.qcum[lo];
    long long p, r;
    if (CB == CK) {
        p = (long long)floor((sqrt(8.0 * (double)q + 1.0) - 1.0) * 0.5);
        while (tri(p) > q) --p;
        while (tri(p + 1) <= q) ++p;
        r = q - tri(p);
    } else {
        const int nk = mol.ncls[CK];
        p = q / nk;
        r = q - p * nk;
    }
    const int *idb = CB == 0 ? a.cls0 : CB == 1 ? a.cls1 : a.cls2;
    const int *idk = CK == 0 ? a.cls0 : CK == 1 ? a.cls1 : a.cls2;
    const ShellPair bra = a.pairs[idb[mol.cls0[CB] + p]], ket = a.pairs[idk[mol.cls0[CK] + r]];
    constexpr int LA = BPL<CB>::a, LB = BPL<CB>::b, LC = BPL<CK>::a, LD = BPL<CK>::b;
    constexpr int na = ncart(LA), nb = ncart(LB), nc = ncart(LC), nd = ncart(LD);
    QuartetAcc<LA, LB, LC, LD> acc;
    quartet_prims_f<LA, LB, LC, LD>(bra, ket, a.prims, KetSoa{a.ksoa, a.nket, mol.cls0[CK] + r}, ft, acc);
    const double CD[3] = {ket.AB[0], ket.AB[1], ket.AB[2]};
    double out[na * nb * nc * nd];
    quartet_hrr<LA, LB, LC, LD>(acc, bra.AB, CD, out);
    double *E = a.eri + mol.eri0;
#pragma unroll
    for (int ia = 0; ia < na; ++ia)
#pragma unroll
        for (int ib = 0; ib < nb; ++ib)
#pragma unroll
            for (int ic = 0; ic < nc; ++ic)
#pragma unroll
                for (int id = 0; id < nd; ++id) {
                    const int i = bra.ao_a + ia, j = bra.ao_b + ib, k = ket.ao_a + ic, l = ket.ao_b + id;
                    const long long IJ = tri(max(i, j)) + min(i, j), KL = tri(max(k, l)) + min(k, l);
                    const bool same = IJ >= KL ? i == j : k == l;
                    E[tri(max(IJ, KL)) + min(IJ, KL)] =
                        (same ? 0.5 : 1.0) * (IJ == KL ? 0.5 : 1.0) * out[((ia * nb + ib) * nc + ic) * nd + id];
                }
}

// ---------------------------------------------------------------------------
// the persistent SCF
// ---------------------------------------------------------------------------
struct BScfArgs {
    const BMol *mols;
    const int *order;          // molecules, largest first
    int nmol;
    int *counter;              // work queue head (zeroed before the launch)
    const double *eri, *S, *H, *guess;   // guess: NULL or n^2 blocks
    double *scratch;           // 4 n^2 blocks per molecule: X, the projector, F', a density
    double *hist;              // 2 kBatchDiis n^2 blocks per molecule
    double *Dout;
    double *energy;
    int *iters, *conv;
    int *fallback;             // NULL, or 1 where a learned start restarted from the core guess
    double e_tol, d_tol;
    int max_iter;
    int learned_iter;          // iterations a start from `guess` gets before the restart
    int restart;               // 1: restart an unconverged start from `guess` from the core guess
    int check_it;              // a start from `guess` whose DIIS error after check_it
    double check_err;          // iterations is above check_err restarts at once
};

// Workgroup reductions: a wavefront butterfly, then the per-wave results
// summed in a fixed order (every thread returns the same value).
__device__ __forceinline__ double wg_sum(double v, double *s_red) {
    const int t = thread_index();
    v = wave_total(v);
    __syncthreads();   // s_red free
    if ((t & 63) == 0) s_red[t >> 6] = v;
    __syncthreads();
    double r = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) r += s_red[w];
    return r;
}

__device__ __forceinline__ double wg_max(double v, double *s_red) {
    const int t = thread_index();
    v = wave_largest(v);
    __syncthreads();
    if ((t & 63) == 0) s_red[t >> 6] = v;
    __syncthreads();
    double r = -1e300;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) r = fmax(r, s_red[w]);
    return r;
}

// Cyclic Jacobi on the symmetric A (n x n, LDS): eigenvalues on A's diagonal,
// eigenvectors in the columns of U.  Rounds pair the indices round-robin so
// the n/2 rotations of a round are disjoint; each thread applies J^T A J to
// whole 2x2 blocks in place, so one barrier separates the rounds.
__device__ void jacobi(double *A, double *U, int n, double *s_rot, double *s_red) {
    const int t0 = thread_index();
    const int npad = n + (n & 1), half = npad >> 1;
    for (int e = t0; e < n * n; e += blockDim.x) U[e] = (e % n == e / n) ? 1.0 : 0.0;
    __syncthreads();
    for (int sweep = 0; sweep < 30; ++sweep) {
        double off = 0.0, dia = 0.0;
        for (int e = t0; e < n * n; e += blockDim.x) {
            const double v = A[e];
            if (e % n == e / n) dia += v * v;
            else off += v * v;
        }
        off = wg_sum(off, s_red);
        dia = wg_sum(dia, s_red);
        if (off <= 1e-28 * fmax(dia, 1e-300)) break;
        for (int r = 0; r < npad - 1; ++r) {
            // rotation of pair k: s_rot[4k] = p, [4k+1] = q, [4k+2] = c, [4k+3] = s
            for (int k = t0; k < half; k += blockDim.x) {
                const int a = k == 0 ? 0 : ((k - 1 + r) % (npad - 1)) + 1;
                const int kb = npad - 1 - k;
                const int b = ((kb - 1 + r) % (npad - 1)) + 1;
                const int p = min(a, b), q = max(a, b);
                double c = 1.0, s = 0.0;
                if (q < n) {
                    const double apq = A[p + n * q];
                    if (fabs(apq) > 1e-300) {
                        const double th = (A[q + n * q] - A[p + n * p]) / (2.0 * apq);
                        const double t = (th >= 0.0 ? 1.0 : -1.0) / (fabs(th) + sqrt(th * th + 1.0));
                        c = 1.0 / sqrt(t * t + 1.0);
                        s = t * c;
                    }
                }
                s_rot[4 * k] = p;
                s_rot[4 * k + 1] = q;
                s_rot[4 * k + 2] = c;
                s_rot[4 * k + 3] = s;
            }
            __syncthreads();
            // A <- J^T A J on 2x2 blocks (pair k1 rows, pair k2 columns)
            for (int w = t0; w < half * half; w += blockDim.x) {
                const int k1 = w % half, k2 = w / half;
                const int p1 = (int)s_rot[4 * k1], q1 = (int)s_rot[4 * k1 + 1];
                const int p2 = (int)s_rot[4 * k2], q2 = (int)s_rot[4 * k2 + 1];
                const double c1 = s_rot[4 * k1 + 2], s1 = s_rot[4 * k1 + 3];
                const double c2 = s_rot[4 * k2 + 2], s2 = s_rot[4 * k2 + 3];
                const bool q1ok = q1 < n, q2ok = q2 < n;
                const double M00 = A[p1 + n * p2];
                const double M01 = q2ok ? A[p1 + n * q2] : 0.0;
                const double M10 = q1ok ? A[q1 + n * p2] : 0.0;
                const double M11 = (q1ok && q2ok) ? A[q1 + n * q2] : 0.0;
                const double T00 = c1 * M00 - s1 * M10, T01 = c1 * M01 - s1 * M11;
                const double T10 = s1 * M00 + c1 * M10, T11 = s1 * M01 + c1 * M11;
                A[p1 + n * p2] = T00 * c2 - T01 * s2;
                if (q2ok) A[p1 + n * q2] = T00 * s2 + T01 * c2;
                if (q1ok) A[q1 + n * p2] = T10 * c2 - T11 * s2;
                if (q1ok && q2ok) A[q1 + n * q2] = T10 * s2 + T11 * c2;
            }
            // U <- U J
            for (int w = t0; w < n * half; w += blockDim.x) {
                const int row = w % n, k = w / n;
                const int p = (int)s_rot[4 * k], q = (int)s_rot[4 * k + 1];
                if (q >= n) continue;
                const double c = s_rot[4 * k + 2], s = s_rot[4 * k + 3];
                const double up = U[row + n * p], uq = U[row + n * q];
                U[row + n * p] = c * up - s * uq;
                U[row + n * q] = s * up + c * uq;
            }
            __syncthreads();
        }
    }
}

// indices of the nocc lowest eigenvalues (diagonal of A) into s_occ; thread 0
__device__ void select_occ(const double *A, int n, int nocc, int *s_occ, int *s_tmp) {
    if (threadIdx.x == 0) {
        for (int i = 0; i < n; ++i) s_tmp[i] = i;
        for (int a = 0; a < nocc; ++a) {
            int best = a;
            for (int b = a + 1; b < n; ++b)
                if (A[s_tmp[b] * (n + 1)] < A[s_tmp[best] * (n + 1)]) best = b;
            const int t = s_tmp[a];
            s_tmp[a] = s_tmp[best];
            s_tmp[best] = t;
            s_occ[a] = s_tmp[a];
        }
    }
    __syncthreads();
}

// Element (i, j), i >= j, of the packed lower triangle
__device__ __forceinline__ int packed(int i, int j) { return i * (i + 1) / 2 + j; }

// T = A + A^T (packed) for the A of G(D) = A + A^T, from the packed unique
// integrals (degeneracy weights 1/2 per index coincidence).  A wavefront takes
// rows ij of the triangle (one, two of up to 32 functions or four of up to 16):
//   - its 64 lanes load the row, kets kl = lane, lane + 64, ..., ahead of the
//     work on the row before, apply the weights, sum the row's J(ij) and, in
//     registers over all rows, J(kl), and lay the row down in LDS;
//   - then lane m takes row m of the symmetric matrix V(kl) whose triangle the
//     row is, and forms (V D_j)_m and (V D_i)_m for the exchange rows i and j.
//     The lane's LDS addresses in V are the same for every ij and stay in
//     registers; for t <= m they start at m (m + 1) / 2, which falls in distinct
//     banks for 32 consecutive m, and for t > m they are consecutive.  D is read
//     by broadcasts of two, and no two lanes add into one element.
// Every integral costs one HBM read, an LDS write and two LDS reads, against
// five reads of D, two of the index tables and three colliding atomics per
// value when each value is digested by itself.  Bounded by LDS (the broadcasts
// of D are half of its cycles): 35 functions, eight wavefronts alone on a CU
// 123 us, two workgroups of four 192 us each, against 400 us with two of eight;
// the integrals' HBM read alone is 83 us when every CU has its own.
template <class C>
struct FockRows {
    static constexpr int LANES = C::NP <= 16 ? 16 : C::NP <= 32 ? 32 : 64, ROWS = 64 / LANES;
    static constexpr int NMAX = C::NP < kBatchMaxN ? C::NP : kBatchMaxN;
    static constexpr int U = (NMAX * (NMAX + 1) / 2 + 63) / 64;
    static __host__ __device__ constexpr int ld(int n) { return (n + 7) & ~7; }
    // a row in LDS, with the zeros that its last 64 loads bring
    static __host__ __device__ constexpr int row(int n) {
        return ld(n) * (ld(n) + 1) / 2 > 64 * U ? ld(n) * (ld(n) + 1) / 2 : 64 * U;
    }
    // doubles of LDS: D's rows, T, and each wavefront's rows
    static __host__ __device__ constexpr int lds(int n) {
        return ld(n) * n + ((n * (n + 1) / 2 + 1) & ~1) + C::WAVES * ROWS * row(n);
    }
};
__device__ __forceinline__ void row_of(int r, int &i, int &j) {
    i = (int)((__builtin_amdgcn_sqrtf(8.0f * r + 1.0f) - 1.0f) * 0.5f);
    i += (i + 1) * (i + 2) / 2 <= r ? 1 : 0;   // (the root is within a rounding of it)
    i -= i * (i + 1) / 2 > r ? 1 : 0;
    j = r - i * (i + 1) / 2;
}

template <class C>
__device__ __forceinline__ void batch_fock(const double *__restrict__ eri, const double *__restrict__ D, double *arena,
                                           int n) {
    using R = FockRows<C>;
    constexpr int U = R::U, G = R::ROWS, STEP = C::WAVES * G;
    const int t = thread_index(), lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int P = n * (n + 1) / 2, ld = R::ld(n), PS = R::row(n);
    double *Dt = arena, *T = Dt + ld * n, *rows = T + ((P + 1) & ~1) + w * G * PS;
    // row i of D at Dt + ld i, zero beyond n
    for (int e = t; e < ld * n; e += C::THREADS) {
        const int i = e % n, j = e / n;
        Dt[j + ld * i] = j < n ? D[i + n * j] : 0.0;
    }
    for (int e = t; e < P; e += C::THREADS) T[e] = 0.0;
    for (int e = lane; e < G * PS; e += 64) rows[e] = 0.0;   // a row's entries beyond its own stay zero
    // a row's loads end at its length: buffer loads past it give 0 and read nothing
    double v[G][U];
    auto fetch = [&](int base) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int r = min(base + g, P - 1);
            const auto row = __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(eri + r * (r + 1) / 2), (short)0,
                                                               8 * (r + 1), 0x00020000);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                typedef int i2_t __attribute__((ext_vector_type(2)));
                const i2_t x = __builtin_amdgcn_raw_buffer_load_b64(row, 8 * lane + 512 * u, 0, 0);
                v[g][u] = __longlong_as_double(((long long)x.y << 32) | (unsigned)x.x);
            }
        }
    };
    fetch(w * G);
    __syncthreads();
    // the lane's kets: first the chunks of 64 that every row has work in, then the others
    constexpr int UA = (U + 1) / 2, UB = U - UA;
    double dka[UA], jka[UA], dkb[UB + 1], jkb[UB + 1];
    auto ket = [&](int u) {
        int k, l;
        row_of(min(lane + 64 * u, P - 1), k, l);
        return lane + 64 * u < P ? (k == l ? 1.0 : 2.0) * Dt[l + ld * k] : 0.0;
    };
#pragma unroll
    for (int u = 0; u < UA; ++u) {
        dka[u] = ket(u);
        jka[u] = 0.0;
    }
#pragma unroll
    for (int u = 0; u < UB; ++u) {
        dkb[u] = ket(UA + u);
        jkb[u] = 0.0;
    }
    const int g = lane / R::LANES, m = lane % R::LANES;
    // where row min(m, n - 1) of V holds column s
    const double *Vs[R::NMAX];
    {
        const int mm = min(m, n - 1);
#pragma unroll
        for (int s = 0; s < R::NMAX; ++s) Vs[s] = rows + g * PS + packed(max(mm, s), min(mm, s));
    }
    for (int base = w * G; base < P; base += STEP) {
        int imax = 0;
#pragma unroll
        for (int q = 0; q < G; ++q) {
            const int r = min(base + q, P - 1);   // (past the last row: it again, its sums dropped)
            int i, j;
            row_of(r, i, j);
            imax = __builtin_amdgcn_readfirstlane(i);
            const double d2 = base + q < P ? 2.0 * Dt[j + ld * i] : 0.0;
            double jr = 0.0, *to = rows + q * PS + lane;
#pragma unroll
            for (int u = 0; u < UA; ++u) {
                jr += v[q][u] * dka[u];
                jka[u] += v[q][u] * d2;
                to[64 * u] = v[q][u];
            }
            if (r >= 64 * UA) {   // (uniform)
#pragma unroll
                for (int u = 0; u < UB; ++u) {
                    jr += v[q][UA + u] * dkb[u];
                    jkb[u] += v[q][UA + u] * d2;
                    to[64 * (UA + u)] = v[q][UA + u];
                }
            }
            jr = wave_total(jr);
            if (lane == 0 && base + q < P) atomicAdd(&T[r], i == j ? 2.0 * jr : jr);
        }
        fetch(base + STEP);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the rows' writes before their reads
        const int r = base + g;
        int i, j;
        row_of(min(r, P - 1), i, j);
        const double *Di = Dt + ld * i, *Dj = Dt + ld * j;
        double y = 0.0, z = 0.0;
#pragma unroll
        for (int s = 0; s < R::NMAX; s += 8) {
            if (s <= imax) {   // (uniform)
                double vs[8];
                double2 di[4], dj[4];
#pragma unroll
                for (int k = 0; k < 8; ++k) vs[k] = *Vs[s + k];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    di[k] = *reinterpret_cast<const double2 *>(Di + s + 2 * k);
                    dj[k] = *reinterpret_cast<const double2 *>(Dj + s + 2 * k);
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    y += vs[2 * k] * dj[k].x;
                    z += vs[2 * k] * di[k].x;
                    y += vs[2 * k + 1] * dj[k].y;
                    z += vs[2 * k + 1] * di[k].y;
                }
            }
        }
        if (r < P && m <= i) {
            atomicAdd(&T[packed(i, m)], m == i ? -y : -0.5 * y);
            atomicAdd(&T[packed(max(j, m), min(j, m))], m == j ? -z : -0.5 * z);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the reads before the next rows' writes
    }
#pragma unroll
    for (int u = 0; u < UA; ++u)
        if (lane + 64 * u < P) atomicAdd(&T[lane + 64 * u], jka[u]);
#pragma unroll
    for (int u = 0; u < UB; ++u)
        if (lane + 64 * (UA + u) < P) atomicAdd(&T[lane + 64 * (UA + u)], jkb[u]);
    __syncthreads();
}

// LDS of a workgroup: the arena (two matrices of the dense part, the Fock
// build's D, T and rows, or the Jacobi fallback's matrices), then reductions
struct BScfLds {
    double *arena, *red, *part, *sum, *c, *B, *rot;
    int *occ, *tmp;
};
template <int WV>
__host__ __device__ constexpr int scf_tail_doubles() {
    // red, part, sum, c, B, rot, occ and tmp, the job
    return WV + 16 * WV + 10 * WV + kBatchDiis + kBatchDiis * kBatchDiis + 2 * (kBatchMaxN + 2) + kBatchMaxN + 2;
}
template <class C>
__host__ __device__ constexpr int scf_arena_doubles(int n) {
    const int dense = 2 * C::NP * (C::LD > C::NP + 1 ? C::LD : C::NP + 1), fock = FockRows<C>::lds(n);
    const int jac = 2 * n * n;
    const int x = dense > fock ? dense : fock;
    return ((x > jac ? x : jac) + 1) & ~1;
}

template <class C>
__device__ __forceinline__ void batch_solve(const BScfArgs &a, const BMol &mol, int m, const BScfLds &s) {
    constexpr int NP = C::NP, LD = C::LD, MD = kBatchDiis, MT = C::MT, TH = C::THREADS, WV = C::WAVES;
    constexpr int EL = (NP * NP + TH - 1) / TH;
    const int n = mol.n, nocc = mol.nocc, nn = n * n;
    const double *Sg = a.S + mol.mat0, *Hg = a.H + mol.mat0, *eri = a.eri + mol.eri0;
    double *X = a.scratch + 4 * mol.mat0, *Do = X + nn, *Fx = Do + nn, *D1 = Fx + nn, *D0 = a.Dout + mol.mat0;
    double *hF = a.hist + 2 * MD * mol.mat0, *hE = hF + MD * nn;
    double *sA = s.arena, *sB = s.arena + NP * LD;
    d4_t acc[MT];
    // X = S^-1/2 and S^1/2 (the latter in the DIIS history's place until that
    // is written); where 24 steps do not converge (condition numbers beyond
    // about 1e8) by the eigen-decomposition, which sees a singular S
    double *Xi = hE;
    {
    const int t = thread_index();
    if (!inv_sqrt_ns<C>(n, Sg, X, Xi, hF, hF + nn, s.arena, s.red, 24)) {
        double *A = s.arena, *Uv = A + nn;
        __syncthreads();
        for (int e = t; e < nn; e += TH) A[e] = Sg[e];
        __syncthreads();
        jacobi(A, Uv, n, s.rot, s.red);
        double smin = 1e300;
        for (int i = t; i < n; i += TH) smin = fmin(smin, A[i * (n + 1)]);
        smin = -wg_max(-smin, s.red);
        if (smin <= 1e-10) {
            if (t == 0) {
                a.energy[m] = 0.0;
                a.iters[m] = 0;
                a.conv[m] = -1;   // overlap numerically singular
                if (a.fallback) a.fallback[m] = 0;
            }
            return;
        }
        for (int e = t; e < nn; e += TH) {
            const int i = e % n, j = e / n;
            double x = 0.0, y = 0.0;
            for (int k = 0; k < n; ++k) {
                const double q = sqrt(A[k * (n + 1)]), uu = Uv[i + n * k] * Uv[j + n * k];
                x += uu / q;
                y += uu * q;
            }
            X[e] = x;
            Xi[e] = y;
        }
        __syncthreads();
    }
    }
    // From the Fock matrix in sA (and in Fx): the projector onto its nocc lowest
    // levels by purification, or by diagonalisation when the frontier levels
    // are too close for it, into Do; the density 2 X P X into Dn.
    auto new_density = [&](double *Dn) {
        const int t = thread_index();
        int steps;
        if (nocc == n) {
            for (int e = t; e < NP * NP; e += TH) {
                const int i = e % NP, j = e / NP;
                sA[i + LD * j] = i == j && i < n ? 1.0 : 0.0;
            }
        } else if (!purify<C>(sA, sB, n, nocc, 100, s.red, s.part, steps)) {
            double *A = s.arena, *Uv = A + nn;
            __syncthreads();
            for (int e = t; e < nn; e += TH) A[e] = Fx[e];
            __syncthreads();
            jacobi(A, Uv, n, s.rot, s.red);
            select_occ(A, n, nocc, s.occ, s.tmp);
            double p[EL];
#pragma unroll
            for (int q = 0; q < EL; ++q) {
                const int e = t + q * TH, i = e % NP, j = e / NP;
                p[q] = 0.0;
                if (i < n && j < n)
                    for (int x = 0; x < nocc; ++x) p[q] += Uv[i + n * s.occ[x]] * Uv[j + n * s.occ[x]];
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < EL; ++q) {
                const int e = t + q * TH;
                if (e < NP * NP) sA[e % NP + LD * (e / NP)] = p[q];
            }
        }
        __syncthreads();
        for (int e = t; e < nn; e += TH) Do[e] = sA[e % n + LD * (e / n)];
        load<C>(sB, X, n);
        __syncthreads();
        product<C>(sB, sA, acc);   // X P
        __syncthreads();
        to_lds<C>(sA, acc);
        __syncthreads();
        product<C>(sA, sB, acc);
        each<C>(acc, [&](int i, int j, double v) {
            if (i < n && j < n) Dn[i + n * j] = 2.0 * v;
        });
        __syncthreads();
    };
    // the Fock matrix in sB to the orthonormal basis, into sA
    auto orthonormal = [&]() {
        load<C>(sA, X, n);
        __syncthreads();
        product<C>(sA, sB, acc);   // X F
        __syncthreads();
        to_lds<C>(sB, acc);
        __syncthreads();
        product<C>(sB, sA, acc);
        __syncthreads();
        to_lds<C>(sA, acc);
    };
    // a start from the given density gets learned_iter iterations; if it
    // does not converge, the molecule restarts from the core guess in the
    // same workgroup with the full budget
    int it_total = 0, conv = 0, it = 0;
    double E = 0.0;
    double *D = D0;
    for (int attempt = a.guess ? 0 : 1; attempt < 2; ++attempt) {
        const bool from_guess = attempt == 0;
        const int maxit = from_guess ? a.learned_iter : a.max_iter;
        D = D0;
        if (from_guess) {
            const int t = thread_index(), lane = t & 63, w = t >> 6;
            // Do = S^{1/2} D S^{1/2} / 2; the given D need not be symmetric
            for (int e = t; e < nn; e += TH) D0[e] = a.guess[mol.mat0 + e];
            load<C>(sA, a.guess + mol.mat0, n);
            load<C>(sB, Xi, n);
            __syncthreads();
            product<C>(sA, sB, acc);
            __syncthreads();
            to_lds<C>(sA, acc);
            __syncthreads();
            const int g = lane >> 4, c = lane & 15;
#pragma unroll
            for (int q = 0; q < MT; ++q) {
                const int tile = w + q * WV;
                if (tile >= C::T2) break;
                const double *pa = sB + 16 * (tile % C::NT) + c + LD * g, *pb = sA + LD * (16 * (tile / C::NT) + c) + g;
                acc[q] = (d4_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int k = 0; k < NP; k += 4) acc[q] = mfma64(pa[LD * k], pb[k], acc[q]);
            }
            each<C>(acc, [&](int i, int j, double v) {
                if (i < n && j < n) Do[i + n * j] = 0.5 * v;
            });
            __syncthreads();
        } else {
            // core Hamiltonian guess (scf.f90:410-512)
            load<C>(sB, Hg, n);
            orthonormal();
            each<C>(acc, [&](int i, int j, double v) {
                if (i < n && j < n) Fx[i + n * j] = v;
            });
            __syncthreads();
            new_density(D0);
        }
        int hist = 0, head = 0;
        double E_old = 0.0, dE_prev = 1e300, err_prev = 1e300;
        bool abandoned = false;
        E = 0.0;
        for (it = 1; it <= maxit + 1; ++it) {
            // F = H + G(D); E = (D.F + D.H)/2 + E_nuc, and the density's change
            const int t = thread_index(), lane = t & 63, w = t >> 6;
            double *Dn = D == D0 ? D1 : D0;   // D_{k-1}, and D_{k+1}'s place
            batch_fock<C>(eri, D, s.arena, n);
            double f[EL], ed = 0.0, dd = 0.0;
            {
                const int ld = FockRows<C>::ld(n);
                const double *Dt = s.arena, *T = Dt + ld * n;
#pragma unroll
                for (int q = 0; q < EL; ++q) {
                    const int e = t + q * TH, i = e % NP, j = e / NP;
                    f[q] = 0.0;
                    if (i < n && j < n) {
                        const double h = Hg[i + n * j], d = Dt[j + ld * i];
                        f[q] = h + T[packed(max(i, j), min(i, j))];
                        ed += d * (f[q] + h);
                        if (it > 1) dd = fmax(dd, fabs(d - Dn[i + n * j]));
                    }
                }
            }
            ed = wave_total(ed);
            dd = wave_largest(dd);
            if (lane == 0) {
                s.sum[2 * w] = ed;
                s.sum[2 * w + 1] = dd;
            }
            __syncthreads();   // (and D, T and the rows are free)
            ed = dd = 0.0;
            for (int q = 0; q < WV; ++q) {
                ed += s.sum[2 * q];
                dd = fmax(dd, s.sum[2 * q + 1]);
            }
            E = 0.5 * ed + mol.e_nuc;
            // the previous iteration's convergence
            if (it > 2 && dE_prev < a.e_tol && dd < a.d_tol && err_prev < 100.0 * a.d_tol) {
                conv = 1;
                break;
            }
            if (it > maxit) break;
#pragma unroll
            for (int q = 0; q < EL; ++q) {
                const int e = t + q * TH;
                if (e < NP * NP) sB[e % NP + LD * (e / NP)] = f[q];
            }
            // F' = X F X into the history; error F' Do - Do F'
            orthonormal();
            double *fs = hF + head * nn, *es = hE + head * nn;
            each<C>(acc, [&](int i, int j, double v) {
                if (i < n && j < n) fs[i + n * j] = v;
            });
            load<C>(sB, Do, n);
            __syncthreads();
            product<C>(sA, sB, acc);
            __syncthreads();
            to_lds<C>(sB, acc);
            __syncthreads();
            const int hn = min(hist + 1, MD);
            double dots[MD];
#pragma unroll
            for (int q = 0; q < MD; ++q) dots[q] = 0.0;
            for (int e = t; e < nn; e += TH) {
                const int i = e % n, j = e / n;
                const double ev = sB[i + LD * j] - sB[j + LD * i];
                es[e] = ev;
#pragma unroll
                for (int q = 0; q < MD; ++q)
                    if (q < hn) dots[q] += ev * (q == head ? ev : hE[q * nn + e]);
            }
#pragma unroll
            for (int q = 0; q < MD; ++q) {
                const double v = wave_total(dots[q]);
                if (lane == 0) s.sum[w * MD + q] = v;
            }
            __syncthreads();
            if (t < hn) {
                double v = 0.0;
                for (int q = 0; q < WV; ++q) v += s.sum[q * MD + t];
                s.B[head * MD + t] = v;
                s.B[t * MD + head] = v;
            }
            __syncthreads();
            hist = hn;
            // DIIS extrapolation of F' into sA
            if (w == 0) diis_wave(s.B, hist, head, s.c);
            __syncthreads();
            for (int e = t; e < NP * NP; e += TH) {
                const int i = e % NP, j = e / NP;
                double v = 0.0;
                if (i < n && j < n) {
                    const int x = i + n * j;
#pragma unroll
                    for (int q = 0; q < MD; ++q)
                        if (q < hist) v += s.c[q] * hF[q * nn + x];
                    Fx[x] = v;
                }
                sA[i + LD * j] = v;
            }
            err_prev = sqrt(fabs(s.B[head * MD + head]));
            dE_prev = fabs(E - E_old);
            E_old = E;
            head = (head + 1) % MD;
            __syncthreads();
            // a start from the guess that is far from converging by
            // check_it iterations restarts now rather than at learned_iter
            if (from_guess && a.restart && it == a.check_it && err_prev > a.check_err) {
                abandoned = true;
                break;
            }
            new_density(Dn);
            D = Dn;
        }
        it_total += abandoned ? it : min(it - 1, maxit);
        if (conv || !from_guess || !a.restart) {
            if (threadIdx.x == 0 && a.fallback) a.fallback[m] = from_guess ? 0 : (a.guess ? 1 : 0);
            break;
        }
    }
    const int t = thread_index();
    if (D != D0)
        for (int e = t; e < nn; e += TH) D0[e] = D[e];
    if (t == 0) {
        a.energy[m] = E;
        a.iters[m] = it_total;
        a.conv[m] = conv;
    }
}

// Registers bound the residency (256 VGPRs: two wavefronts per SIMD; at 128 the
// Fock rows spill and a build takes twice as long).  1024 clusters of 2 to 5
// waters: 17 ms -> 6.3 ms; of an iteration's 218 us at 35 functions (eight
// wavefronts) 123 are the Fock build, 51 the 30 purification steps, 10 X F X, 21
// the DIIS error, its dots and the extrapolation.  The two Jacobi
// diagonalisations of a molecule's start, 870 us, are 81 us of Newton-Schulz and
// a purification.
// arena_doubles: the largest of the batch's molecules (scf_lds_bytes)
template <int WV>
__global__ __launch_bounds__(64 * WV, 2) void k_batch_scf(BScfArgs a, int arena_doubles) {
    extern __shared__ __attribute__((aligned(16))) double smem[];
    BScfLds s;
    s.arena = smem;
    s.red = s.arena + arena_doubles;
    s.part = s.red + WV;
    s.sum = s.part + 16 * WV;
    s.c = s.sum + 10 * WV;
    s.B = s.c + kBatchDiis;
    s.rot = s.B + kBatchDiis * kBatchDiis;
    s.occ = reinterpret_cast<int *>(s.rot + 2 * (kBatchMaxN + 2));
    s.tmp = s.occ + kBatchMaxN;
    int *s_job = s.tmp + kBatchMaxN;
    while (true) {
        __syncthreads();
        if (threadIdx.x == 0) *s_job = atomicAdd(a.counter, 1);
        __syncthreads();
        const int job = __builtin_amdgcn_readfirstlane(*s_job);
        if (job >= a.nmol) break;
        const int m = __builtin_amdgcn_readfirstlane(a.order[job]);
        // (in scalar registers, which the compiler cannot tell by itself)
        union {
            BMol mol;
            int word[sizeof(BMol) / 4];
        } x;
#pragma unroll
        for (int k = 0; k < (int)(sizeof(BMol) / 4); ++k)
            x.word[k] = __builtin_amdgcn_readfirstlane(reinterpret_cast<const int *>(a.mols + m)[k]);
        const BMol mol = x.mol;
        if (mol.n <= 16) batch_solve<DenseLds<16, WV>>(a, mol, m, s);
        else if (mol.n <= 32) batch_solve<DenseLds<32, WV>>(a, mol, m, s);
        else batch_solve<DenseLds<48, WV>>(a, mol, m, s);
    }
}

template <int WV>
static size_t scf_lds_doubles(const std::vector<BMol> &mols, int *arena) {
    int x = 0;
    for (const BMol &m : mols)
        x = std::max(x, m.n <= 16 ? scf_arena_doubles<DenseLds<16, WV>>(m.n)
                                  : m.n <= 32 ? scf_arena_doubles<DenseLds<32, WV>>(m.n)
                                              : scf_arena_doubles<DenseLds<48, WV>>(m.n));
    *arena = x;
    return x + scf_tail_doubles<WV>();
}
// bytes of LDS and the arena's doubles at `threads` per workgroup
static size_t scf_lds_bytes(const std::vector<BMol> &mols, int threads, int *arena) {
    const size_t d = threads == 64    ? scf_lds_doubles<1>(mols, arena)
                     : threads == 128 ? scf_lds_doubles<2>(mols, arena)
                     : threads == 256 ? scf_lds_doubles<4>(mols, arena)
                                      : scf_lds_doubles<8>(mols, arena);
    return sizeof(double) * d;
}

__global__ void k_zero_int(int *p, int cnt) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < cnt) p[i] = 0;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
constexpr int kScfThreads = 256;   // of a batch that is not tuned; its LDS fits for every n

struct BatchState {
    int nmol = 0, nmax = 0, npairs = 0, natom = 0;
    long long total_eri = 0, total_mat = 0, nq[6] = {0, 0, 0, 0, 0, 0};
    std::vector<BMol> mols;
    std::vector<int> order;
    BMol *d_mols = nullptr;
    int *d_order = nullptr, *d_pair_mol = nullptr, *d_cls[3] = {nullptr, nullptr, nullptr};
    int ncls[3] = {0, 0, 0};
    double *d_ksoa[3] = {nullptr, nullptr, nullptr};   // per class list (ket_soa.h)
    ShellPair *d_pairs = nullptr;
    PrimPair *d_prims = nullptr;
    double *d_atoms = nullptr, *d_ftT = nullptr;
    long long *d_qcum[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    int *d_qfirst[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    double *d_eri = nullptr, *d_S = nullptr, *d_H = nullptr, *d_D = nullptr, *d_guess = nullptr, *d_scratch = nullptr,
           *d_hist = nullptr, *d_energy = nullptr;
    int *d_iters = nullptr, *d_conv = nullptr, *d_counter = nullptr;
    // atom pairs of the learned guess
    bool guess_ok = false;
    int npair = 0;
    PairRec *d_pairrec = nullptr;
    int *d_mol_atoms = nullptr, *d_fail = nullptr;
    std::vector<int> pair_mol_of;   // molecule of each pair record
    hipGraphExec_t graph_learned = nullptr;
    double gl_etol = 0, gl_dtol = 0;
    int gl_maxit = 0, gl_gen = -1;
    // launch shapes (autotuned) and the captured graph
    int eri_threads[6] = {256, 256, 256, 256, 256, 256};
    int scf_threads = kScfThreads;
    bool tuned = false;
    hipGraphExec_t graph = nullptr;
    bool graph_guess = false;
    double g_etol = 0, g_dtol = 0;
    int g_maxit = 0;
    int replays = 0;
    void release() {
        void **ps[] = {(void **)&d_mols,   (void **)&d_order,  (void **)&d_pair_mol, (void **)&d_cls[0],
                       (void **)&d_cls[1], (void **)&d_cls[2], (void **)&d_pairs,    (void **)&d_prims,
                       (void **)&d_atoms,  (void **)&d_ftT,    (void **)&d_eri,      (void **)&d_S,
                       (void **)&d_H,      (void **)&d_D,      (void **)&d_guess,    (void **)&d_scratch,
                       (void **)&d_hist,   (void **)&d_energy, (void **)&d_iters,    (void **)&d_conv,
                       (void **)&d_counter, (void **)&d_pairrec, (void **)&d_mol_atoms, (void **)&d_fail};
        for (auto p : ps) dfree(p);
        if (graph_learned) (void)hipGraphExecDestroy(graph_learned);
        graph_learned = nullptr;
        for (auto &q : d_qcum) dfree((void **)&q);
        for (auto &q : d_qfirst) dfree((void **)&q);
        for (auto &q : d_ksoa) dfree((void **)&q);
        if (graph) (void)hipGraphExecDestroy(graph);
        graph = nullptr;
        nmol = 0;
        tuned = false;
    }
};

void free_batch(myqc_ctx *ctx) {
    if (ctx->batch) {
        ctx->batch->release();
        delete ctx->batch;
        ctx->batch = nullptr;
    }
}

static const int kCB[6] = {0, 1, 1, 2, 2, 2}, kCK[6] = {0, 0, 1, 0, 1, 2};

static void launch_batch_eri(myqc_ctx *ctx, BatchState &b, int c, int threads) {
    BEriArgs a;
    a.pairs = b.d_pairs;
    a.prims = b.d_prims;
    a.ftT = b.d_ftT;
    a.mols = b.d_mols;
    a.cls0 = b.d_cls[0];
    a.cls1 = b.d_cls[1];
    a.cls2 = b.d_cls[2];
    a.ksoa = b.d_ksoa[kCK[c]];
    a.nket = b.ncls[kCK[c]];
    a.qcum = b.d_qcum[c];
    a.qfirst = b.d_qfirst[c];
    a.nq = b.nq[c];
    a.eri = b.d_eri;
    const unsigned grid = (unsigned)((b.nq[c] + threads - 1) / threads);
    switch (c) {
        case 0: k_batch_eri<0, 0><<<grid, threads, 0, ctx->stream>>>(a); break;
        case 1: k_batch_eri<1, 0><<<grid, threads, 0, ctx->stream>>>(a); break;
        case 2: k_batch_eri<1, 1><<<grid, threads, 0, ctx->stream>>>(a); break;
        case 3: k_batch_eri<2, 0><<<grid, threads, 0, ctx->stream>>>(a); break;
        case 4: k_batch_eri<2, 1><<<grid, threads, 0, ctx->stream>>>(a); break;
        default: k_batch_eri<2, 2><<<grid, threads, 0, ctx->stream>>>(a); break;
    }
}

static void launch_batch_one_e(myqc_ctx *ctx, const BatchState &b) {
    const int per = 256 / kOneELanes;
    k_batch_one_e<<<std::min((b.npairs + per - 1) / per, kOneEBlocks), 256, 0, ctx->stream>>>(
        b.d_pairs, b.d_prims, b.d_ftT, b.d_atoms, b.d_pair_mol, b.d_mols, b.d_cls[0], b.d_cls[1], b.d_cls[2],
        b.ncls[0], b.ncls[1], b.ncls[2], b.d_S, b.d_H);
}

// as many workgroups as the registers of the SCF kernel let a CU hold
static int scf_grid(myqc_ctx *ctx, const BatchState &b, int threads) {
    int cus = 256;
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device);
    return std::max(1, std::min(b.nmol, std::max(1024 / threads, 4) * cus));
}

// A start from the guess whose DIIS error is still above kCheckErr after
// kCheckIt iterations restarts from the core guess there (not at
// learned_iter).  Measured on the seeded 4096 batch: 25 / 1e-3 keeps 99.05 %
// converged (20 / 1e-3: 98.9 %, but 16 % faster).
constexpr int kCheckIt = 25;
constexpr double kCheckErr = 1e-3;

// restart: a start from the guess that does not converge within
// learned_iter iterations restarts from the core guess (same launch)
static void launch_batch_scf(myqc_ctx *ctx, BatchState &b, bool guess, double e_tol, double d_tol, int max_iter,
                             int threads, const int *order = nullptr, int count = -1, bool restart = false,
                             int learned_iter = 0) {
    BScfArgs a;
    a.mols = b.d_mols;
    a.order = order ? order : b.d_order;
    a.nmol = count >= 0 ? count : b.nmol;
    a.counter = b.d_counter;
    a.eri = b.d_eri;
    a.S = b.d_S;
    a.H = b.d_H;
    a.guess = guess ? b.d_guess : nullptr;
    a.scratch = b.d_scratch;
    a.hist = b.d_hist;
    a.Dout = b.d_D;
    a.energy = b.d_energy;
    a.iters = b.d_iters;
    a.conv = b.d_conv;
    a.e_tol = e_tol;
    a.d_tol = d_tol;
    a.max_iter = max_iter;
    a.restart = (guess && restart) ? 1 : 0;
    a.learned_iter = a.restart ? std::min(learned_iter, max_iter) : max_iter;
    a.fallback = b.d_fail;
    a.check_it = kCheckIt;
    a.check_err = kCheckErr;
    k_zero_int<<<1, 64, 0, ctx->stream>>>(b.d_counter, 1);
    const int grid = std::max(1, std::min(scf_grid(ctx, b, threads), a.nmol));
    int arena = 0;
    const size_t lds = scf_lds_bytes(b.mols, threads, &arena);
    switch (threads) {
        case 64: k_batch_scf<1><<<grid, threads, lds, ctx->stream>>>(a, arena); break;
        case 128: k_batch_scf<2><<<grid, threads, lds, ctx->stream>>>(a, arena); break;
        case 256: k_batch_scf<4><<<grid, threads, lds, ctx->stream>>>(a, arena); break;
        default: k_batch_scf<8><<<grid, threads, lds, ctx->stream>>>(a, arena); break;
    }
}

// the whole pipeline: integrals, then the SCF
static void launch_batch(myqc_ctx *ctx, BatchState &b, bool guess, double e_tol, double d_tol, int max_iter) {
    launch_batch_one_e(ctx, b);
    for (int c = 0; c < 6; ++c)
        if (b.nq[c] > 0) launch_batch_eri(ctx, b, c, b.eri_threads[c]);
    launch_batch_scf(ctx, b, guess, e_tol, d_tol, max_iter, b.scf_threads);
}

// Autotuner: times each candidate launch shape on this batch with HIP events
// and keeps the fastest (ERI: 64/128/256 threads per class; SCF: 64/128/256/512
// threads per molecule's workgroup).
static int batch_tune(myqc_ctx *ctx, BatchState &b, bool guess, double e_tol, double d_tol, int max_iter) {
    hipEvent_t e0, e1;
    MYQC_HIP(ctx, hipEventCreate(&e0));
    MYQC_HIP(ctx, hipEventCreate(&e1));
    auto timed = [&](auto &&launch) -> float {
        float best = 1e30f;
        for (int rep = 0; rep < 2; ++rep) {
            (void)hipEventRecord(e0, ctx->stream);
            launch();
            (void)hipEventRecord(e1, ctx->stream);
            (void)hipEventSynchronize(e1);
            float ms = 0.f;
            (void)hipEventElapsedTime(&ms, e0, e1);
            best = std::min(best, ms);
        }
        return best;
    };
    for (int c = 0; c < 6; ++c) {
        if (b.nq[c] == 0) continue;
        float best = 1e30f;
        for (int th : {64, 128, 256}) {
            const float ms = timed([&] { launch_batch_eri(ctx, b, c, th); });
            if (ms < best) {
                best = ms;
                b.eri_threads[c] = th;
            }
        }
    }
    launch_batch_one_e(ctx, b);
    float best = 1e30f;
    int lds_limit = 65536;
    (void)hipDeviceGetAttribute(&lds_limit, hipDeviceAttributeMaxSharedMemoryPerBlock, ctx->device);
    for (int th : {64, 128, 256, 512}) {
        int arena = 0;
        if (scf_lds_bytes(b.mols, th, &arena) > (size_t)lds_limit) continue;
        const float ms = timed([&] { launch_batch_scf(ctx, b, guess, e_tol, d_tol, max_iter, th); });
        if (ms < best) {
            best = ms;
            b.scf_threads = th;
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    MYQC_HIP(ctx, hipGetLastError());
    b.tuned = true;
    return 0;
}

template <typename T>
static int upload(myqc_ctx *ctx, T **dst, const std::vector<T> &src) {
    MYQC_CHECK(dalloc(ctx, (void **)dst, sizeof(T) * std::max<size_t>(src.size(), 1)));
    if (!src.empty())
        MYQC_HIP(ctx, hipMemcpyAsync(*dst, src.data(), sizeof(T) * src.size(), hipMemcpyHostToDevice, ctx->stream));
    return 0;
}

}  // namespace myqc

using namespace myqc;

extern "C" int myqc_batch_set(myqc_ctx *ctx, int nmol, const int *mol_nnuc, const int *mol_norb, const int *mol_nocc,
                              const int *Z, const double *xyz_bohr, const double *set_alpha, const int *setinfo,
                              const double *bas, const int *basinfo, const int *offsets, const double *Ftab) {
    if (!ctx || nmol <= 0 || !mol_nnuc || !mol_norb || !mol_nocc || !Z || !xyz_bohr || !set_alpha || !setinfo ||
        !bas || !basinfo || !offsets || !Ftab)
        return MYQC_E_ARG;
    free_batch(ctx);
    ctx->batch = new BatchState();
    BatchState &b = *ctx->batch;
    std::vector<ShellPair> pairs;
    std::vector<PrimPair> prims;
    std::vector<int> cls[3], pair_mol, weight;
    std::vector<double> atoms;
    b.mols.resize(nmol);
    int atom0 = 0;
    long long eri0 = 0, mat0 = 0;
    for (int m = 0; m < nmol; ++m) {
        const int nnuc = mol_nnuc[m], norb = mol_norb[m];
        if (nnuc <= 0 || norb <= 0 || norb > kBatchMaxN || mol_nocc[m] < 1 || mol_nocc[m] > norb)
            return set_error(ctx, MYQC_E_ARG, "myqc_batch_set: molecule %d: %d atoms, %d functions, %d occupied "
                             "(1..%d functions per molecule)", m, nnuc, norb, mol_nocc[m], kBatchMaxN);
        // this molecule's slices: offsets[4 m + {0: set_alpha, 1: setinfo, 2: bas, 3: basinfo}]
        const int *o = offsets + 4 * m;
        std::vector<double> xyz(3 * nnuc);
        for (int a = 0; a < nnuc; ++a)
            for (int c = 0; c < 3; ++c) xyz[3 * a + c] = xyz_bohr[3 * atom0 + a + nnuc * c];
        std::vector<Shell> shells;
        std::vector<ShellPair> mp;
        std::vector<PrimPair> mpr;
        std::vector<int> ids[3];
        const int *si = setinfo + o[1];
        const std::string why = build_system(nnuc, xyz.data(), si[0], set_alpha + o[0], si, bas + o[2], norb,
                                             basinfo + o[3], shells, mp, mpr, ids);
        if (!why.empty()) return set_error(ctx, MYQC_E_ARG, "myqc_batch_set: molecule %d: %s", m, why.c_str());
        // kets with similar numbers of primitive pairs above the screen run in
        // the same wavefronts (of 5 waters, a wavefront executed 0.62 of all
        // primitive quartets of (ss|ss) in the pairs' own order, 0.39 in this one;
        // 0.28 survive; 1024 clusters 2.98 -> 2.21 ms): by the primitive pairs
        // that pass alone halfway to it, then at it
        {
            weight.assign(mp.size(), 0);
            for (size_t q = 0; q < mp.size(); ++q)
                for (int i = 0; i < mp[q].npp; ++i) {
                    const double e = mpr[mp[q].pp0 + i].EIJ;
                    if (e < 1e-14) break;   // (largest first)
                    weight[q] += e >= 1e-7 ? 101 : 1;
                }
            for (auto &v : ids)
                std::stable_sort(v.begin(), v.end(), [&](int x, int y) { return weight[x] > weight[y]; });
        }
        BMol &mol = b.mols[m];
        mol.n = norb;
        mol.nocc = mol_nocc[m];
        mol.nnuc = nnuc;
        mol.atom0 = atom0;
        mol.eri0 = eri0;
        mol.mat0 = mat0;
        double en = 0.0;
        for (int a = 0; a < nnuc; ++a) {
            atoms.push_back(Z[atom0 + a]);
            for (int c = 0; c < 3; ++c) atoms.push_back(xyz[3 * a + c]);
            for (int c = 0; c < a; ++c) {
                const double dx = xyz[3 * a] - xyz[3 * c], dy = xyz[3 * a + 1] - xyz[3 * c + 1],
                             dz = xyz[3 * a + 2] - xyz[3 * c + 2];
                en += (double)Z[atom0 + a] * Z[atom0 + c] / sqrt(dx * dx + dy * dy + dz * dz);
            }
        }
        mol.e_nuc = en;
        const int p0 = (int)pairs.size(), q0 = (int)prims.size();
        for (auto sp : mp) {
            sp.pp0 += q0;
            pairs.push_back(sp);
            pair_mol.push_back(m);
        }
        prims.insert(prims.end(), mpr.begin(), mpr.end());
        for (int c = 0; c < 3; ++c) {
            mol.cls0[c] = (int)cls[c].size();
            mol.ncls[c] = (int)ids[c].size();
            for (int id : ids[c]) cls[c].push_back(p0 + id);
        }
        atom0 += nnuc;
        eri0 += tri(tri(norb));
        mat0 += (long long)norb * norb;
        b.nmax = std::max(b.nmax, norb);
    }
    // atom pairs A <= B for the learned guess (H, He: 1 function; Li..Ne: 5,
    // atoms' functions contiguous in atom order)
    std::vector<PairRec> prs;
    std::vector<int> mol_atoms(2 * nmol);
    b.guess_ok = true;
    for (int m = 0; m < nmol; ++m) {
        const BMol &mol = b.mols[m];
        mol_atoms[2 * m] = mol.atom0;
        mol_atoms[2 * m + 1] = mol.nnuc;
        std::vector<int> ao(mol.nnuc), nf(mol.nnuc);
        int a0 = 0;
        for (int a = 0; a < mol.nnuc; ++a) {
            const int z = Z[mol.atom0 + a];
            if (z < 1 || z > 10) b.guess_ok = false;
            nf[a] = z <= 2 ? 1 : 5;
            ao[a] = a0;
            a0 += nf[a];
        }
        if (a0 != mol.n) b.guess_ok = false;
        for (int a = 0; a < mol.nnuc; ++a)
            for (int c = a; c < mol.nnuc; ++c) {
                PairRec r;
                r.mol = m;
                r.a = mol.atom0 + a;
                r.b = mol.atom0 + c;
                r.aoA = ao[a];
                r.aoB = ao[c];
                r.nA = nf[a];
                r.nB = nf[c];
                r.n = mol.n;
                r.mat0 = mol.mat0;
                prs.push_back(r);
                b.pair_mol_of.push_back(m);
            }
    }
    b.npair = (int)prs.size();
    MYQC_CHECK(upload(ctx, &b.d_pairrec, prs));
    MYQC_CHECK(upload(ctx, &b.d_mol_atoms, mol_atoms));
    MYQC_CHECK(dalloc(ctx, (void **)&b.d_fail, sizeof(int) * nmol));
    b.nmol = nmol;
    b.npairs = (int)pairs.size();
    b.total_eri = eri0;
    b.total_mat = mat0;
    b.order.resize(nmol);
    std::iota(b.order.begin(), b.order.end(), 0);
    std::stable_sort(b.order.begin(), b.order.end(), [&](int x, int y) { return b.mols[x].n > b.mols[y].n; });
    std::vector<long long> qcum[6];
    std::vector<int> qfirst[6];
    for (int c = 0; c < 6; ++c) {
        std::vector<long long> &qc = qcum[c];
        qc.assign(nmol + 1, 0);
        for (int m = 0; m < nmol; ++m) {
            const long long nb = b.mols[m].ncls[kCB[c]], nk = b.mols[m].ncls[kCK[c]];
            qc[m + 1] = qc[m] + (kCB[c] == kCK[c] ? tri(nb) : nb * nk);
        }
        b.nq[c] = qc[nmol];
        qfirst[c] = quartet_marks(qc);
        MYQC_CHECK(upload(ctx, &b.d_qcum[c], qc));
        MYQC_CHECK(upload(ctx, &b.d_qfirst[c], qfirst[c]));
    }
    std::vector<double> ftT(FT_TOTAL);
    boys_inputs(Ftab, ftT.data() + FT_EG);
    MYQC_CHECK(upload(ctx, &b.d_mols, b.mols));
    MYQC_CHECK(upload(ctx, &b.d_order, b.order));
    MYQC_CHECK(upload(ctx, &b.d_pair_mol, pair_mol));
    for (int c = 0; c < 3; ++c) MYQC_CHECK(upload(ctx, &b.d_cls[c], cls[c]));
    MYQC_CHECK(upload(ctx, &b.d_pairs, pairs));
    MYQC_CHECK(upload(ctx, &b.d_prims, prims));
    for (const ShellPair &sp : pairs)
        if (sp.npp > kKetPrims)
            return set_error(ctx, MYQC_E_ARG, "myqc_batch_set: a shell pair has %d primitive pairs (at most %d)", sp.npp,
                             kKetPrims);
    for (int c = 0; c < 3; ++c) {
        b.ncls[c] = (int)cls[c].size();
        if (b.ncls[c] == 0) continue;
        MYQC_CHECK(dalloc(ctx, (void **)&b.d_ksoa[c], sizeof(double) * kKetPrims * kKetFields * (size_t)b.ncls[c]));
        k_ket_soa<<<dim3((b.ncls[c] + 255) / 256, kKetPrims), 256, 0, ctx->stream>>>(b.d_pairs, b.d_prims, b.d_cls[c],
                                                                                  b.ncls[c], b.d_ksoa[c]);
        MYQC_HIP(ctx, hipGetLastError());
    }
    MYQC_CHECK(upload(ctx, &b.d_atoms, atoms));
    b.natom = (int)(atoms.size() / 4);
    MYQC_CHECK(upload(ctx, &b.d_ftT, ftT));
    k_boys_rows<<<kBoysRowBlocks, 64, 0, ctx->stream>>>(b.d_ftT);
    MYQC_HIP(ctx, hipGetLastError());
    const size_t M = (size_t)std::max<long long>(b.total_mat, 1);
    MYQC_CHECK(dalloc(ctx, (void **)&b.d_eri, sizeof(double) * std::max<long long>(b.total_eri, 1)));
    MYQC_CHECK(dalloc(ctx, (void **)&b.d_S, sizeof(double) * M));
    MYQC_CHECK(dalloc(ctx, (void **)&b.d_H, sizeof(double) * M));
    MYQC_CHECK(dalloc(ctx, (void **)&b.d_D, sizeof(double) * M));
    MYQC_CHECK(dalloc(ctx, (void **)&b.d_guess, sizeof(double) * M));
    MYQC_CHECK(dalloc(ctx, (void **)&b.d_scratch, sizeof(double) * 4 * M));
    MYQC_CHECK(dalloc(ctx, (void **)&b.d_hist, sizeof(double) * 2 * kBatchDiis * M));
    MYQC_CHECK(dalloc(ctx, (void **)&b.d_energy, sizeof(double) * nmol));
    MYQC_CHECK(dalloc(ctx, (void **)&b.d_iters, sizeof(int) * nmol));
    MYQC_CHECK(dalloc(ctx, (void **)&b.d_conv, sizeof(int) * nmol));
    MYQC_CHECK(dalloc(ctx, (void **)&b.d_counter, sizeof(int) * 64));
    MYQC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    int lds_limit = 65536;
    (void)hipDeviceGetAttribute(&lds_limit, hipDeviceAttributeMaxSharedMemoryPerBlock, ctx->device);
    int arena = 0;
    if (scf_lds_bytes(b.mols, kScfThreads, &arena) > (size_t)lds_limit)
        return set_error(ctx, MYQC_E_ARG, "myqc_batch_set: n=%d needs %zu B of LDS per workgroup (limit %d)", b.nmax,
                         scf_lds_bytes(b.mols, kScfThreads, &arena), lds_limit);
    return 0;
}

extern "C" int myqc_batch_rhf(myqc_ctx *ctx, const double *D_guess, double e_tol, double d_tol, int max_iter,
                              double *energy, int *iterations, int *converged) {
    if (!ctx || !energy || e_tol <= 0 || d_tol <= 0 || max_iter < 1) return MYQC_E_ARG;
    if (!ctx->batch || ctx->batch->nmol == 0) return set_error(ctx, MYQC_E_STATE, "myqc_batch_rhf: no batch set");
    BatchState &b = *ctx->batch;
    const bool guess = D_guess != nullptr;
    if (guess)
        MYQC_HIP(ctx, hipMemcpyAsync(b.d_guess, D_guess, sizeof(double) * b.total_mat, hipMemcpyHostToDevice,
                                     ctx->stream));
    if (!b.tuned) MYQC_CHECK(batch_tune(ctx, b, guess, e_tol, d_tol, max_iter));
    if (!b.graph || b.graph_guess != guess || b.g_etol != e_tol || b.g_dtol != d_tol || b.g_maxit != max_iter) {
        if (b.graph) (void)hipGraphExecDestroy(b.graph);
        b.graph = nullptr;
        hipGraph_t g;
        MYQC_HIP(ctx, hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
        launch_batch(ctx, b, guess, e_tol, d_tol, max_iter);
        MYQC_HIP(ctx, hipStreamEndCapture(ctx->stream, &g));
        hipError_t e = hipGraphInstantiate(&b.graph, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) {
            b.graph = nullptr;
            return set_error(ctx, MYQC_E_HIP, "myqc_batch_rhf: graph instantiation failed: %s", hipGetErrorString(e));
        }
        b.graph_guess = guess;
        b.g_etol = e_tol;
        b.g_dtol = d_tol;
        b.g_maxit = max_iter;
    }
    MYQC_HIP(ctx, hipGraphLaunch(b.graph, ctx->stream));
    ++b.replays;
    MYQC_HIP(ctx, d2h(ctx, energy, b.d_energy, sizeof(double) * b.nmol));
    if (iterations) MYQC_HIP(ctx, d2h(ctx, iterations, b.d_iters, sizeof(int) * b.nmol));
    std::vector<int> conv(b.nmol);
    MYQC_HIP(ctx, d2h(ctx, conv.data(), b.d_conv, sizeof(int) * b.nmol));
    if (converged) std::copy(conv.begin(), conv.end(), converged);
    return 0;
}

extern "C" int myqc_batch_density(myqc_ctx *ctx, double *D) {
    if (!ctx || !D) return MYQC_E_ARG;
    if (!ctx->batch || ctx->batch->nmol == 0) return set_error(ctx, MYQC_E_STATE, "myqc_batch_density: no batch set");
    MYQC_HIP(ctx, d2h(ctx, D, ctx->batch->d_D, sizeof(double) * ctx->batch->total_mat));
    return 0;
}

extern "C" int myqc_batch_info(myqc_ctx *ctx, int *eri_threads, int *scf_threads, int *graph_replays,
                               long long *n_integrals) {
    if (!ctx) return MYQC_E_ARG;
    if (!ctx->batch) return set_error(ctx, MYQC_E_STATE, "myqc_batch_info: no batch set");
    const BatchState &b = *ctx->batch;
    if (eri_threads)
        for (int c = 0; c < 6; ++c) eri_threads[c] = b.eri_threads[c];
    if (scf_threads) *scf_threads = b.scf_threads;
    if (graph_replays) *graph_replays = b.replays;
    if (n_integrals) *n_integrals = b.total_eri;
    return 0;
}

extern "C" int myqc_batch_pair_data(myqc_ctx *ctx, int *npair, float *features, float *targets, float *mask) {
    if (!ctx || !npair) return MYQC_E_ARG;
    if (!ctx->batch || ctx->batch->nmol == 0) return set_error(ctx, MYQC_E_STATE, "myqc_batch_pair_data: no batch set");
    BatchState &b = *ctx->batch;
    if (!b.guess_ok)
        return set_error(ctx, MYQC_E_ARG, "myqc_batch_pair_data: the learned guess covers H..Ne with STO-3G only");
    *npair = b.npair;
    if (!features && !targets && !mask) return 0;
    MYQC_CHECK(guess_export(ctx, b.d_pairrec, b.npair, b.d_atoms, b.d_mol_atoms, b.nmol, b.natom, b.d_D, features, targets, mask));
    if (mask) {
        // pairs of molecules that did not converge carry no target
        std::vector<int> conv(b.nmol);
        MYQC_HIP(ctx, d2h(ctx, conv.data(), b.d_conv, sizeof(int) * b.nmol));
        for (int p = 0; p < b.npair; ++p)
            if (conv[b.pair_mol_of[p]] != 1)
                for (int c = 0; c < kGuessOut; ++c) mask[(size_t)p * kGuessOut + c] = 0.f;
    }
    return 0;
}

extern "C" int myqc_batch_rhf_learned(myqc_ctx *ctx, double e_tol, double d_tol, int max_iter, double *energy,
                                      int *iterations, int *converged, int *fallback) {
    if (!ctx || !energy || e_tol <= 0 || d_tol <= 0 || max_iter < 1) return MYQC_E_ARG;
    if (!ctx->batch || ctx->batch->nmol == 0)
        return set_error(ctx, MYQC_E_STATE, "myqc_batch_rhf_learned: no batch set");
    BatchState &b = *ctx->batch;
    if (!b.guess_ok)
        return set_error(ctx, MYQC_E_ARG, "myqc_batch_rhf_learned: the learned guess covers H..Ne with STO-3G only");
    MYQC_CHECK(guess_reserve(ctx, b.npair, b.natom));
    if (!b.tuned) MYQC_CHECK(batch_tune(ctx, b, false, e_tol, d_tol, max_iter));
    // the learned start gets a shorter budget (typical solves take about 25
    // iterations); a molecule it leaves unconverged restarts from the core
    // guess inside the same persistent launch
    const int learned_iter = std::min(max_iter, 48);
    if (!b.graph_learned || b.gl_etol != e_tol || b.gl_dtol != d_tol || b.gl_maxit != max_iter ||
        b.gl_gen != ctx->mlp_gen) {
        if (b.graph_learned) (void)hipGraphExecDestroy(b.graph_learned);
        b.graph_learned = nullptr;
        hipGraph_t g;
        MYQC_HIP(ctx, hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
        launch_batch_one_e(ctx, b);
        for (int c = 0; c < 6; ++c)
            if (b.nq[c] > 0) launch_batch_eri(ctx, b, c, b.eri_threads[c]);
        guess_launch(ctx, b.d_pairrec, b.npair, b.d_atoms, b.d_mol_atoms, b.nmol, b.natom, b.d_guess);
        launch_batch_scf(ctx, b, true, e_tol, d_tol, max_iter, b.scf_threads, nullptr, -1, true, learned_iter);
        MYQC_HIP(ctx, hipStreamEndCapture(ctx->stream, &g));
        hipError_t e = hipGraphInstantiate(&b.graph_learned, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) {
            b.graph_learned = nullptr;
            return set_error(ctx, MYQC_E_HIP, "myqc_batch_rhf_learned: graph instantiation failed: %s",
                             hipGetErrorString(e));
        }
        b.gl_etol = e_tol;
        b.gl_dtol = d_tol;
        b.gl_maxit = max_iter;
        b.gl_gen = ctx->mlp_gen;
    }
    MYQC_HIP(ctx, hipGraphLaunch(b.graph_learned, ctx->stream));
    ++b.replays;
    MYQC_HIP(ctx, d2h(ctx, energy, b.d_energy, sizeof(double) * b.nmol));
    if (iterations) MYQC_HIP(ctx, d2h(ctx, iterations, b.d_iters, sizeof(int) * b.nmol));
    if (converged) MYQC_HIP(ctx, d2h(ctx, converged, b.d_conv, sizeof(int) * b.nmol));
    if (fallback) MYQC_HIP(ctx, d2h(ctx, fallback, b.d_fail, sizeof(int) * b.nmol));
    return 0;
}
