// eri.hip -- system setup (shells, shell pairs, primitive pairs), Schwarz
// factors, and the contracted shell-quartet ERI kernels.
//
// Work decomposition: one thread per unique contracted shell quartet of one
// angular class; the thread loops over the quartet's primitive quartets (up
// to 3x3x3x3 for STO-3G), builds [e0|f0] by OS vertical recursion in
// registers, contracts, then applies the HGP horizontal recursion.  Unique
// quartets are enumerated implicitly from Schwarz-sorted pair lists, so no
// quartet list is materialised: thread t finds its bra rank by binary search
// over per-bra prefix counts, and its ket rank follows.
//
// Reference: src/integrals/int2e.f90:78-351 (proc2e), :618-726 (clmnew),
// :540-613 (fillsym); src/integrals/auxilary.f90 (Boys, gtoD, getDk).
#include <algorithm>
#include <limits>
#include <cmath>
#include <cstdarg>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <unordered_map>

#include "boys_dev.h"
#include "context.h"
#include "dense.h"
#include "wave.h"
#include "ket_soa.h"
#include "system.h"

namespace myqc {

int set_error(myqc_ctx *ctx, int code, const char *fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (ctx) ctx->err = buf;
    return code;
}

// Device allocations keep their capacity: a buffer is only replaced when a
// request outgrows it, so repeated solves of same-sized systems reuse their
// memory instead of paying hipFree/hipMalloc (and the 1-2 GB integral store)
// every time.  The capacities are kept per address in one process-wide
// registry (contexts may run on several host threads), and dfree drops the
// entry of the buffer it frees, so an address the allocator hands out again
// never inherits a stale size.
namespace {
std::mutex g_cap_mutex;
std::unordered_map<void *, size_t> g_cap;
}  // namespace

static size_t cap_lookup(void *p) {
    std::lock_guard<std::mutex> lk(g_cap_mutex);
    auto it = g_cap.find(p);
    return it == g_cap.end() ? 0 : it->second;
}
static void cap_set(void *p, size_t bytes) {
    std::lock_guard<std::mutex> lk(g_cap_mutex);
    if (bytes) g_cap[p] = bytes;
    else g_cap.erase(p);
}

int dalloc(myqc_ctx *ctx, void **p, size_t bytes) {
    if (*p) {
        if (bytes > 0 && cap_lookup(*p) >= bytes) return 0;
        dfree(p);
    }
    if (bytes == 0) return 0;
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) {
        *p = nullptr;
        return set_error(ctx, MYQC_E_NOMEM, "hipMalloc(%zu bytes) failed: %s", bytes, hipGetErrorString(e));
    }
    cap_set(*p, bytes);
    return 0;
}

size_t dcapacity(const void *p) { return p ? cap_lookup(const_cast<void *>(p)) : 0; }

// Small device-to-host reads (per-iteration scalars, status words) land in
// the context's pinned staging buffer first; larger ones go straight to the
// caller's memory.  Complete at return either way.
hipError_t d2h(myqc_ctx *ctx, void *dst, const void *src, size_t bytes) {
    if (ctx->h_pin && bytes <= kPinBytes) {
        hipError_t e = hipMemcpyAsync(ctx->h_pin, src, bytes, hipMemcpyDeviceToHost, ctx->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
        if (e == hipSuccess) memcpy(dst, ctx->h_pin, bytes);
        return e;
    }
    hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream);
    if (e != hipSuccess) return e;
    return hipStreamSynchronize(ctx->stream);
}

void dfree(void **p) {
    if (*p) {
        cap_set(*p, 0);
        (void)hipFree(*p);
    }
    *p = nullptr;
}

void dtmp_end(myqc_ctx *ctx, int slot) {
    if (dcapacity(ctx->d_tmp[slot]) > kKeepWork) dfree(&ctx->d_tmp[slot]);
}

int timer_begin(myqc_ctx *ctx, int cat, hipEvent_t *ev) {
    *ev = nullptr;
    if (!ctx->timing) return 0;
    MYQC_HIP(ctx, hipEventCreate(ev));
    MYQC_HIP(ctx, hipEventRecord(*ev, ctx->stream));
    return 0;
}

int timer_end(myqc_ctx *ctx, int cat, hipEvent_t ev, double work) {
    if (!ctx->timing || !ev) return 0;
    hipEvent_t b;
    MYQC_HIP(ctx, hipEventCreate(&b));
    MYQC_HIP(ctx, hipEventRecord(b, ctx->stream));
    ctx->events.push_back(EventRec{cat, ev, b, work});
    return 0;
}

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------

template <int C> struct PairL;
template <> struct PairL<0> { static constexpr int a = 0, b = 0; };
template <> struct PairL<1> { static constexpr int a = 1, b = 0; };
template <> struct PairL<2> { static constexpr int a = 1, b = 1; };

struct EriArgs {
    const ShellPair *pairs;
    const PrimPair *prims;
    const double *ksoa;        // ket primitives of the ket class (k_ket_soa)
    long long nket;            // pairs in the ket class
    const double *ftT;
    const int *sorted_b;
    const int *sorted_k;
    const long long *cum;
    int nbra;
    long long nq;
    int same_class;
    // the stored (pre-weighted) block of each quartet
    const long long *segoff;   // [bra pair*3 + ket class]: element e of ket rank r at segoff + r + e*len
    double *x64;
    float *x32;
};

__device__ __forceinline__ void find_quartet(const long long *__restrict__ cum, int nbra, long long t, int same,
                                             int &rb, long long &rk) {
    // last r with cum[r] <= t
    int lo = 0, hi = nbra;   // cum[0] = 0 <= t < cum[nbra]
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (cum[mid] <= t) lo = mid;
        else hi = mid;
    }
    rb = lo;
    rk = t - cum[lo] + (same ? lo : 0);
}

// SPLIT lanes per shell quartet: they share its primitive quartets, add their
// sums (group_sum), and each stores every SPLIT-th element of the block.
// Waves per SIMD asked of the register allocator per class: the staged tables'
// 39 to 41 KB of LDS allow four 256-thread workgroups per CU, so four at most
// (the compiler drops a request that LDS cannot meet): ps|ps and pp|ss 4, the
// rest unconstrained.  ss|ss then has 92 registers and four waves, ps|ss 137 and
// three; ps|ss held to four spills (52 B of scratch): the class in 0.55 instead
// of 0.62 ms at 40 waters, but 54 instead of 51 us at 13.
//
// Bounded by FP64 VALU issue (70 % of it in ss|ss, 64 in ps|ss): about 90 instructions per
// primitive quartet of ss|ss, 30 of the 81 surviving the screen.  40 waters,
// the six classes together: 2.33 ms with every primitive pair tested and the
// reference's downward recursion from F_Q, 2.00 with rows cut at the screen
// (eri_math.h), 1.90 with F_M tabulated, 1.78 with one transcendental less, K/p
// and fewer conversions.  512 threads (eight waves per SIMD on the same
// staged tables): 1.79, and small systems 30 % slower.
constexpr int eri_waves(int cb, int ck) { return cb + ck == 2 ? 4 : 1; }
template <int CB, int CK, int SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(eri_waves(CB, CK)))) void k_eri(EriArgs a) {
    constexpr int M = CB + CK;
    __shared__ __attribute__((aligned(16))) double s_ft[ft_staged(M)];
    const BoysTab ft = stage_boys<M>(a.ftT, s_ft);
    const long long tid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long t = tid / SPLIT;
    const int sub = (int)(tid % SPLIT);
    if (t >= a.nq) return;
    constexpr int LA = PairL<CB>::a, LB = PairL<CB>::b, LC = PairL<CK>::a, LD = PairL<CK>::b;
    constexpr int na = ncart(LA), nb = ncart(LB), nc = ncart(LC), nd = ncart(LD);
    constexpr int BLK = na * nb * nc * nd;
    int rb;
    long long rk;
    find_quartet(a.cum, a.nbra, t, a.same_class, rb, rk);
    const int pb = a.sorted_b[rb], pk = a.sorted_k[rk];
    const ShellPair ket = a.pairs[pk];
    QuartetAcc<LA, LB, LC, LD> acc;
    // A wavefront whose lanes share the bra pair (most do: its lanes take
    // consecutive kets of one bra) reads the bra's pair and primitive data
    // through scalar loads; the classes with few kets per bra, and waves that
    // straddle two bras, load them per lane.
    constexpr bool kUniformPath = CB + CK <= 2;
    const int pb0 = __builtin_amdgcn_readfirstlane(pb);
    ShellPair bra;
    if constexpr (SPLIT > 1) {
        bra = a.pairs[pb];
        quartet_prims_split<LA, LB, LC, LD, SPLIT>(bra, ket, a.prims, KetSoa{a.ksoa, a.nket, rk}, ft, acc, sub);
        using AQ = QuartetAcc<LA, LB, LC, LD>;
#pragma unroll
        for (int e = 0; e < AQ::NE; ++e)
#pragma unroll
            for (int f = 0; f < AQ::NF; ++f) acc.v[e][f] = group_sum<SPLIT>(acc.v[e][f]);
    } else if (kUniformPath && __all(pb == pb0)) {
        bra = a.pairs[pb0];
        quartet_prims_f<LA, LB, LC, LD>(bra, ket, a.prims, KetSoa{a.ksoa, a.nket, rk}, ft, acc);
    } else {
        bra = a.pairs[pb];
        quartet_prims_f<LA, LB, LC, LD>(bra, ket, a.prims, KetSoa{a.ksoa, a.nket, rk}, ft, acc);
    }
    double CD[3] = {ket.AB[0], ket.AB[1], ket.AB[2]};
    double out[BLK];
    quartet_hrr<LA, LB, LC, LD>(acc, bra.AB, CD, out);
    const int same_pair = (pb == pk);
    // one copy under the bra pair, each element times its degeneracy
    // weight (the digestion then applies the same six updates to all);
    // element-major over the bra's kets of this class (len of them)
    const long long base = a.segoff[(long long)pb * 3 + CK] + rk;
    const long long len = a.cum[rb + 1] - a.cum[rb];
#pragma unroll
    for (int ia = 0; ia < na; ++ia)
#pragma unroll
        for (int ib = 0; ib < nb; ++ib)
#pragma unroll
            for (int ic = 0; ic < nc; ++ic)
#pragma unroll
                for (int id = 0; id < nd; ++id) {
                    const int e = ((ia * nb + ib) * nc + ic) * nd + id;
                    if (SPLIT > 1 && e % SPLIT != sub) continue;
                    const double w = block_weight(ia, ib, ic, id, bra.same, ket.same, same_pair, nb, nd,
                                                  bra.ao_a + ia, bra.ao_b + ib, ket.ao_a + ic, ket.ao_b + id);
                    const double v = out[e] * w;
                    a.x64[base + e * len] = v;
                    if (a.x32) a.x32[base + e * len] = (float)v;
                }
}

// Schwarz factors sqrt(max_ab |(ab|ab)|) of the pairs of all three classes,
// kSchwarzLanes lanes per pair sharing its up to 81 primitive quartets.  With
// a lane per pair and a launch per class this was bounded by one lane's
// serial chain (66 + 71 + 94 us for 40 waters, 55 + 55 + 86 for one water);
// eight lanes each and one launch take 34 and 17 us.
constexpr int kSchwarzLanes = 8, kSchwarzPairs = 256 / kSchwarzLanes;

template <int C>
__device__ __forceinline__ void schwarz_pair(const ShellPair *__restrict__ pairs, const PrimPair *__restrict__ prims,
                                             const double *__restrict__ ftT, double *s_ft, int p, bool on, int sub, double *__restrict__ q,
                                             int *__restrict__ rank) {
    constexpr int LA = PairL<C>::a, LB = PairL<C>::b;
    constexpr int na = ncart(LA), nb = ncart(LB);
    const BoysTab ft = stage_boys<2 * C>(ftT, s_ft);
    const ShellPair sp = pairs[p];
    using AQ = QuartetAcc<LA, LB, LA, LB>;
    AQ acc;
    quartet_prims_split<LA, LB, LA, LB, kSchwarzLanes, false>(sp, sp, prims, [&](int j) { return prims[sp.pp0 + j]; },
                                                              ft, acc, sub);
#pragma unroll
    for (int e = 0; e < AQ::NE; ++e)
#pragma unroll
        for (int f = 0; f < AQ::NF; ++f) acc.v[e][f] = group_sum<kSchwarzLanes>(acc.v[e][f]);
    double out[na * nb * na * nb];
    quartet_hrr<LA, LB, LA, LB>(acc, sp.AB, sp.AB, out);
    double m = 0.0;
#pragma unroll
    for (int ia = 0; ia < na; ++ia)
#pragma unroll
        for (int ib = 0; ib < nb; ++ib) m = fmax(m, fabs(out[((ia * nb + ib) * na + ia) * nb + ib]));
    if (on && sub == 0) {
        q[p] = sqrt(m);
        rank[p] = 0;
    }
}

struct SchwarzArgs {
    const int *ids[3];   // pairs of each class
    int np[3];
    int blk[3];          // first workgroup of each class: blk[c] .. (pp pairs, the longest, come first)
};

__global__ __launch_bounds__(256) void k_schwarz(const ShellPair *__restrict__ pairs, const PrimPair *__restrict__ prims,
                                                 const double *__restrict__ ftT, SchwarzArgs a, double *__restrict__ q,
                                                 int *__restrict__ rank) {
    __shared__ __attribute__((aligned(16))) double s_ft[ft_staged(4)];
    const int b = blockIdx.x, c = b >= a.blk[0] ? 0 : b >= a.blk[1] ? 1 : 2;
    // lanes past the last pair repeat it (the group sums need every lane)
    const int t = (b - a.blk[c]) * kSchwarzPairs + threadIdx.x / kSchwarzLanes, sub = threadIdx.x % kSchwarzLanes;
    const bool on = t < a.np[c];
    const int p = a.ids[c][on ? t : a.np[c] - 1];
    if (c == 0) schwarz_pair<0>(pairs, prims, ftT, s_ft, p, on, sub, q, rank);
    else if (c == 1) schwarz_pair<1>(pairs, prims, ftT, s_ft, p, on, sub, q, rank);
    else schwarz_pair<2>(pairs, prims, ftT, s_ft, p, on, sub, q, rank);
}

// The order of each class by Schwarz factor, largest first (ties by position,
// which is by pair id): a pair's rank is the number of pairs before it.  Every
// comparison of a class is made, n^2 of them, a tile of keys in LDS at a time:
// for 12880 pairs that is less than a radix sort's launches take, and the host
// sort it replaces took 0.5 ms with the GPU idle.  The keys are the factors'
// bits (non-negative, so ordered like them; not-a-number has its place too).
// A workgroup takes 256 pairs and every kRankSplit-th tile: more splits spend
// their time in the atomics (50 us with one tile each at 40 waters), fewer leave
// the chip idle (78 us with four times larger tiles).
constexpr int kRankTile = 256, kRankSplit = 16;
__global__ __launch_bounds__(kRankTile) void k_rank(SchwarzArgs a, const double *__restrict__ q,
                                                    int *__restrict__ rank) {
    __shared__ unsigned long long s_key[kRankTile];
    const int b = blockIdx.x, c = b >= a.blk[0] ? 0 : b >= a.blk[1] ? 1 : 2;
    const int np = a.np[c], i0 = (b - a.blk[c]) * kRankTile, i = i0 + threadIdx.x;
    const int p = a.ids[c][min(i, np - 1)];
    const unsigned long long key = __double_as_longlong(q[p]);
    int before = 0;
    for (int j0 = blockIdx.y * kRankTile; j0 < np; j0 += kRankSplit * kRankTile) {
        const int nj = min(kRankTile, np - j0);
        __syncthreads();
        // (past the class: 0, which is before nothing by the strict comparison of a last tile)
        s_key[threadIdx.x] = (int)threadIdx.x < nj ? __double_as_longlong(q[a.ids[c][j0 + threadIdx.x]]) : 0;
        __syncthreads();
        if (j0 < i0) {   // every position of the tile is before the thread's: equal keys are too
#pragma unroll 16
            for (int j = 0; j < kRankTile; ++j) before += s_key[j] >= key ? 1 : 0;
        } else if (j0 > i0) {
#pragma unroll 16
            for (int j = 0; j < kRankTile; ++j) before += s_key[j] > key ? 1 : 0;
        } else {
            for (int j = 0; j < nj; ++j) before += s_key[j] > key || (s_key[j] == key && j0 + j < i) ? 1 : 0;
        }
    }
    if (i < np && before) atomicAdd(&rank[p], before);
}
// sorted (the three classes one after another, as ids)
__global__ __launch_bounds__(256) void k_by_rank(const int *__restrict__ ids, const int *__restrict__ rank, int np0,
                                                 int np1, int np, int *__restrict__ sorted) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= np) return;
    const int first = i < np0 ? 0 : i < np0 + np1 ? np0 : np0 + np1, p = ids[i];
    sorted[first + rank[p]] = p;
}

// The shells as k_prim_pairs reads them: kShellDoubles each
constexpr int kShellPrims = 6, kShellDoubles = 16;   // exponents, coefficients, centre, primitives

// The primitive pairs of every shell pair (fill_prims, system.h), a thread
// each: its place is the number of the pair's primitives with a larger screen
// factor (or an equal one and before it).  The host took 18 ms of core time for
// the 181k of 40 waters and sent 17 MB.
__global__ __launch_bounds__(256) void k_prim_pairs(const ShellPair *__restrict__ pairs, int npairs, int most,
                                                    const double *__restrict__ shells, PrimPair *__restrict__ prims) {
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    if (t >= (long long)npairs * most) return;
    const ShellPair sp = pairs[t / most];
    const int x = (int)(t % most);
    if (x >= sp.npp) return;
    const double *A = shells + kShellDoubles * sp.sa, *B = shells + kShellDoubles * sp.sb;
    const int nb = (int)B[kShellDoubles - 1];
    const double ab2 = sp.AB[0] * sp.AB[0] + sp.AB[1] * sp.AB[1] + sp.AB[2] * sp.AB[2];
    auto screen = [&](int y) {
        const double aa = A[y / nb], bb = B[y % nb];
        return exp(-aa * bb * ab2 / (aa + bb));
    };
    // (not a number: before every number, so that each still has its own place)
    auto key = [](double e) { return e == e ? e : 2.0; };
    const double e = screen(x);
    int place = 0;
    for (int y = 0; y < sp.npp; ++y) {
        const double f = key(screen(y));
        place += f > key(e) || (f == key(e) && y < x) ? 1 : 0;
    }
    PrimPair pp;
    prim_pair(pp, A[x / nb], B[x % nb], A[kShellPrims + x / nb], B[kShellPrims + x % nb], A + 2 * kShellPrims,
              B + 2 * kShellPrims, e);
    prims[sp.pp0 + place] = pp;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

static const int kCB[6] = {0, 1, 1, 2, 2, 2};
static const int kCK[6] = {0, 0, 1, 0, 1, 2};
static const int kBLK[6] = {1, 3, 9, 9, 27, 81};

// Drops the stored integrals; with keep_memory the device buffers stay
// allocated (their capacity is reused by the next build).
void free_eri(myqc_ctx *ctx, bool keep_memory) {
    for (auto &c : ctx->cls) {
        if (!keep_memory) dfree((void **)&c.d_cum);
        c.nq = 0;
    }
    void **ptrs[] = {(void **)&ctx->d_segoff,   (void **)&ctx->d_rank,        (void **)&ctx->d_x64,
                     (void **)&ctx->d_x32,      (void **)&ctx->d_wg,          (void **)&ctx->d_unit,
                     (void **)&ctx->d_unit_off, (void **)&ctx->d_shell,       (void **)&ctx->d_ao_shell,
                     (void **)&ctx->d_partial,  (void **)&ctx->d_Dpair,       (void **)&ctx->d_Dpair32,
                     (void **)&ctx->d_chunk,    (void **)&ctx->d_row_ao,      (void **)&ctx->d_row_list,
                     (void **)&ctx->d_row_list_off, (void **)&ctx->d_jk_list, (void **)&ctx->d_jk_list_off,
                     (void **)&ctx->d_jkoff,    (void **)&ctx->d_jk_part,     (void **)&ctx->d_jk,
                     (void **)&ctx->d_jk_group};
    if (!keep_memory) {
        for (auto p : ptrs) dfree(p);
        for (int c = 0; c < 3; ++c) dfree((void **)&ctx->d_meta[c]);
        for (int c = 0; c < 3; ++c) dfree((void **)&ctx->d_qrank[c]);
    }
    ctx->n_wg = 0;
    ctx->have_eri = false;
    ctx->have_eri32 = false;
}

int eri_schwarz(myqc_ctx *ctx) {
    if (ctx->have_schwarz) return 0;
    const int np = (int)ctx->pairs.size();
    for (const ShellPair &sp : ctx->pairs)
        if (sp.npp > kKetPrims)
            return set_error(ctx, MYQC_E_ARG, "a shell pair has %d primitive pairs (at most %d: STO-3G shells)",
                             sp.npp, kKetPrims);
    // one allocation: the factors and the sorted pairs (which the host takes
    // together), then ranks and the pairs by class
    const size_t back = (sizeof(double) + sizeof(int)) * (size_t)np;
    MYQC_CHECK(dalloc(ctx, (void **)&ctx->d_schwarz, back + 2 * sizeof(int) * (size_t)np));
    int *sorted = reinterpret_cast<int *>(ctx->d_schwarz + np), *rank = sorted + np, *ids = rank + np;
    std::vector<int> all;
    all.reserve(np);
    SchwarzArgs sa{}, ra{};
    int nblk = 0, nrank = 0, most = 0;
    for (int c = 0; c < 3; ++c) {
        ctx->d_sorted[c] = sorted + all.size();
        sa.ids[c] = ra.ids[c] = ids + all.size();
        sa.np[c] = ra.np[c] = (int)ctx->pair_ids[c].size();
        most = std::max(most, sa.np[c]);
        all.insert(all.end(), ctx->pair_ids[c].begin(), ctx->pair_ids[c].end());
    }
    for (int c = 2; c >= 0; --c) {
        sa.blk[c] = nblk;
        ra.blk[c] = nrank;
        nblk += (sa.np[c] + kSchwarzPairs - 1) / kSchwarzPairs;
        nrank += (sa.np[c] + kRankTile - 1) / kRankTile;
    }
    MYQC_HIP(ctx, hipMemcpyAsync(ids, all.data(), sizeof(int) * np, hipMemcpyHostToDevice, ctx->stream));
    k_schwarz<<<nblk, 256, 0, ctx->stream>>>(ctx->d_pairs, ctx->d_prims, ctx->d_ftT, sa, ctx->d_schwarz, rank);
    k_rank<<<dim3(nrank, std::min(kRankSplit, (most + kRankTile - 1) / kRankTile)), kRankTile, 0, ctx->stream>>>(ra, ctx->d_schwarz, rank);
    k_by_rank<<<(np + 255) / 256, 256, 0, ctx->stream>>>(ids, rank, sa.np[0], sa.np[1], np, sorted);
    for (int c = 0; c < 3; ++c) {
        if (sa.np[c] == 0) continue;
        MYQC_CHECK(dalloc(ctx, (void **)&ctx->d_ksoa[c], sizeof(double) * kKetPrims * kKetFields * (size_t)sa.np[c]));
        k_ket_soa<<<dim3((sa.np[c] + 255) / 256, kKetPrims), 256, 0, ctx->stream>>>(
            ctx->d_pairs, ctx->d_prims, ctx->d_sorted[c], sa.np[c], ctx->d_ksoa[c]);
    }
    MYQC_HIP(ctx, hipGetLastError());
    std::vector<double> host((back + sizeof(double) - 1) / sizeof(double));
    MYQC_HIP(ctx, hipMemcpyAsync(host.data(), ctx->d_schwarz, back, hipMemcpyDeviceToHost, ctx->stream));
    MYQC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    ctx->schwarz.assign(host.begin(), host.begin() + np);
    const int *order = reinterpret_cast<const int *>(host.data() + np);
    for (int c = 0; c < 3; ++c) {
        ctx->pair_ids[c].assign(order, order + sa.np[c]);
        order += sa.np[c];
    }
    ctx->have_schwarz = true;
    return 0;
}

// Per-bra counts of surviving kets and their prefix sums for class (cb, ck).
static void class_counts(myqc_ctx *ctx, int cb, int ck, double tol, std::vector<long long> &cum) {
    const auto &B = ctx->pair_ids[cb];
    const auto &K = ctx->pair_ids[ck];
    cum.assign(B.size() + 1, 0);
    std::vector<double> qk(K.size());
    for (size_t i = 0; i < K.size(); ++i) qk[i] = ctx->schwarz[K[i]];
    // bras in descending Schwarz order need ascending thresholds: the number
    // of kets with qk >= tol / qb only shrinks, so one pointer walks down
    size_t ptr = qk.size();
    for (size_t r = 0; r < B.size(); ++r) {
        const double qb = ctx->schwarz[B[r]];
        long long ub;
        if (tol <= 0.0) ub = (long long)K.size();
        else if (qb <= 0.0) ub = 0;
        else {
            const double need = tol / qb;
            while (ptr > 0 && !(qk[ptr - 1] >= need)) --ptr;
            ub = (long long)ptr;
        }
        long long cnt = (cb == ck) ? std::max(0LL, ub - (long long)r) : ub;
        cum[r + 1] = cum[r] + cnt;
    }
}

// Launch shape of each quartet class in the stored build: lanes per shell
// quartet (1, 2, 4, 8) and threads per workgroup (64, 128, 256).  The lanes
// follow the class's size, unless myqc_eri_set_shapes gives a shape or
// myqc_eri_tune has measured the candidates: what it kept holds for classes of
// half to twice the quartets it was measured at, the step of lanes of the
// rule.  (Kept for every size, the shapes tuned at 40 waters took 0.31 ms for
// a build of one water and 0.39 for 8, against 0.25 and 0.30 by the rule.)
struct EriShape {
    int split = 0, tpb = 256;   // split 0: by the rule
    long long nq = 0;           // quartets it was tuned at; 0: for every size
};
static std::mutex g_shape_mu;
static EriShape g_shape[6];

// A class with few quartets is bounded by one lane's chain of up to 81
// primitive quartets, not by throughput, so its quartets are spread over as
// many lanes as keep it under 2^18 lanes (a full chip of four wavefronts per
// SIMD): one water's build took 387 us with a lane per quartet, 102 us with
// eight; eight waters 393 -> 157.  The best of 1, 2, 4, 8 lanes as measured:
// ss|ss 16k quartets 8, 72k 4, 140k 2, 358k 1; ps|ps 33k 8, 77k 2, 222k 1;
// pp|ss 19k 8, 47k 4, 125k 2, 340k 1; pp|ps 22k 8, 62k 4, 154k 1.  pp|pp, whose
// lane holds the most registers, gains from eight lanes only below 8k
// quartets (4.6k 8, 10k 4), and one lane of it never pays (20k quartets: 213
// us with one lane, 81 with four).
static int rule_split(int c, long long nq) {
    if (c == 5) return nq <= (1 << 13) ? 8 : 4;
    int s = 8;
    while (s > 1 && nq * s > (1 << 18)) s >>= 1;
    return s;
}

static EriShape class_shape(int c, long long nq, bool given) {
    EriShape sh;
    if (given) {
        std::lock_guard<std::mutex> g(g_shape_mu);
        sh = g_shape[c];
    }
    if (sh.nq > 0 && (nq > 2 * sh.nq || 2 * nq < sh.nq)) sh = EriShape{};
    if (sh.split == 0) sh.split = rule_split(c, nq);
    return sh;
}

template <int CB, int CK>
static void launch_eri(myqc_ctx *ctx, const QuartetClass &qc, hipStream_t s, EriShape sh) {
    EriArgs a;
    a.pairs = ctx->d_pairs;
    a.prims = ctx->d_prims;
    a.ftT = ctx->d_ftT;
    a.sorted_b = ctx->d_sorted[CB];
    a.sorted_k = ctx->d_sorted[CK];
    a.ksoa = ctx->d_ksoa[CK];
    a.nket = (long long)ctx->pair_ids[CK].size();
    a.cum = qc.d_cum;
    a.nbra = qc.nbra;
    a.nq = qc.nq;
    a.same_class = (CB == CK);
    a.segoff = ctx->d_segoff;
    a.x64 = ctx->d_x64;
    a.x32 = ctx->d_x32;
    const long long nblk = (qc.nq * sh.split + sh.tpb - 1) / sh.tpb;
    switch (sh.split) {
        case 2: k_eri<CB, CK, 2><<<(unsigned)nblk, sh.tpb, 0, s>>>(a); break;
        case 4: k_eri<CB, CK, 4><<<(unsigned)nblk, sh.tpb, 0, s>>>(a); break;
        case 8: k_eri<CB, CK, 8><<<(unsigned)nblk, sh.tpb, 0, s>>>(a); break;
        default: k_eri<CB, CK, 1><<<(unsigned)nblk, sh.tpb, 0, s>>>(a); break;
    }
}

static void launch_class(myqc_ctx *ctx, int c, hipStream_t s, EriShape sh) {
    const QuartetClass &qc = ctx->cls[c];
    if (qc.nq == 0) return;
    switch (c) {
        case 0: launch_eri<0, 0>(ctx, qc, s, sh); break;
        case 1: launch_eri<1, 0>(ctx, qc, s, sh); break;
        case 2: launch_eri<1, 1>(ctx, qc, s, sh); break;
        case 3: launch_eri<2, 0>(ctx, qc, s, sh); break;
        case 4: launch_eri<2, 1>(ctx, qc, s, sh); break;
        case 5: launch_eri<2, 2>(ctx, qc, s, sh); break;
    }
}

// FP64 operations per contracted shell quartet of each class (FMA = 2,
// transcendental = 1), for the roofline's flops: the FP64 VALU instruction
// counters (ADD, MUL, FMA, TRANS _F64, each x 64 lanes) of one build of the
// 40-water STO-3G cluster at Schwarz 1e-12, divided by the class's quartet
// count.  They include lanes that sit idle while a neighbour computes a
// primitive quartet that its own pair screen drops, and both sides of a
// divergent Boys branch, so they count issued rather than strictly useful work.
static const double kQuartetFlops[6] = {2297.3, 2893.7, 4533.7, 4648.9, 9444.8, 30695.8};

static int build_classes(myqc_ctx *ctx, double tol) {
    std::vector<long long> cum;
    ctx->n_quartets = 0;
    ctx->n_stored = 0;
    ctx->eri_flops = 0.0;
    for (int c = 0; c < 6; ++c) {
        QuartetClass &qc = ctx->cls[c];
        qc.cb = kCB[c];
        qc.ck = kCK[c];
        qc.blk = kBLK[c];
        qc.nbra = (int)ctx->pair_ids[qc.cb].size();
        if (qc.nbra == 0 || ctx->pair_ids[qc.ck].empty()) {
            qc.nq = 0;
            continue;
        }
        class_counts(ctx, qc.cb, qc.ck, tol, cum);
        qc.nq = cum.back();
        MYQC_CHECK(dalloc(ctx, (void **)&qc.d_cum, sizeof(long long) * cum.size()));
        MYQC_HIP(ctx, hipMemcpyAsync(qc.d_cum, cum.data(), sizeof(long long) * cum.size(), hipMemcpyHostToDevice,
                                     ctx->stream));
        ctx->n_quartets += qc.nq;
        ctx->n_stored += qc.nq * qc.blk;
        ctx->eri_flops += (double)qc.nq * kQuartetFlops[c];
        if (getenv("MYQC_HOST_TIMING"))
            fprintf(stderr, "[host] eri class (%d,%d): %lld quartets, %.6e flops by the table\n", qc.cb, qc.ck, qc.nq,
                    (double)qc.nq * kQuartetFlops[c]);
    }
    MYQC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return 0;
}

// copies a host vector to a device buffer kept by the context
template <typename T>
static int upload(myqc_ctx *ctx, T **dst, const std::vector<T> &src) {
    MYQC_CHECK(dalloc(ctx, (void **)dst, sizeof(T) * std::max<size_t>(src.size(), 1)));
    if (!src.empty())
        MYQC_HIP(ctx, hipMemcpyAsync(*dst, src.data(), sizeof(T) * src.size(), hipMemcpyHostToDevice, ctx->stream));
    return 0;
}

// LDS the digestion kernel may use per workgroup: three workgroups per CU
constexpr size_t kDigestLds = 52 * 1024;

// The layout of the stored integrals (digest_plan.h): each screened unique
// quartet's block offset under its bra pair.  The ERI kernels need only this.
static int build_layout(myqc_ctx *ctx, double tol) {
    const int ns = (int)ctx->shells.size();
    ctx->ns = ns;
    std::vector<int> sao(ns);
    for (int X = 0; X < ns; ++X) sao[X] = ctx->shells[X].ao;
    const std::string e = build_digest_layout(ctx->plan, ctx->n, sao, ctx->pairs, ctx->pair_ids, ctx->schwarz, tol);
    if (!e.empty()) return set_error(ctx, MYQC_E_ARG, "%s", e.c_str());
    if (ctx->plan.n_values != ctx->n_stored || ctx->plan.n_quartets != ctx->n_quartets)
        return set_error(ctx, MYQC_E_STATE, "integral layout (%lld values) disagrees with the quartet classes (%lld)",
                         ctx->plan.n_values, ctx->n_stored);
    MYQC_CHECK(upload(ctx, &ctx->d_segoff, ctx->plan.off));
    MYQC_CHECK(upload(ctx, &ctx->d_rank, ctx->plan.rank));
    MYQC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return 0;
}

// The digestion schedule over the layout, built on the host while the ERI
// kernels that fill the store run, and its device copies.
static int build_schedule(myqc_ctx *ctx) {
    const int ns = ctx->ns, n = ctx->n;
    std::vector<int> sao(ns), sL(ns);
    for (int X = 0; X < ns; ++X) {
        sao[X] = ctx->shells[X].ao;
        sL[X] = ctx->shells[X].L;
    }
    // Rows and values per workgroup.  LDS holds the G rows (FP64) and the D
    // rows (FP64 for the plain pass), which bounds the rows; a system small
    // enough to leave the chip short of workgroups takes fewer rows (down to
    // one pair of p shells), and its values are cut into about 600 runs of at
    // least 8k values, where a pass is bounded by its longest wavefronts'
    // chains of row loads: measured (FP64 kernel, waters, with rows / values):
    // 8: 131 us (58 rows, 64k) -> 24 us (6, 8k); 13: 104 -> 30; 24: 94 -> 69.
    // A large one is bounded by traffic: fewer rows mean more partial rows to
    // write and gather (40 waters: 171 us with 11 rows, 174 with 8, 189 with
    // 6; 183 with 128k values each, 185 with 32k).  In between, 28 waters: 95
    // us with 8 rows, 102 with 6, 105 with 11 of 64k.
    const long long stored = ctx->n_stored;
    const int lds_rows = (int)(kDigestLds / (2 * sizeof(double) * (size_t)n));
    const int max_rows = std::min(lds_rows, stored < 12000000 ? 6 : stored < 32000000 ? 8 : 64);
    const long long target = std::min(1LL << 16, std::max(1LL << 13, stored / 600));
    if (max_rows < 6)
        return set_error(ctx, MYQC_E_ARG, "digestion: n=%d leaves fewer than 6 rows of G and D in %zu bytes of LDS", n,
                         kDigestLds);
    DigestPlan &pl = ctx->plan;
    const std::string e =
        build_digest_schedule(pl, sao, sL, ctx->pairs, ctx->pair_ids, ctx->schwarz, max_rows, target);
    if (!e.empty()) return set_error(ctx, MYQC_E_ARG, "%s", e.c_str());
    ctx->n_wg = (int)(pl.wg.size() / kWgInts);
    MYQC_CHECK(upload(ctx, &ctx->d_wg, pl.wg));
    MYQC_CHECK(upload(ctx, &ctx->d_unit, pl.unit));
    MYQC_CHECK(upload(ctx, &ctx->d_unit_off, pl.unit_off));
    MYQC_CHECK(upload(ctx, &ctx->d_chunk, pl.chunk));
    MYQC_CHECK(upload(ctx, &ctx->d_row_ao, pl.row_ao));
    MYQC_CHECK(upload(ctx, &ctx->d_row_list, pl.row_list));
    MYQC_CHECK(upload(ctx, &ctx->d_row_list_off, pl.row_list_off));
    MYQC_CHECK(upload(ctx, &ctx->d_jk_list, pl.jk_list));
    MYQC_CHECK(upload(ctx, &ctx->d_jk_list_off, pl.jk_list_off));
    MYQC_CHECK(upload(ctx, &ctx->d_jk_group, pl.jk_group));
    MYQC_CHECK(upload(ctx, &ctx->d_jkoff, pl.jkoff));
    MYQC_CHECK(dalloc(ctx, (void **)&ctx->d_jk_part, sizeof(double) * kJkSlot * std::max<size_t>(pl.n_jk_slots, 1)));
    MYQC_CHECK(dalloc(ctx, (void **)&ctx->d_jk, sizeof(double) * std::max(pl.jk_base[3], 1)));
    MYQC_CHECK(dalloc(ctx, (void **)&ctx->d_partial, sizeof(double) * (size_t)std::max(pl.n_rows, 1) * n));
    // ket metadata and Schwarz factors in rank order per class
    for (int c = 0; c < 3; ++c) {
        const auto &ids = ctx->pair_ids[c];
        if (ids.empty()) continue;
        std::vector<int> meta(ids.size());
        std::vector<float> qrank(ids.size());
        for (size_t r = 0; r < ids.size(); ++r) {
            const ShellPair &sp = ctx->pairs[ids[r]];
            meta[r] = sp.ao_a | (sp.ao_b << 15);
            // rounded up, so that the screen never drops a ket the exact factor keeps
            qrank[r] = std::nextafter((float)ctx->schwarz[ids[r]], std::numeric_limits<float>::infinity());
        }
        MYQC_CHECK(upload(ctx, &ctx->d_meta[c], meta));
        MYQC_CHECK(upload(ctx, &ctx->d_qrank[c], qrank));
    }
    std::vector<int> shell(4 * ns, 0), ao_shell(n);
    for (int X = 0; X < ns; ++X) {
        shell[4 * X] = ctx->shells[X].ao;
        shell[4 * X + 1] = ctx->shells[X].L;
        for (int k = 0; k < (ctx->shells[X].L ? 3 : 1); ++k) ao_shell[ctx->shells[X].ao + k] = X;
    }
    MYQC_CHECK(upload(ctx, &ctx->d_shell, shell));
    MYQC_CHECK(upload(ctx, &ctx->d_ao_shell, ao_shell));
    MYQC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return 0;
}

// the side streams and fork/join events, created on first use
static int ensure_side_streams(myqc_ctx *ctx) {
    if (ctx->fork_ev) return 0;
    for (int k = 0; k < 2; ++k) {
        MYQC_HIP(ctx, hipStreamCreateWithFlags(&ctx->side[k], hipStreamNonBlocking));
        MYQC_HIP(ctx, hipEventCreateWithFlags(&ctx->join_ev[k], hipEventDisableTiming));
    }
    MYQC_HIP(ctx, hipEventCreateWithFlags(&ctx->fork_ev, hipEventDisableTiming));
    return 0;
}

// The values of every screened quartet at threshold tol, and their layout:
// all of the stored build but the digestion schedule.  Leaves the kernels
// in flight on the context stream.  given_shapes: the shapes tuned or set for
// stored builds; without, the rule's alone, so that dense results do not
// depend on what the process has tuned (a stored build serves them only if its
// shapes were the rule's, DenseSource::open).
int eri_values(myqc_ctx *ctx, double tol, bool want32, bool given_shapes) {
    HostClock hc(ctx);
    MYQC_CHECK(eri_schwarz(ctx));
    hc.mark("eri_store: Schwarz factors");
    MYQC_CHECK(build_classes(ctx, tol));
    hc.mark("eri_store: quartet classes");
    MYQC_CHECK(build_layout(ctx, tol));
    hc.mark("eri_store: layout");
    const size_t nx = (size_t)std::max<long long>(ctx->n_stored, 1);
    MYQC_CHECK(dalloc(ctx, (void **)&ctx->d_x64, sizeof(double) * nx));
    if (want32) MYQC_CHECK(dalloc(ctx, (void **)&ctx->d_x32, sizeof(float) * nx));
    else dfree((void **)&ctx->d_x32);   // a kept buffer may be smaller than this build
    MYQC_CHECK(ensure_side_streams(ctx));
    hipEvent_t ev;
    MYQC_CHECK(timer_begin(ctx, T_ERI, &ev));
    // the classes write disjoint blocks of the store, so they may overlap:
    // the L-bra classes (few waves, long ones) start first on side stream 0,
    // (Ls|Ls) on side stream 1, the two large s-ket classes on the context
    // stream; the context stream then waits for both side streams
    MYQC_HIP(ctx, hipEventRecord(ctx->fork_ev, ctx->stream));
    for (int k = 0; k < 2; ++k) MYQC_HIP(ctx, hipStreamWaitEvent(ctx->side[k], ctx->fork_ev, 0));
    static const int kOrder[6] = {5, 4, 3, 2, 0, 1};
    ctx->eri_by_rule = true;
    for (int c : kOrder) {
        if (ctx->cls[c].nq == 0) continue;
        const EriShape sh = class_shape(c, ctx->cls[c].nq, given_shapes), rule = class_shape(c, ctx->cls[c].nq, false);
        if (sh.split != rule.split || sh.tpb != rule.tpb) ctx->eri_by_rule = false;
        launch_class(ctx, c, c >= 3 ? ctx->side[0] : c == 2 ? ctx->side[1] : ctx->stream, sh);
        MYQC_HIP(ctx, hipGetLastError());
    }
    for (int k = 0; k < 2; ++k) {
        MYQC_HIP(ctx, hipEventRecord(ctx->join_ev[k], ctx->side[k]));
        MYQC_HIP(ctx, hipStreamWaitEvent(ctx->stream, ctx->join_ev[k], 0));
    }
    MYQC_CHECK(timer_end(ctx, T_ERI, ev, ctx->eri_flops));
    hc.mark("eri_store: allocations and launches");
    return 0;
}

int eri_store(myqc_ctx *ctx, double tol, bool want32) {
    HostClock hc(ctx);
    free_eri(ctx, true);
    MYQC_CHECK(eri_values(ctx, tol, want32, true));
    MYQC_CHECK(dalloc(ctx, (void **)&ctx->d_Dpair, sizeof(double) * 9 * ctx->pairs.size()));
    MYQC_CHECK(dalloc(ctx, (void **)&ctx->d_Dpair32, sizeof(float) * 9 * ctx->pairs.size()));
    hc.mark("eri_store: values");
    // the digestion schedule is built while the kernels run
    MYQC_CHECK(build_schedule(ctx));
    hc.mark("eri_store: schedule (host, beside the kernels)");
    MYQC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    hc.mark("eri_store: kernels");
    ctx->have_eri = true;
    ctx->have_eri32 = want32;
    ctx->eri_tol = tol;
    return 0;
}

// The launch-shape search of the stored build: every (lanes per quartet,
// threads per workgroup) candidate of every class with quartets in the
// current system is timed on the context stream (the fastest of `reps`
// launches; each launch rewrites the same values into the store), and the
// fastest shape of each class is kept for the process's builds of that size.
static const int kSplits[4] = {1, 2, 4, 8}, kTpbs[3] = {64, 128, 256};

int eri_tune(myqc_ctx *ctx, int reps, int *shape_out, double *ms_out) {
    if (!ctx->have_eri) return set_error(ctx, MYQC_E_STATE, "myqc_eri_tune: call myqc_eri_build first");
    if (reps < 1 || reps > 100) return set_error(ctx, MYQC_E_ARG, "myqc_eri_tune: reps=%d (1..100)", reps);
    hipEvent_t e0, e1;
    MYQC_HIP(ctx, hipEventCreate(&e0));
    MYQC_HIP(ctx, hipEventCreate(&e1));
    int rc = 0;
    ctx->eri_by_rule = false;   // the store ends with the last candidates' values
    EriShape best[6];
    double best_ms[6];
    for (int c = 0; c < 6 && rc == 0; ++c) {
        best[c] = class_shape(c, ctx->cls[c].nq, true);
        best_ms[c] = 0.0;
        if (ctx->cls[c].nq == 0) continue;
        best_ms[c] = 1e300;
        for (int sp : kSplits)
            for (int tpb : kTpbs) {
                const EriShape sh{sp, tpb, ctx->cls[c].nq};
                double t = 1e300;
                for (int r = 0; r < reps && rc == 0; ++r) {
                    float ms = 0.0f;
                    if (hipEventRecord(e0, ctx->stream) != hipSuccess) rc = set_error(ctx, MYQC_E_HIP, "event");
                    launch_class(ctx, c, ctx->stream, sh);
                    if (!rc && (hipGetLastError() != hipSuccess || hipEventRecord(e1, ctx->stream) != hipSuccess ||
                                hipEventSynchronize(e1) != hipSuccess || hipEventElapsedTime(&ms, e0, e1) != hipSuccess))
                        rc = set_error(ctx, MYQC_E_HIP, "myqc_eri_tune: class %d launch failed", c);
                    t = std::min(t, (double)ms);
                }
                if (t < best_ms[c]) {
                    best_ms[c] = t;
                    best[c] = sh;
                }
            }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc) return rc;
    {
        std::lock_guard<std::mutex> g(g_shape_mu);
        for (int c = 0; c < 6; ++c)
            if (ctx->cls[c].nq > 0) g_shape[c] = best[c];
    }
    for (int c = 0; c < 6; ++c) {
        if (shape_out) {
            shape_out[2 * c] = best[c].split;
            shape_out[2 * c + 1] = best[c].tpb;
        }
        if (ms_out) ms_out[c] = best_ms[c];
    }
    return 0;
}

// sets the launch shapes directly, for every size of a class (a shape of 0
// lanes keeps that class's, one of -1 goes back to the rule)
int eri_set_shapes(myqc_ctx *ctx, const int *shape) {
    for (int c = 0; c < 6; ++c) {
        const int sp = shape[2 * c], tpb = shape[2 * c + 1];
        if (sp == 0 || sp == -1) continue;
        if ((sp != 1 && sp != 2 && sp != 4 && sp != 8) || (tpb != 64 && tpb != 128 && tpb != 256))
            return set_error(ctx, MYQC_E_ARG, "myqc_eri_set_shapes: class %d: %d lanes, %d threads", c, sp, tpb);
    }
    std::lock_guard<std::mutex> g(g_shape_mu);
    for (int c = 0; c < 6; ++c)
        if (shape[2 * c] == -1) g_shape[c] = EriShape{};
        else if (shape[2 * c] != 0) g_shape[c] = EriShape{shape[2 * c], shape[2 * c + 1]};
    return 0;
}

}  // namespace myqc

using namespace myqc;

extern "C" int myqc_set_system(myqc_ctx *ctx, int nnuc, const int *Z, const double *xyz_bohr, int nset,
                               const double *set_alpha, const int *setinfo, const double *bas, int norb,
                               const int *basinfo, const double *Ftab, int flags) {
    if (!ctx) return MYQC_E_ARG;
    if (nnuc <= 0 || nset <= 0 || norb <= 0 || !Z || !xyz_bohr || !set_alpha || !setinfo || !bas || !basinfo || !Ftab)
        return set_error(ctx, MYQC_E_ARG, "myqc_set_system: invalid arguments");
    if (flags != MYQC_REF_COMPAT) return set_error(ctx, MYQC_E_ARG, "myqc_set_system: unknown flags %d", flags);
    HostClock hc(ctx);
    free_eri(ctx, true);
    ctx->have_system = false;
    ctx->have_schwarz = false;
    ctx->n = norb;
    ctx->nnuc = nnuc;
    ctx->Z.assign(Z, Z + nnuc);
    ctx->xyz.resize(3 * nnuc);
    for (int a = 0; a < nnuc; ++a)
        for (int c = 0; c < 3; ++c) ctx->xyz[3 * a + c] = xyz_bohr[a + nnuc * c];
    size_t nprims = 0;
    const std::string why = build_pairs(nnuc, nset, set_alpha, setinfo, bas, norb, basinfo, ctx->xyz.data(),
                                        ctx->shells, ctx->pairs, nprims, ctx->pair_ids);
    if (!why.empty()) return set_error(ctx, MYQC_E_ARG, "myqc_set_system: %s", why.c_str());
    hc.mark("set_system: shells and pairs");
    const int np = (int)ctx->pairs.size();
    int most = 0;
    std::vector<double> sh(kShellDoubles * ctx->shells.size(), 0.0);
    for (size_t k = 0; k < ctx->shells.size(); ++k) {
        const Shell &x = ctx->shells[k];
        double *d = sh.data() + kShellDoubles * k;
        std::copy(x.alpha.begin(), x.alpha.end(), d);
        std::copy(x.coef.begin(), x.coef.end(), d + kShellPrims);
        std::copy(&ctx->xyz[3 * x.center], &ctx->xyz[3 * x.center] + 3, d + 2 * kShellPrims);
        d[kShellDoubles - 1] = (double)x.alpha.size();
        most = std::max(most, (int)(x.alpha.size() * x.alpha.size()));
    }
    ctx->ftT.resize(FT_TOTAL - FT_EG);
    boys_inputs(Ftab, ctx->ftT.data());
    double *d_sh = nullptr;
    MYQC_CHECK(dalloc(ctx, (void **)&ctx->d_pairs, sizeof(ShellPair) * np));
    MYQC_CHECK(dalloc(ctx, (void **)&ctx->d_prims, sizeof(PrimPair) * nprims));
    MYQC_CHECK(dalloc(ctx, (void **)&ctx->d_ftT, sizeof(double) * FT_TOTAL));
    MYQC_CHECK(dtmp(ctx, TMP_SHELLS, &d_sh, sizeof(double) * sh.size()));
    MYQC_HIP(ctx, hipMemcpyAsync(ctx->d_pairs, ctx->pairs.data(), sizeof(ShellPair) * np, hipMemcpyHostToDevice,
                                 ctx->stream));
    MYQC_HIP(ctx, hipMemcpyAsync(d_sh, sh.data(), sizeof(double) * sh.size(), hipMemcpyHostToDevice, ctx->stream));
    k_prim_pairs<<<(unsigned)(((long long)np * most + 255) / 256), 256, 0, ctx->stream>>>(ctx->d_pairs, np, most, d_sh,
                                                                                         ctx->d_prims);
    MYQC_HIP(ctx, hipMemcpyAsync(ctx->d_ftT + FT_EG, ctx->ftT.data(), sizeof(double) * ctx->ftT.size(),
                                 hipMemcpyHostToDevice, ctx->stream));
    k_boys_rows<<<kBoysRowBlocks, 64, 0, ctx->stream>>>(ctx->d_ftT);
    MYQC_HIP(ctx, hipGetLastError());
    MYQC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    hc.mark("set_system: uploads");
    ctx->have_system = true;
    ctx->work_n = -1;
    return 0;
}

extern "C" int myqc_eri_full(myqc_ctx *ctx, double schwarz_tol, double *XX) {
    if (!ctx || !XX) return MYQC_E_ARG;
    if (!ctx->have_system) return set_error(ctx, MYQC_E_STATE, "myqc_eri_full: no system set");
    // through the context's work buffer, a slab of the last index at a time where
    // the array is too large to keep: beside the stored integrals (an eighth of
    // it) the device need not hold the array
    const size_t n = ctx->n, n3 = n * n * n, col = sizeof(double) * n3;
    const int per = (int)std::min(n, std::max<size_t>(1, kKeepWork / col));
    DenseSource src(ctx);
    int rc = dalloc(ctx, (void **)&ctx->d_xwork, col * per);
    if (rc == 0) rc = src.open(schwarz_tol);
    for (int d0 = 0; d0 < ctx->n && rc == 0; d0 += per) {
        const int d1 = std::min(ctx->n, d0 + per);
        rc = src.expand_full(ctx->d_xwork, d0, d1);
        if (rc) break;
        const hipError_t e = d2h(ctx, XX + n3 * d0, ctx->d_xwork, col * (d1 - d0));
        if (e != hipSuccess) rc = set_error(ctx, MYQC_E_HIP, "myqc_eri_full: copy failed: %s", hipGetErrorString(e));
    }
    if (rc) (void)hipStreamSynchronize(ctx->stream);   // nothing in flight when the store is given back
    if (dcapacity(ctx->d_xwork) > kKeepWork) dfree((void **)&ctx->d_xwork);
    return rc;
}

extern "C" int myqc_eri_build(myqc_ctx *ctx, double schwarz_tol, long long *n_stored) {
    if (!ctx) return MYQC_E_ARG;
    if (!ctx->have_system) return set_error(ctx, MYQC_E_STATE, "myqc_eri_build: no system set");
    if (schwarz_tol < 0) return set_error(ctx, MYQC_E_ARG, "myqc_eri_build: negative tolerance");
    MYQC_CHECK(eri_store(ctx, schwarz_tol, true));
    if (n_stored) *n_stored = ctx->n_stored;
    return 0;
}

extern "C" int myqc_eri_tune(myqc_ctx *ctx, int reps, int *shapes, double *ms) {
    if (!ctx) return MYQC_E_ARG;
    return eri_tune(ctx, reps, shapes, ms);
}

extern "C" int myqc_eri_set_shapes(myqc_ctx *ctx, const int *shapes) {
    if (!ctx || !shapes) return MYQC_E_ARG;
    return eri_set_shapes(ctx, shapes);
}
