// dense.hip -- dense AO integrals from the stored ones (dense.h), for the int2e
// record and the four-index transforms.
//
// The integrals are computed once into the element-major store, where every
// write of a wavefront is contiguous, and expanded from there: writing each
// value to its eight places of the dense array straight from the integral
// kernels makes eight stores of 8 bytes to as many cache lines (24 waters: 20
// ms for the classes against 2 ms into the store).  The transforms take
// the blocks of l >= d only, a buffer's worth at a time, so that a block is
// still in cache when it is contracted and no n^4 array is held.
#include <cstring>

#include "dense.h"

namespace myqc {

// values of a block in LDS: small blocks, and a range of u of large ones
constexpr int kExpSmall = 2048, kExpLarge = 16384;
constexpr int kExpParts = 64;   // ranges of u at most (n <= 1425: a range ends with a whole row)
struct ExpandArgs {
    const double *x;
    const int *inv;            // per class-sorted pair and element: 2 (u (u + 1) / 2 + v) + (u == v), -1: not kept
    const long long *off;      // [ket class][pos]: value offset (element e of ket rank r at off + r + e len)
    const int *range;          // [ket class][pos]: its ket ranks {lo, hi}
    const ExpandRec *rec;
    double *X;
    int n, nrec;
    int pos[4];                // first position of each class, and the end
    int inv0[3];               // first entry of inv of each class
    int d0, d1;                // blocks (l, d) and (d, l) at l + n (d - d0) and d + n (l - d0) as far as the second
                               // index is within [d0, d1); d1 = 0: the record's block alone, at rec.blk
    int m[kExpParts + 1];      // the ranges of u (blockIdx.y)
};

// wave-uniform read-only records through scalar loads
template <typename T>
using cptr = const __attribute__((address_space(4))) T *;

// The block of one function pair (l, d), element ep of shell pair P, over the
// u >= v with u in [m0, m1), assembled in LDS and written out as the square.
//
// Its values lie in two places: where P is the bra, P's own rows of the
// store, read along the ket ranks (contiguous); where Q is the bra, one value
// per (Q, element), at P's rank.  Those single values share their cache lines
// with the pairs of neighbouring rank, so 32 consecutive pairs (same element)
// run on one XCD at a time (workgroup b runs on XCD b mod 8), in step, and a
// line is fetched from memory once for 16 of them.  The scatter into (u, v)
// order happens in LDS, and the stores are whole columns.
// Bound by one workgroup's phases in turn (LDS holds one block; two half
// blocks per CU read P's rows twice: 2.5 ms): 24 waters, 3.2 GB of blocks in
// 1.8 ms, of which their plain write is 0.7.  Before: 3.4
// ms with lanes in (u, v) order gathering from both places (0.96 GB fetched
// per 290 MB chunk), 20.9 ms with the integral kernels storing to the dense
// array themselves.
// LDS: VALS values, THREADS threads: 16 KiB for n <= 63, several workgroups
// per CU; 128 KiB above, n > 180 in several ranges of u.
template <int VALS, int THREADS>
__global__ __launch_bounds__(THREADS) void k_expand(ExpandArgs a) {
    const int m0 = a.m[blockIdx.y], m1 = a.m[blockIdx.y + 1];
    __shared__ double s_b[VALS];
    const int b = blockIdx.x, irec = (b & ~255) + (b & 7) * 32 + ((b & 255) >> 3);
    if (irec >= a.nrec) return;   // (uniform over the workgroup)
    const cptr<ExpandRec> rec = (cptr<ExpandRec>)(a.rec + irec);
    const cptr<long long> c_off = (cptr<long long>)a.off;
    const cptr<int> c_range = (cptr<int>)a.range;
    const int n = a.n, p = rec->pos, ep = rec->ep, l = rec->l, d = rec->d;
    const int cp = (p >= a.pos[1]) + (p >= a.pos[2]);
    const int nfp = cp == 0 ? 1 : cp == 1 ? 3 : 9;
    const int rp = p - (cp == 0 ? a.pos[0] : cp == 1 ? a.pos[1] : a.pos[2]);
    const int t0 = m0 * (m0 + 1) / 2, t1 = m1 * (m1 + 1) / 2, own = l * (l + 1) / 2 + d;
    const int t = threadIdx.x;
    for (int i = t; i < t1 - t0; i += THREADS) s_b[i] = 0.0;
    __syncthreads();
    // a value of (P | Q) to its place, without the degeneracy weights the
    // store carries (powers of two)
    const double w = l == d ? 2.0 : 1.0;
    auto put = [&](int code, double x) {
        const int at = code >> 1;
        if (code < 0 || at < t0 || at >= t1) return;
        x *= w;
        if (code & 1) x *= 2.0;
        if (at == own) x *= 2.0;
        s_b[at - t0] = x;
    };
    // P the bra: kets of its own class from its own rank on, and of the lower
    // classes; four values per thread in flight
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if (c > cp) break;
        const int nfq = c == 0 ? 1 : c == 1 ? 3 : 9;
        const int lo = c_range[2 * ((size_t)a.pos[3] * c + p)], len = c_range[2 * ((size_t)a.pos[3] * c + p) + 1] - lo;
        const int total = len * nfq;
        if (total == 0) continue;
        const double *src = a.x + c_off[(size_t)a.pos[3] * c + p] + lo;
        const int *inv = a.inv + a.inv0[c] + lo * nfq;
        const int self = c == cp ? rp - lo : -1;   // the ket that is P itself
        for (int i0 = t; i0 < total; i0 += 4 * THREADS) {
            int code[4];
            double x[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = min(i0 + k * THREADS, total - 1);
                const int eq = c == 0 ? 0 : i / len, r = i - eq * len;
                // within one pair only the elements in ascending order are kept
                const int e = r == self ? min(ep, eq) * nfq + max(ep, eq) : ep * nfq + eq;
                code[k] = inv[r * nfq + eq];
                x[k] = src[r + (long long)e * len];
            }
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (i0 + k * THREADS < total) put(code[k], x[k]);
        }
    }
    // Q the bra: the higher classes, and its own class up to the rank before
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if (c < cp) continue;
        constexpr int kQ[3] = {4, 2, 1};   // pairs Q per thread in flight
        const int nfq = c == 0 ? 1 : c == 1 ? 3 : 9;
        const int q0 = a.pos[c], q1 = c == cp ? p : a.pos[c + 1];
        const int *inv = a.inv + a.inv0[c];
        const long long *off = a.off + (size_t)a.pos[3] * cp;
        const int2 *range = reinterpret_cast<const int2 *>(a.range) + (size_t)a.pos[3] * cp;
        for (int qt = q0 + t; qt < q1; qt += kQ[c] * THREADS) {
            double v[4][9];
            bool ok[4];
#pragma unroll
            for (int k = 0; k < kQ[c]; ++k) {
                const int q = min(qt + k * THREADS, q1 - 1);
                const int2 r = range[q];
                ok[k] = qt + k * THREADS < q1 && rp >= r.x && rp < r.y;
                const int len = r.y - r.x, at = min(max(rp, r.x), max(r.y - 1, r.x));
                const double *src = a.x + (len > 0 ? off[q] + at + (long long)ep * len : 0);
                const long long step = len > 0 ? (long long)nfp * len : 0;
#pragma unroll
                for (int e = 0; e < nfq; ++e) v[k][e] = src[e * step];
            }
#pragma unroll
            for (int k = 0; k < kQ[c]; ++k)
                if (ok[k])
#pragma unroll
                    for (int e = 0; e < nfq; ++e) put(inv[(qt + k * THREADS - q0) * nfq + e], v[k][e]);
        }
    }
    __syncthreads();
    // the square: a wavefront per column v, rows u with max(u, v) in [m0, m1)
    double *X = a.X + (size_t)n * n * rec->blk, *X2 = nullptr;
    if (a.d1 > 0) {
        // (one of them at least is within the slab)
        const bool in = d >= a.d0 && d < a.d1, in2 = l >= a.d0 && l < a.d1;
        double *Y = a.X + (size_t)n * n * (d + (size_t)n * (l - a.d0));
        X = in ? a.X + (size_t)n * n * (l + (size_t)n * (d - a.d0)) : Y;
        if (in && in2 && l != d) X2 = Y;
    }
    for (int v = t >> 6; v < m1; v += THREADS / 64)
        for (int u = (v < m0 ? m0 : 0) + (t & 63); u < m1; u += 64) {
            const int hi = max(u, v), lo = min(u, v);
            const double x = s_b[hi * (hi + 1) / 2 + lo - t0];
            X[u + (size_t)n * v] = x;
            if (X2) X2[u + (size_t)n * v] = x;
        }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

// Bytes of expanded blocks held at a time: a few rounds of the transforms'
// workgroups, and of the order of the last-level cache.
constexpr size_t kChunkBytes = kKeepWork;
// a value store of the expansion's own above this is given back after the call
constexpr size_t kKeepStore = (size_t)2 << 30;

int DenseSource::open(double tol) {
    if (ctx->have_eri && ctx->eri_tol == tol && ctx->eri_by_rule) {
        opened = true;
        return 0;
    }
    if (ctx->have_eri) {
        for (int c = 0; c < 6; ++c) {
            saved.cls[c] = ctx->cls[c];
            ctx->cls[c] = QuartetClass{};
        }
        saved.plan = std::move(ctx->plan);
        ctx->plan = DigestPlan();
        saved.d_segoff = ctx->d_segoff;
        saved.d_rank = ctx->d_rank;
        saved.d_x64 = ctx->d_x64;
        saved.d_x32 = ctx->d_x32;
        ctx->d_segoff = nullptr;
        ctx->d_rank = nullptr;
        ctx->d_x64 = nullptr;
        ctx->d_x32 = nullptr;
        saved.n_stored = ctx->n_stored;
        saved.n_quartets = ctx->n_quartets;
        saved.eri_flops = ctx->eri_flops;
        saved.ns = ctx->ns;
        saved.by_rule = ctx->eri_by_rule;
        swapped = true;
    }
    opened = true;
    return eri_values(ctx, tol, false, false);
}

void DenseSource::close() {
    if (!opened) return;
    opened = false;
    if (swapped) {
        for (int c = 0; c < 6; ++c) {
            dfree((void **)&ctx->cls[c].d_cum);
            ctx->cls[c] = saved.cls[c];
        }
        dfree((void **)&ctx->d_segoff);
        dfree((void **)&ctx->d_rank);
        dfree((void **)&ctx->d_x64);
        dfree((void **)&ctx->d_x32);
        ctx->plan = std::move(saved.plan);
        ctx->d_segoff = saved.d_segoff;
        ctx->d_rank = saved.d_rank;
        ctx->d_x64 = saved.d_x64;
        ctx->d_x32 = saved.d_x32;
        ctx->n_stored = saved.n_stored;
        ctx->n_quartets = saved.n_quartets;
        ctx->eri_flops = saved.eri_flops;
        ctx->ns = saved.ns;
        ctx->eri_by_rule = saved.by_rule;
        swapped = false;
    } else if (!ctx->have_eri && dcapacity(ctx->d_x64) > kKeepStore) {
        dfree((void **)&ctx->d_x64);
    }
}

// The tables and records, in one upload to ctx->d_dtab: chunks of all blocks
// (d1 = 0), or the records of the blocks with an index within [d0, d1).
int DenseSource::tables(int d0, int d1) {
    const DigestPlan &pl = ctx->plan;
    const int n = ctx->n, np = (int)ctx->pairs.size();
    pos[0] = inv0[0] = 0;
    int ninv = 0;
    for (int c = 0; c < 3; ++c) {
        pos[c + 1] = pos[c] + (int)ctx->pair_ids[c].size();
        inv0[c] = ninv;
        ninv += (int)ctx->pair_ids[c].size() * dig_ncd(c);
    }
    std::vector<long long> off(3 * (size_t)np);
    std::vector<int> range(6 * (size_t)np), inv(ninv), tri;
    std::vector<ExpandRec> recs;
    recs.reserve((size_t)n * (n + 1) / 2);
    tri.reserve((size_t)n * (n + 1) / 2);
    for (int c = 0; c < 3; ++c) {
        const auto &ids = ctx->pair_ids[c];
        const int nf = dig_ncd(c), nb = c == 2 ? 3 : 1;
        for (size_t r = 0; r < ids.size(); ++r) {
            const int p = ids[r];
            const size_t q = pos[c] + r;
            for (int k = 0; k < 3; ++k) {
                const size_t at = (size_t)np * k + q;
                off[at] = pl.off[3 * (size_t)p + k];
                range[2 * at] = pl.lo[3 * (size_t)p + k];
                range[2 * at + 1] = pl.hi[3 * (size_t)p + k];
            }
        }
        // element by element over the class's pairs: neighbours in rank are
        // neighbours in the list.  Of a shell with itself only the elements
        // in ascending order are kept.
        for (int e = 0; e < nf; ++e)
            for (size_t r = 0; r < ids.size(); ++r) {
                const ShellPair &sp = ctx->pairs[ids[r]];
                const int x = e / nb, y = e % nb, i = sp.ao_a + x, j = sp.ao_b + y;
                const int l = std::max(i, j), d = std::min(i, j), at = l * (l + 1) / 2 + d;
                const bool kept = !(sp.same && x > y);
                inv[inv0[c] + r * nf + e] = kept ? 2 * at + (l == d) : -1;
                if (!kept || (d1 > 0 && (d < d0 || d >= d1) && (l < d0 || l >= d1))) continue;
                recs.push_back(ExpandRec{pos[c] + (int)r, e, l, d, 0});
                tri.push_back(at);
            }
    }
    nrec = (int)recs.size();
    // chunks of whole rounds of a workgroup per CU
    const size_t nn8 = sizeof(double) * (size_t)n * n;
    int most = d1 > 0 ? nrec : (int)std::min<size_t>(nrec, std::max<size_t>(1, kChunkBytes / nn8));
    if (most > 256 && most < nrec) most -= most % 256;
    chunks.clear();
    for (int r = 0; r < nrec; r += most) chunks.push_back(ExpandChunk{r, std::min(most, nrec - r)});
    for (int r = 0; r < nrec; ++r) recs[r].blk = r % most;
    const size_t b_off = sizeof(long long) * off.size(), b_range = sizeof(int) * range.size(),
                 b_rec = sizeof(ExpandRec) * recs.size(), b_inv = sizeof(int) * inv.size(),
                 b_tri = sizeof(int) * tri.size();
    std::vector<unsigned char> h(b_off + b_range + b_rec + b_inv + b_tri);
    unsigned char *w = h.data();
    auto put = [&](const void *src, size_t b) {
        memcpy(w, src, b);
        w += b;
    };
    put(off.data(), b_off);
    put(range.data(), b_range);
    put(recs.data(), b_rec);
    put(inv.data(), b_inv);
    put(tri.data(), b_tri);
    MYQC_CHECK(dalloc(ctx, &ctx->d_dtab, h.size()));
    MYQC_HIP(ctx, hipMemcpyAsync(ctx->d_dtab, h.data(), h.size(), hipMemcpyHostToDevice, ctx->stream));
    MYQC_HIP(ctx, hipStreamSynchronize(ctx->stream));   // (h goes out of scope)
    const unsigned char *dev = static_cast<const unsigned char *>(ctx->d_dtab);
    d_off = reinterpret_cast<const long long *>(dev);
    d_range = reinterpret_cast<const int *>(dev + b_off);
    d_rec = reinterpret_cast<const ExpandRec *>(dev + b_off + b_range);
    d_inv = reinterpret_cast<const int *>(dev + b_off + b_range + b_rec);
    d_tri = reinterpret_cast<const int *>(dev + b_off + b_range + b_rec + b_inv);
    return 0;
}

int DenseSource::plan_chunks() { return tables(0, 0); }

size_t DenseSource::chunk_bytes() const {
    return chunks.empty() ? 0 : sizeof(double) * (size_t)ctx->n * ctx->n * chunks[0].nblk;
}

int DenseSource::launch(const ExpandChunk &c, double *X, int d0, int d1) {
    const int n = ctx->n;
    ExpandArgs a{ctx->d_x64, d_inv, d_off, d_range, d_rec + c.blk0, X, n, c.nblk, {pos[0], pos[1], pos[2], pos[3]},
                 {inv0[0], inv0[1], inv0[2]}, d0, d1, {}};
    const unsigned grid = (unsigned)((c.nblk + 255) / 256 * 256);
    constexpr int kLT = 1024;
    const int tri = n * (n + 1) / 2;
    if (tri <= kExpSmall) {
        a.m[1] = n;
        k_expand<kExpSmall, 256><<<grid, 256, 0, ctx->stream>>>(a);
    } else {
        // ranges of u of about equal size
        int parts = 0, m = 0;
        const int want = (tri + kExpLarge - 1) / kExpLarge;
        for (; m < n && parts < kExpParts; ++parts) {
            const int t0 = m * (m + 1) / 2;
            const long long goal = std::min<long long>((long long)tri * (parts + 1) / want, (long long)t0 + kExpLarge);
            while (m < n && (long long)(m + 1) * (m + 2) / 2 <= goal) ++m;
            a.m[parts + 1] = m;
            if (m * (m + 1) / 2 == t0) return set_error(ctx, MYQC_E_ARG, "dense integrals: n=%d too large", n);
        }
        if (m < n) return set_error(ctx, MYQC_E_ARG, "dense integrals: n=%d too large", n);
        k_expand<kExpLarge, kLT><<<dim3(grid, (unsigned)parts), kLT, 0, ctx->stream>>>(a);
    }
    MYQC_HIP(ctx, hipGetLastError());
    return 0;
}

int DenseSource::expand(const ExpandChunk &c, double *X) { return launch(c, X, 0, 0); }

int DenseSource::expand_full(double *XX, int d0, int d1) {
    MYQC_CHECK(tables(d0, d1));
    return launch(ExpandChunk{0, nrec}, XX, d0, d1);
}

}  // namespace myqc
