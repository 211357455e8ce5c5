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

struct ExpandArgs {
    const double *x;
    const int *T;              // [u + n v]: position of the function pair's shell pair << 4 | element
    const long long *off;      // [3 pos + ket class]: value offset (element e of ket rank r at off + r + e len)
    const int2 *range;         // [3 pos + ket class]: its ket ranks [lo, hi)
    const ExpandRec *rec;
    double *X;
    int n, pos1, pos2;         // first position of classes 1 and 2
    int full;                  // blocks at l + n d and d + n l
};

// One record's blocks over one 32 x 32 tile of (u, v) and its mirror image
// (tiles tu >= tv).  A lane owns four (u, v) of the tile; for the record's
// pairs P in turn it reads the element of (P | Q), Q the shell pair of (u, v),
// from whichever of the two is the bra.  As P runs over consecutive ranks,
// the reads from Q's block walk along one cache line; the reads from P's
// block are spread over it by Q's rank, but all of it is read by the
// record's other tiles.  Bound by those line fetches from L2: 24 waters,
// 3.2 GB of blocks in 3.4 ms (before: 20 ms of scattered stores and 0.83
// ms of clearing).
__global__ __launch_bounds__(256) void k_expand(ExpandArgs a) {
    constexpr int G = 4;   // pairs at a time
    __shared__ double s_t[G][32][33];
    const ExpandRec &rec = a.rec[blockIdx.x];
    int tu = 0, rem = blockIdx.y;
    while (rem > tu) rem -= ++tu;
    const int tv = rem;   // blockIdx.y = tu (tu + 1) / 2 + tv
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int n = a.n, cp = rec.cls, ep = rec.ep;
    const size_t nn = (size_t)n * n;
    const int base_p = cp == 0 ? 0 : cp == 1 ? a.pos1 : a.pos2;
    const int nfp = cp == 0 ? 1 : cp == 1 ? 3 : 9;
    const int u = tu * 32 + tx;
    // the lane's four (u, v): position, element and class of Q, and Q's
    // block for kets of P's class
    int q[4], eq[4], cq[4], lenq[4], loq[4], hiq[4];
    long long offq[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int v = tv * 32 + ty + 8 * k;
        const int t = (u < n && v < n) ? a.T[u + n * v] : a.T[0];
        q[k] = t >> 4;
        eq[k] = t & 15;
        cq[k] = (q[k] >= a.pos1) + (q[k] >= a.pos2);
        const int2 r = a.range[3 * q[k] + cp];
        loq[k] = r.x;
        hiq[k] = r.y;
        lenq[k] = r.y - r.x;
        offq[k] = a.off[3 * q[k] + cp] + (long long)(eq[k] * nfp + ep) * lenq[k];
    }
    for (int h = 0; h < kExpPairs; h += G) {
        double val[G][4];
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const int ld = rec.ld[h + j];
            if (ld < 0) continue;   // (uniform over the workgroup)
            const int p = rec.pos0 + h + j, rp = p - base_p;
            const int l = ld % n, d = ld / n;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int v = tv * 32 + ty + 8 * k;
                const int rq = q[k] - (cq[k] == 0 ? 0 : cq[k] == 1 ? a.pos1 : a.pos2);
                const int nfq = cq[k] == 0 ? 1 : cq[k] == 1 ? 3 : 9;
                bool ok;
                long long at;
                if (cp > cq[k] || (cp == cq[k] && rp <= rq)) {
                    const int2 r = a.range[3 * p + cq[k]];
                    ok = rq >= r.x && rq < r.y;
                    // within one pair only the elements in ascending order are kept
                    const int e = p == q[k] ? min(ep, eq[k]) * nfq + max(ep, eq[k]) : ep * nfq + eq[k];
                    at = a.off[3 * p + cq[k]] + rq + (long long)e * (r.y - r.x);
                } else {
                    ok = rp >= loq[k] && rp < hiq[k];
                    at = offq[k] + rp;
                }
                double x = ok ? a.x[at] : 0.0;
                // the degeneracy weights the store carries (powers of two)
                if (l == d) x *= 2.0;
                if (u == v) x *= 2.0;
                if ((u == l && v == d) || (u == d && v == l)) x *= 2.0;
                val[j][k] = x;
            }
        }
#pragma unroll
        for (int j = 0; j < G; ++j) {
            if (rec.ld[h + j] < 0) continue;
            double *X = a.X + nn * rec.blk[h + j];
            const int l = rec.ld[h + j] % n, d = rec.ld[h + j] / n;
            double *X2 = a.full && l != d ? a.X + nn * ((size_t)d + (size_t)n * l) : nullptr;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int v = tv * 32 + ty + 8 * k;
                s_t[j][ty + 8 * k][tx] = val[j][k];
                if (u >= n || v >= n) continue;
                X[u + (size_t)n * v] = val[j][k];
                if (X2) X2[u + (size_t)n * v] = val[j][k];
            }
        }
        if (tu != tv) {
            __syncthreads();
#pragma unroll
            for (int j = 0; j < G; ++j) {
                if (rec.ld[h + j] < 0) continue;
                double *X = a.X + nn * rec.blk[h + j];
                const int l = rec.ld[h + j] % n, d = rec.ld[h + j] / n;
                double *X2 = a.full && l != d ? a.X + nn * ((size_t)d + (size_t)n * l) : nullptr;
                const int v = tv * 32 + tx;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int uu = tu * 32 + ty + 8 * k;
                    if (uu >= n || v >= n) continue;
                    const double x = s_t[j][tx][ty + 8 * k];
                    X[v + (size_t)n * uu] = x;
                    if (X2) X2[v + (size_t)n * uu] = x;
                }
            }
            __syncthreads();
        }
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
    if (ctx->have_eri && ctx->eri_tol == tol) {
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
        swapped = true;
    }
    opened = true;
    return eri_values(ctx, tol, false);
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
        swapped = false;
    } else if (!ctx->have_eri && dcapacity(ctx->d_x64) > kKeepStore) {
        dfree((void **)&ctx->d_x64);
    }
}

// The tables and records, in one upload to ctx->d_dtab.
int DenseSource::tables(bool full) {
    const DigestPlan &pl = ctx->plan;
    const int n = ctx->n, np = (int)ctx->pairs.size();
    pos1 = (int)ctx->pair_ids[0].size();
    pos2 = pos1 + (int)ctx->pair_ids[1].size();
    const int pos0[3] = {0, pos1, pos2};
    std::vector<long long> off(3 * (size_t)np);
    std::vector<int> range(6 * (size_t)np), T((size_t)n * n), tri;
    std::vector<ExpandRec> recs;
    const size_t nn8 = sizeof(double) * (size_t)n * n;
    long long most = full ? 1LL << 60 : std::max<long long>(kExpPairs, (long long)(kChunkBytes / nn8));
    if (!full && most > 256) most -= most % 256;   // whole rounds of a workgroup per CU
    chunks.clear();
    ExpandChunk ch{0, 0, 0, 0};
    for (int c = 0; c < 3; ++c) {
        const auto &ids = ctx->pair_ids[c];
        for (size_t r = 0; r < ids.size(); ++r) {
            const int p = ids[r], pos = pos0[c] + (int)r;
            for (int k = 0; k < 3; ++k) {
                off[3 * (size_t)pos + k] = pl.off[3 * (size_t)p + k];
                range[6 * (size_t)pos + 2 * k] = pl.lo[3 * (size_t)p + k];
                range[6 * (size_t)pos + 2 * k + 1] = pl.hi[3 * (size_t)p + k];
            }
            const ShellPair &sp = ctx->pairs[p];
            const int na = sp.la ? 3 : 1, nb = sp.lb ? 3 : 1;
            for (int x = 0; x < na; ++x)
                for (int y = 0; y < nb; ++y) {
                    // of a shell with itself only the elements x <= y are kept
                    const int e = sp.same && x > y ? y * nb + x : x * nb + y;
                    T[(sp.ao_a + x) + (size_t)n * (sp.ao_b + y)] = pos << 4 | e;
                    T[(sp.ao_b + y) + (size_t)n * (sp.ao_a + x)] = pos << 4 | e;
                }
        }
        // records: element by element over runs of pairs
        const int nf = c == 0 ? 1 : c == 1 ? 3 : 9, nb = c == 2 ? 3 : 1;
        for (size_t r0 = 0; r0 < ids.size(); r0 += kExpPairs)
            for (int e = 0; e < nf; ++e) {
                ExpandRec rec;
                rec.pos0 = pos0[c] + (int)r0;
                rec.cls = c;
                rec.ep = e;
                rec.pad = 0;
                int cnt = 0;
                for (int j = 0; j < kExpPairs; ++j) {
                    rec.ld[j] = rec.blk[j] = -1;
                    if (r0 + j >= ids.size()) continue;
                    const ShellPair &sp = ctx->pairs[ids[r0 + j]];
                    const int x = e / nb, y = e % nb;
                    if (sp.same && x > y) continue;
                    const int l = std::max(sp.ao_a + x, sp.ao_b + y), d = std::min(sp.ao_a + x, sp.ao_b + y);
                    rec.ld[j] = l + n * d;
                    ++cnt;
                }
                if (cnt == 0) continue;
                if (ch.nblk + cnt > most) {
                    chunks.push_back(ch);
                    ch = ExpandChunk{ch.rec0 + ch.nrec, 0, ch.blk0 + ch.nblk, 0};
                }
                for (int j = 0; j < kExpPairs; ++j) {
                    if (rec.ld[j] < 0) continue;
                    const int l = rec.ld[j] % n, d = rec.ld[j] / n;
                    rec.blk[j] = full ? rec.ld[j] : ch.nblk;
                    tri.push_back(l * (l + 1) / 2 + d);
                    ++ch.nblk;
                }
                ++ch.nrec;
                recs.push_back(rec);
            }
    }
    if (ch.nrec) chunks.push_back(ch);
    nrec = (int)recs.size();
    const size_t b_off = sizeof(long long) * off.size(), b_range = sizeof(int) * range.size(),
                 b_rec = sizeof(ExpandRec) * recs.size(), b_T = sizeof(int) * T.size(), b_tri = sizeof(int) * tri.size();
    std::vector<unsigned char> h(b_off + b_range + b_rec + b_T + b_tri);
    unsigned char *w = h.data();
    auto put = [&](const void *src, size_t b) {
        memcpy(w, src, b);
        w += b;
    };
    put(off.data(), b_off);
    put(range.data(), b_range);
    put(recs.data(), b_rec);
    put(T.data(), b_T);
    put(tri.data(), b_tri);
    MYQC_CHECK(dalloc(ctx, &ctx->d_dtab, h.size()));
    MYQC_HIP(ctx, hipMemcpyAsync(ctx->d_dtab, h.data(), h.size(), hipMemcpyHostToDevice, ctx->stream));
    MYQC_HIP(ctx, hipStreamSynchronize(ctx->stream));   // (h goes out of scope)
    const unsigned char *dev = static_cast<const unsigned char *>(ctx->d_dtab);
    d_off = reinterpret_cast<const long long *>(dev);
    d_range = reinterpret_cast<const int2 *>(dev + b_off);
    d_rec = reinterpret_cast<const ExpandRec *>(dev + b_off + b_range);
    d_T = reinterpret_cast<const int *>(dev + b_off + b_range + b_rec);
    d_tri = reinterpret_cast<const int *>(dev + b_off + b_range + b_rec + b_T);
    return 0;
}

int DenseSource::plan_chunks() { return tables(false); }

size_t DenseSource::chunk_bytes() const {
    size_t most = 1;
    for (const auto &c : chunks) most = std::max(most, (size_t)c.nblk);
    return sizeof(double) * (size_t)ctx->n * ctx->n * most;
}

int DenseSource::expand(const ExpandChunk &c, double *X) {
    const int tiles = (ctx->n + 31) / 32;
    ExpandArgs a{ctx->d_x64, d_T, d_off, d_range, d_rec + c.rec0, X, ctx->n, pos1, pos2, 0};
    k_expand<<<dim3((unsigned)c.nrec, (unsigned)(tiles * (tiles + 1) / 2)), 256, 0, ctx->stream>>>(a);
    MYQC_HIP(ctx, hipGetLastError());
    return 0;
}

int DenseSource::expand_full(double *XX) {
    MYQC_CHECK(tables(true));
    const int tiles = (ctx->n + 31) / 32;
    ExpandArgs a{ctx->d_x64, d_T, d_off, d_range, d_rec, XX, ctx->n, pos1, pos2, 1};
    k_expand<<<dim3((unsigned)nrec, (unsigned)(tiles * (tiles + 1) / 2)), 256, 0, ctx->stream>>>(a);
    MYQC_HIP(ctx, hipGetLastError());
    return 0;
}

}  // namespace myqc
