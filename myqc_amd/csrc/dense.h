// dense.h -- square blocks of the AO integrals, (uv|ld) over all u, v for one
// function pair (l, d), expanded from the stored (element-major, pre-weighted)
// integrals of digest_plan.h.
#pragma once

#include "context.h"

namespace myqc {

// One function pair l >= d: its class-sorted shell pair, the element of it,
// and the block it goes to.
struct ExpandRec {
    int pos, ep, l, d, blk;
};

// A run of function pairs whose blocks fit the work buffer
struct ExpandChunk {
    int blk0, nblk;
};

// The values of the quartets above the Schwarz threshold `tol`, opened for
// expansion: the context's stored integrals when they were built at that
// threshold and in the rule's launch shapes (others sum in another order),
// else a build of its own, which leaves the context's stored integrals as
// they are.  close() (or the destructor) gives back what the open made.
class DenseSource {
  public:
    explicit DenseSource(myqc_ctx *c) : ctx(c) {}
    ~DenseSource() { close(); }
    int open(double tol);
    void close();

    // Blocks of the pairs l >= d in chunks: records and tables go to the
    // device; chunk c's blocks are written by expand() to X, block b of the
    // chunk at X + b n^2, and d_tri + chunk.blk0 + b holds its l (l + 1) / 2 + d.
    int plan_chunks();
    std::vector<ExpandChunk> chunks;
    const int *d_tri = nullptr;
    int expand(const ExpandChunk &c, double *X);
    size_t chunk_bytes() const;
    // the blocks of second index d0 .. d1 - 1 of the dense n^4 array, in their
    // order, to XX (n^3 (d1 - d0) values)
    int expand_full(double *XX, int d0, int d1);

  private:
    int tables(int d0, int d1);
    int launch(const ExpandChunk &c, double *X, int d0, int d1);
    myqc_ctx *ctx;
    bool opened = false, swapped = false;
    // the context's own store, put aside while another is open
    struct Saved {
        QuartetClass cls[6];
        DigestPlan plan;
        long long *d_segoff;
        int *d_rank;
        double *d_x64;
        float *d_x32;
        long long n_stored, n_quartets;
        double eri_flops;
        int ns;
        bool by_rule;
    } saved;
    // device tables (ctx->d_dtab)
    const long long *d_off = nullptr;
    const int *d_range = nullptr, *d_inv = nullptr;
    const ExpandRec *d_rec = nullptr;
    int nrec = 0, pos[4] = {0, 0, 0, 0}, inv0[3] = {0, 0, 0};
};

// The transforms' limit: what quarter steps 1 and 2 leave is at most 8 n^3 nvirt
// bytes (both spins' virtual pairs, l >= d), here 200 GB beside the store's n^4.
inline int transform_fits(myqc_ctx *ctx, const char *who) {
    const size_t n = ctx->n;
    if (n * n * n * n * 8 > (size_t)200 << 30)
        return set_error(ctx, MYQC_E_ARG, "%s: n=%zu: the transforms take up to 404 functions", who, n);
    return 0;
}

// One product of quarter steps 1 and 2: M(p, q, l d) from the orbital blocks
// Cp (n x np) and Cq (n x nq), both with leading dimension n.
struct TransformJob {
    const double *Cp;
    int np;
    const double *Cq;
    int nq;
    double *M;
};

}  // namespace myqc
