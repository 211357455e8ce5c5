// batch_find.h -- which molecule of a batch a quartet of a class belongs to.
#pragma once

#include <vector>

#include "eri_math.h"

namespace myqc {

// qcum: prefix counts of the molecules' quartets, one more than molecules.
// The molecules of quartets 0, 64, 128, ... and, one entry more, of the last.
inline std::vector<int> quartet_marks(const std::vector<long long> &qcum) {
    const int nmol = (int)qcum.size() - 1;
    const long long nq = qcum[nmol];
    std::vector<int> first(nq > 0 ? (size_t)((nq + 63) / 64) + 1 : 0);
    for (int m = 0; m < nmol; ++m) {   // the quartets 64 k of molecule m
        for (long long k = (qcum[m] + 63) / 64; 64 * k < qcum[m + 1]; ++k) first[k] = m;
        if (qcum[m] < qcum[m + 1]) first.back() = m;
    }
    return first;
}

// The molecule of quartet t: the last with qcum <= t, by bisection between the
// marks before and after t.  Within one molecule, the ordinary case, that is
// the two marks alone; a wavefront that straddles a long run of molecules
// without a quartet of the class reads no more than a search over the batch.
// (A walk from the mark reads them one after another, each load waiting for the
// one before: 8 clusters of 5 waters with 4000 helium atoms after each, one whole
// batch, 6.3 ms against 4.5; 1024 clusters 10.9 either way.)
template <typename Q>
MYQC_HD int quartet_molecule(const Q &qcum, const int *first, long long t) {
    int lo = first[t >> 6], hi = first[(t >> 6) + 1];
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (qcum[mid] <= t) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

}  // namespace myqc
