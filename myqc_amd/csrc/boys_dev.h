// boys_dev.h -- the Boys tables (eri_math.h) on the device: their rows, and
// their staging in LDS.
#pragma once

#include "eri_math.h"

namespace myqc {

// Every row of the array, which holds boys_inputs' parts: a thread each,
// kBoysRowBlocks x 64.  A thread's work is a chain of up to 12 recursion steps of
// ten coefficients; on the host the 605 rows would take longer than a small
// system's integrals.
constexpr int kBoysRowBlocks = (FT_NQ * FT_NT + 63) / 64;
static __global__ __launch_bounds__(64) void k_boys_rows(double *full) {
    const int t = blockIdx.x * 64 + threadIdx.x;
    if (t < FT_NQ * FT_NT) boys_row(full, t / FT_NT, t % FT_NT);
}

// Stages the tables of order M: s has ft_staged(M) doubles, 16-byte aligned.
template <int M>
__device__ __forceinline__ BoysTab stage_boys(const double *__restrict__ full, double *s) {
    const double2 *poly = reinterpret_cast<const double2 *>(full + M * FT_BLOCK);
    const double2 *eg = reinterpret_cast<const double2 *>(full + FT_EG);
    double2 *d = reinterpret_cast<double2 *>(s);
    constexpr int NP = FT_POLY / 2, NE = FT_EGN / 2, NT = M >= 2 ? FT_TOP / 2 : 0;
    for (int i = threadIdx.x; i < NP; i += blockDim.x) d[i] = poly[i];
    for (int i = threadIdx.x; i < NE; i += blockDim.x) d[NP + i] = eg[i];
    for (int i = threadIdx.x; i < NT; i += blockDim.x) d[NP + NE + i] = poly[NP + i];
    __syncthreads();
    return {s, s + FT_POLY, reinterpret_cast<const float *>(s + FT_POLY + FT_EGN)};
}

}  // namespace myqc
