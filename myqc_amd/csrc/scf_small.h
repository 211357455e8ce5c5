// scf_small.h -- the dense steps of the RHF loop for a system small enough
// that its matrices fit one workgroup's LDS (scf_small.hip).
#pragma once

#include "context.h"

namespace myqc {

// functions at most: above, the general loop's launches over the whole chip are
// no slower than one CU's matrix cores and its Jacobi (figures in scf_small.hip)
constexpr int kSmallScfN = 84;

// results of one small_step, in this order
enum SmallOut { SO_DF = 0, SO_DH, SO_DD, SO_B, SO_OK = SO_B + 8, SO_STEPS, SO_COUNT };

struct SmallStep {
    int n, nocc;
    int core;               // 1: the density of H alone (no error, no DIIS)
    int head, hn;           // DIIS slot of this iteration, history length with it
    int with_dd;            // 1: max |D - Dprev| is wanted
    int g_half;             // 1: G holds A of G(D) = A + A^T (digest_A)
    double shift, shift_err;   // level shift while the DIIS error is above shift_err (shift 0: none)
    const double *H, *G, *X, *D, *Dprev, *Do;
    double *hF, *hE;        // histories, n^2 per slot
    double *B;              // 8 x 8 DIIS matrix
    double *Fx;             // the extrapolated (shifted) Fock matrix, orthonormal basis
    double *Don, *Dnext;    // the new projector and density
    double *out;            // SO_COUNT values (pinned host memory)
};

int small_step(myqc_ctx *ctx, const SmallStep &s);
// X = S^-1/2, Xi = S^1/2; Y, Z: n x n scratch; out[0] = 1 when converged (pinned host memory)
int small_inv_sqrt(myqc_ctx *ctx, int n, const double *S, double *X, double *Xi, double *Y, double *Z, double *out);
// eigenvalues of Fo ascending into eig, C = X times its eigenvectors
int small_orbitals(myqc_ctx *ctx, int n, const double *Fo, const double *X, double *C, double *eig);

}  // namespace myqc
