// FP64 matrix-core products of the density-fitted exchange (mjk_dfgemm.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace mjk {

// The half-transformed tensor Y: element (P, o) of row i at P + i is + o yo, by
// row (i, o, P) or by column (o, i, P); and its rows as columns of the exchange
// product, inner element k = (o, P) at (k / np) os + i is + k % np.  The fitted
// tensor B, symmetric in its orbital pair, reads as Y of all columns does.
struct KLayout {
    long long np, is, os;   // contiguous inner elements, strides of a row and of a contiguous run
    long long yo;           // stride of a column
};
KLayout df_layout(int nao, int naux, int ncol);

// Split of a long-inner-dimension product C = A^T B (C n x n, A and B
// columns of length kin): 64 x 64 tiles x nsplit slices of the inner dimension.
struct TnPlan {
    int nt = 0;            // tiles per dimension
    int ntile = 0;         // tiles computed (the lower triangle when C is symmetric)
    int nsplit = 0;        // slices of the inner dimension, a multiple of 8 (one XCD each)
    long long kc = 0;      // inner length of a slice, a multiple of 16
    size_t ws = 0;         // workspace doubles
};
TnPlan df_tn_plan(int n, long long kin, bool sym);

// C (n x n, column-major) = A^T B; sym: A == B, the lower tiles computed and
// mirrored.  part: plan.ws doubles.
int df_tn(const TnPlan& plan, const double* A, const double* B, int n, long long kin, const KLayout& la, bool sym,
          double* part, double* C, hipStream_t st);

// Y_i = B_i X for i < nao, B_i the naux x nao column-major block at B + i naux
// nao; X given transposed and padded by df_pad_x.
int df_y(const double* B, const double* Xp, int nao, int naux, int ncol, const KLayout& la, double* Y,
         hipStream_t st);

// doubles of the padded copy of X, and the copy: X(l, o) at src[l sl + o so]
size_t df_xp_size(int nao, int ncol);
int df_pad_x(const double* src, long long sl, long long so, int nao, int ncol, double* Xp, hipStream_t st);

// Cholesky factor of a symmetric positive definite n x n matrix (both triangles
// given) into its lower triangle, column-major; the strict upper triangle is
// left undefined.  info (zeroed by the caller): first row whose pivot is not
// positive, from 1.  tmp: CHOL_NB^2 doubles.
constexpr int CHOL_NB = 32;
int df_potrf(double* A, int n, double* tmp, int* info, hipStream_t st);

}  // namespace mjk
