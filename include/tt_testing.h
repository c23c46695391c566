/*
 * tt_testing.h -- test hooks of the trace-transform library (no reference
 * counterpart; not part of the path's interface).  The test suite uses them
 * to reach code the public entry points cannot isolate.
 */
#ifndef TT_TESTING_H
#define TT_TESTING_H

#include "tt.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Lets the next `allowed` workspace allocations of every context succeed and
 * makes the ones after fail as out of memory, so that TT_ERR_NOMEM can be
 * exercised; a negative value removes the limit. */
TT_API tt_status tt_testing_fail_allocations(long long allowed);

/* Makes every workspace allocation of more than `bytes` fail as out of memory,
 * as on a device without room for it; 0 removes the limit. */
TT_API tt_status tt_testing_limit_allocation(size_t bytes);

/* Makes the batched line kernels of the plans that follow sample from the
 * images and their row-major copies (0) or from the pixel pairs (1), whatever
 * the sizes; negative: the rule's choice. */
TT_API tt_status tt_testing_line_pairs(int pairs);

/* Rows and columns of the tiles that P3's DFT products (forward or adjoint) of
 * cols columns of n rows take.  Needs no device. */
TT_API tt_status tt_testing_dft_shape(int n, int cols, int forward, int *rows, int *columns);

/* The launch shape of a single image's transposed rotation (n x n pixels) on a
 * device of `cus` CUs, for the gradients of nt T-functionals: waves per
 * workgroup and angle groups.  Needs no device. */
TT_API tt_status tt_testing_gather_launch(int n, int n_angles, int cus, const int32_t *tcodes,
                                          int nt, int *waves, int *groups);

/* Compares the sort kernel's short square root (v_sqrt_f32 and one residual
 * test per neighbour) with the correctly rounded sqrtf on the GPU for the
 * float bit patterns [lo, lo + count), skipping its documented exceptions
 * (0, 2^-96) and the negative denormals: the number of patterns whose
 * results differ (NaN results compare equal) and the smallest of them
 * (0xFFFFFFFF if none). */
TT_API tt_status tt_testing_short_sqrt(tt_context *ctx, uint32_t lo, uint64_t count,
                                       uint64_t *mismatches, uint32_t *first_bad);

/* The same for the line kernel's root (v_rsq_f32 and one Newton step), on 0,
 * NaN and [2^-96, 2^127). */
TT_API tt_status tt_testing_line_root(tt_context *ctx, uint32_t lo, uint64_t count,
                                      uint64_t *mismatches, uint32_t *first_bad);

/* Runs the FP64 matrix-core products of the nearest-orthonormal iteration
 * on a strided batch of `count` column-major matrices (device pointers,
 * matrices stored back to back): C = A^T B (trans_a: A is k x m) or A B
 * (A is m x k; when k is a multiple of 4, B must be symmetric: it is read
 * transposed), B k x n, C m x n.  sym: m == n and the product is known to
 * be symmetric; only the blocks on and below the diagonal are computed and
 * each value is written to (i, j) and (j, i).  With coef (5 doubles,
 * sym, A = B = S of k x k, k a multiple of 4) the product is the polynomial
 * step's S S, whose kernel also writes T = c3 S + c4 S^2 to d_t and
 * Q = c0 I + c1 S + c2 S^2 to d_q.  Returns after the context's stream has
 * finished. */
TT_API tt_status tt_testing_nos_product(tt_context *ctx, int trans_a, int sym, int count,
                                        int m, int n, int k, const double *d_a,
                                        const double *d_b, double *d_c, const double *coef,
                                        double *d_t, double *d_q);

#ifdef __cplusplus
}
#endif
#endif
