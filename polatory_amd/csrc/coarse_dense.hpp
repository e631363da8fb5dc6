// The coarse grid's dense linear algebra: Cholesky factorisation of one large
// matrix and the grid's solve (coarse_grid.hpp:105-131) as an explicit operator.
#pragma once

#include "common.hpp"

namespace pam {

constexpr int kCoarseBlk = 64;  // panel width and tile edge

// Lower Cholesky factor of the n x n matrix a (column-major, lower triangle;
// the upper one is not touched) in place. Sets *flag where a pivot is not
// positive. lscr: kCoarseBlk^2 scratch. x (n x n, or null): receives the
// inverses of the factor's diagonal blocks, for launch_coarse_inverse.
void launch_coarse_factor(double* a, int n, int32_t* flag, double* x, double* lscr, hipStream_t s);

// x (the diagonal blocks' inverses on entry) becomes the inverse of the factor
// a; t: n x n scratch.
void launch_coarse_inverse(const double* a, int n, double* x, double* t, hipStream_t s);

// op ((m + l) x m, row-major) = [Q W Q^T; pinv (E - A_top Q W Q^T)] with
// W = x^T x (n x n, n = m - l), Q = [-lag^T; I] over the rows idx, E the first
// l rows of the identity and atop = A_top (l x m).
void launch_coarse_operator(const double* x, int m, int l, const int32_t* idx, const double* lag,
                            const double* atop, const double* pinv, double* op, hipStream_t s);

}  // namespace pam
