// Dense LU of the single-network solver (dense.hip).
#pragma once

#include <climits>

#include "kernels.hpp"

namespace pf {

constexpr int kDenseMax = 4096;      // unknowns: four rows per thread of one workgroup
constexpr int kDenseCols = 8;        // columns a workgroup updates
constexpr int kDenseSwaps = 1 + 2 * 2 * 32;   // ints of the panel's swap list

// Solves A x = b (n x n column-major, n <= kDenseMax) with partial pivoting;
// A is overwritten by its factors, b by x.  Raises ctl->singular where a
// column has no positive finite pivot, and leaves b undefined then.
void launch_dense_solve(double *A, double *b, int n, int *chg, Ctl *ctl, int gate, hipStream_t st);

}  // namespace pf
