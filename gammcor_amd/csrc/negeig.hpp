// Eigenpairs below zero of a batch of symmetric FP64 matrices, and from them a
// Cholesky factor of their |A|.
#pragma once
#include "accas.hpp"
#include "common.hpp"

namespace gmc {

// Orders from which abs_factor beats an eigensolve of A (measured, FP64:
// order 2664 x 8 problems 95 ms against 32, 4524 x 16 612 against 150 and 343 in
// FP32; the Krylov basis and its
// Rayleigh-Ritz problem of order 832 cost about the same at every order, so at
// 1359 x 5, 15 ms, there is nothing left to gain).  A spectrum
// that does not converge costs the first basis and its Ritz problem on top of the
// eigensolve (order 2236 x 1: 46 ms of ERPA for 36 with the factor).
constexpr int NEGEIG_MIN = 2048;

// Small scratch of abs_factor (beside the matrix buffers it borrows).
size_t negeig_bytes(int n, int B);

// A (B column-major symmetric n x n matrices, stride n*n): |A| = V |L| V^T is
// formed in place of A and replaced by its Cholesky factor L (strict upper
// triangle zero).  nneg (device, B ints) receives the number of eigenvalues
// below zero.  t0, t1: two buffers of B n x n, overwritten; scratch:
// negeig_bytes; eig: the FP64 eigensolver in ws.  *ok = false (and A
// destroyed) when the eigenpairs did not converge or a pivot of |A| was not
// positive, as when A is singular: the caller then takes the eigensolve.
int abs_factor(hipStream_t s, int n, int B, double* A, double* t0, double* t1, void* scratch, size_t scratch_bytes,
               int* nneg, const EigSolveAt& eig, void* ws, size_t ws_bytes, bool stats, bool* ok);

}  // namespace gmc
