// Kernels of FP32 factorisations without row interchanges and of the
// diagonal-block inverses of FP32 factors (nopiv.hip).  Launches run over the
// batch on blockIdx.z: A (and F) in the batch's matrices, the rest in its
// scratch slabs unless noted.
#pragma once
#include "internal.h"

namespace emfa {

constexpr int kNoPivW = 64;  // widest pivot-free panel
constexpr int kInvB = 256;   // size of the inverted diagonal blocks

// LU of the w x w diagonal block at (js, js), w <= 64, in place, with U^-1
// (64 x 64, row-major) in uinv and L^-1 in linv (row stride ldl).  ipiv gets the
// identity; flags[2] is raised on a zero pivot or a multiplier above sqrt(tau2).
emfa_status nopiv_diag_launch(hipStream_t s, cx<float> *A, long long lda, int js, int w, int *ipiv, int *flags,
                              float tau2, cx<float> *uinv, cx<float> *linv, long long ldl, const Batch &bt);

// Rows [js + w, N) of the panel: L21 = A21 U^-1; and the block's U rows for the
// columns [c0, c1): U12 = L^-1 A12, also written expanded into Bt (row stride
// ldbt) as the operand of the in-panel update.  c1 <= c0: L21 only.
emfa_status nopiv_rows_launch(hipStream_t s, cx<float> *A, long long lda, int js, int w, int N,
                              const cx<float> *uinv, const cx<float> *linv, long long ldl, int *flags, float tau2,
                              int c0, int c1, float *Bt, long long ldbt, const Batch &bt);

}  // namespace emfa
