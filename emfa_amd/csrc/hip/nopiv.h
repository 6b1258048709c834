// Kernels of FP32 factorisations without row interchanges and of the
// diagonal-block inverses of FP32 factors (nopiv.hip).  Launches run over the
// batch on blockIdx.z: A (and F) in the batch's matrices, the rest in its
// scratch slabs unless noted.
#pragma once
#include "internal.h"

namespace emfa {

constexpr int kNoPivW = 64;  // widest pivot-free panel
constexpr int kInvB = 256;   // size of the diagonal blocks that solves invert
constexpr int kURows = 256;  // most U rows of one launch

// LU of the w x w diagonal block at (js, js), w <= 64, in place, with U^-1
// and L^-1 - I (64 x 64, row-major) in uinv and linv.  ipiv gets the identity;
// flags[2] is raised on a zero pivot or a multiplier above sqrt(tau2).
emfa_status nopiv_diag_launch(hipStream_t s, cx<float> *A, long long lda, int js, int w, int *ipiv, int *flags,
                              float tau2, cx<float> *uinv, cx<float> *linv, const Batch &bt);

// Rows [js + w, N) of the panel: L21 = A21 U^-1; and the block's U rows for the
// columns [c0, c1) by substitution with L, also written expanded into Bt (row stride
// ldbt) as the operand of the in-panel update.  c1 <= c0: L21 only.
emfa_status nopiv_rows_launch(hipStream_t s, cx<float> *A, long long lda, int js, int w, int N,
                              const cx<float> *uinv, const cx<float> *linv, int *flags, float tau2, int c0, int c1,
                              float *Bt, long long ldbt, const Batch &bt);

// U rows of up to 256 rows of an outer block, in place: rows [r0, r0 + wb) of A,
// columns [c0, c1), by substitution with L's block there, also expanded into Bt at
// its complex K offset kofs (row stride ldbt).  linv: that block's 64 x 64 diagonal
// tiles' inverses as nopiv_diag_launch leaves them, one after another; cus: CUs to fill.
emfa_status nopiv_urows_launch(hipStream_t s, cx<float> *A, long long lda, int r0, int wb, int c0, int c1,
                               const cx<float> *linv, float *Bt, long long ldbt, int kofs, int cus, const Batch &bt);

// Inverses of the 256 x 256 diagonal blocks of an FP32 factor F (N x N): Dinv
// [2][nblk][256][256], L's (unit) then U's.  F in batch bf, Dinv in batch bd,
// both as matrices.
emfa_status dinv_f32_launch(hipStream_t s, const cx<float> *F, int N, cx<float> *Dinv, int nblk, const Batch &bf,
                            const Batch &bd);

}  // namespace emfa
