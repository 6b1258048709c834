// FP32 factorisations without row interchanges (refined in FP64 afterwards):
// the diagonal block, the panel's rows beside and below it, and inverses of
// triangular diagonal blocks.  Products run on V_MFMA_F32_16X16X4_F32: a
// complex product is a real one on the interleaved storage, the right
// operand's columns expanded in registers (real column 2j + p takes (p ? Im :
// Re) against Re A and (p ? Re : -Im) against Im A).  Lane group g (16 lanes)
// holds K = 8q + 2g, 8q + 2g + 1 of step q, one 16-byte load of A.
#include <algorithm>
#include <cmath>

#include "nopiv.h"

namespace emfa {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f4_a8 __attribute__((ext_vector_type(4), aligned(8)));
using cf = cx<float>;

// LDS row stride of 64-column tiles: rows 16 bytes apart modulo the 64 banks,
// so sixteen rows' 16-byte reads and a row's 64-byte reads are conflict-free
constexpr int kLd = 66;

__device__ __forceinline__ f4 mfma(float a, float b, f4 acc) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
}

// two complex steps of K: a = {A[.][k], A[.][k+1]}, x0 / x1 = column values
__device__ __forceinline__ f4 mac2(f4 acc, f4 a, cf x0, cf x1, bool odd) {
    acc = mfma(a.x, odd ? x0.im : x0.re, acc);
    acc = mfma(a.y, odd ? x0.re : -x0.im, acc);
    acc = mfma(a.z, odd ? x1.im : x1.re, acc);
    return mfma(a.w, odd ? x1.re : -x1.im, acc);
}

__device__ __forceinline__ float rlane(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

__device__ __forceinline__ void fms(cf &x, cf a, cf b) {  // x -= a b
    x.re = fmaf(-a.re, b.re, fmaf(a.im, b.im, x.re));
    x.im = fmaf(-a.re, b.im, fmaf(-a.im, b.re, x.im));
}

// A 64 x 64 triangular pair in LDS: the factored block and the inverses of its
// unit-lower and upper triangles, one array so that join64's operands are
// offsets.
struct Tri64 {
    cf m[3][64][kLd];  // S (L below the diagonal, U on and above), L^-1, U^-1
};
constexpr int kMat = 64 * kLd;

// The eight 8 x 8 diagonal blocks' inverses, one column per lane of the calling
// wave (lane = 8 block + column).  dinv: reciprocals of U's diagonal.
template <bool UPPER>
__device__ __forceinline__ void inv8(Tri64 &T, const cf *dinv, int lane) {
    const int o = lane & 56, col = lane & 7;
    const cf *S = &T.m[0][o][o];
    cf x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = {i == col ? 1.f : 0.f, 0.f};
    if (!UPPER) {
#pragma unroll
        for (int k = 0; k < 7; ++k)
#pragma unroll
            for (int i = k + 1; i < 8; ++i) fms(x[i], S[i * kLd + k], x[k]);
    } else {
#pragma unroll
        for (int k = 7; k >= 0; --k) {
            x[k] = cmul(x[k], dinv[o + k]);
#pragma unroll
            for (int i = 0; i < k; ++i) fms(x[i], S[i * kLd + k], x[k]);
        }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) T.m[UPPER ? 2 : 1][o + i][lane] = x[i];
}

// The inverses' off-diagonal blocks by sixteen waves, block pairs of b = 8, 16,
// 32 (L: X21 = -X22 L21 X11, U: X12 = -X11 U12 X22), each in two products of
// at most one 16 x 8 tile per wave and triangle.  The middle factors go into the
// 32 x 32 quadrant of X across the diagonal, which the caller ignores; the
// rest of X across the diagonal must be zero.  One rolled loop: the kernel
// runs once per launch, and every 64 bytes of code are a cold fetch.
// tris: 3 both, 1 L only, 2 U only.  All waves call it (it synchronises).
__device__ __forceinline__ void join64(Tri64 &T, int tris, int wave, int lane) {
    cf *M = &T.m[0][0][0];
    const int l16 = lane & 15, g = lane >> 4;
    const bool odd = l16 & 1;
#pragma nounroll
    for (int lb = 3; lb <= 5; ++lb) {
        const int b = 1 << lb, lt = lb == 5 ? 3 : 2;      // log2 jobs per triangle
        const int up = (wave >> lt) & 1, j = wave & ((1 << lt) - 1);
        const int p = lb == 3 ? j : lb == 4 ? j >> 1 : 0;  // pair
        const int r = lb == 5 ? 16 * (j >> 2) : 0, c = lb == 3 ? 0 : 8 * (lb == 4 ? j & 1 : j & 3);
        const int s0 = 2 * b * p, s1 = s0 + b, m = 32 + b * p;
        const bool act = (wave >> lt) < 2 && ((tris >> up) & 1);
        cf *X = M + (up ? 2 : 1) * kMat;
        // the middle factor, then the block: offsets of A's rows, B's rows and the result
#pragma nounroll
        for (int step = 0; step < 2; ++step) {
            const cf *A, *B;
            cf *O;
            // the triangular operand is zero outside k0 .. k1
            const int k0 = step == 0 ? (up ? 0 : c) : (up ? r : 0);
            const int k1 = step == 0 ? (up ? c + 8 : b) : (up ? b : min(b, r + 16));
            if (step == 0) {
                A = M + (up ? (s0 + r) * kLd + s1 : (s1 + r) * kLd + s0);
                B = X + (up ? s1 * kLd + s1 + c : s0 * kLd + s0 + c);
                O = X + (up ? (m + r) * kLd + c : r * kLd + m + c);
            } else {
                A = X + (up ? (s0 + r) * kLd + s0 : (s1 + r) * kLd + s1);
                B = X + (up ? m * kLd + c : m + c);
                O = X + (up ? (s0 + r) * kLd + s1 + c : (s1 + r) * kLd + s0 + c);
            }
            if (act) {
                const cf *Al = A + l16 * kLd + 2 * g, *Bl = B + 2 * g * kLd + (l16 >> 1);
                f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma nounroll
                for (int k = k0; k < k1; k += 8)
                    acc = mac2(acc, *(const f4 *)(Al + k), Bl[k * kLd], Bl[(k + 1) * kLd], odd);
                const float sign = step == 0 ? 1.f : -1.f;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (b > 8 || g < 2) ((float *)(O + (4 * g + i) * kLd))[l16] = sign * acc[i];
            }
            __syncthreads();
        }
    }
}

// ---------------------------------------------------------------------------
// Diagonal block: one workgroup of sixteen waves, lane = row, wave v holds
// columns 4v .. 4v + 3 in registers.  Column c's multipliers go through an LDS
// slot of their own and a progress counter (no barriers): a wave applies the
// columns before its own as they appear, pivot rows broadcast with
// v_readlane, then factors its four and publishes them one by one, so the
// next wave is about one column behind when it becomes the owner.  A wave
// issues one VALU instruction per 8 cycles however independent they are, so
// the chain is the owner's instruction count; what is not on it (the growth
// check, the diagonal's reciprocals) waits until its columns are published, and
// waves near their turn run at a higher priority.  Reciprocals are the
// hardware estimate (1 ulp): the factor is refined afterwards.
// Every wait is on an earlier wave of the same workgroup, which waits on
// earlier ones only.
// Then both 64 x 64 inverses: 8 x 8 blocks by substitution, one column per lane,
// joined on the matrix cores.
// 23 us per block (LU 14, inverses 6); 39 us with a barrier per four columns
// and one VALU inverse by doubling.
// ---------------------------------------------------------------------------
constexpr int kDiagThreads = 1024;

__global__ __launch_bounds__(kDiagThreads) void k_nopiv_diag(cf *__restrict__ A, long long lda, int js, int w,
                                                             int *__restrict__ ipiv, int *flags, float tau2,
                                                             cf *__restrict__ uinv, cf *__restrict__ linv,
                                                             long long ldl, Batch bt) {
    A = batch_mat(bt, A);
    ipiv = batch_scr(bt, ipiv);
    flags = batch_scr(bt, flags);
    uinv = batch_scr(bt, uinv);
    linv = batch_scr(bt, linv);
    __shared__ __attribute__((aligned(16))) Tri64 T;
    __shared__ cf Lc[64][64];  // multipliers of column c, zero on and above the diagonal
    __shared__ cf dinv[64];
    __shared__ int progress, s_bad;
    const int tid = threadIdx.x, lane = tid & 63, v = __builtin_amdgcn_readfirstlane(tid >> 6);
    cf a[4];
    {
        const cf *Ar = A + (size_t)(js + lane) * lda + js + 4 * v;
        if (w == 64) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const f4 x = *(const f4_a8 *)(Ar + 2 * q);
                a[2 * q] = {x.x, x.y};
                a[2 * q + 1] = {x.z, x.w};
            }
        } else {  // identity past the block
#pragma unroll
            for (int q = 0; q < 4; ++q)
                a[q] = (lane < w && 4 * v + q < w) ? Ar[q] : cf{lane == 4 * v + q ? 1.f : 0.f, 0.f};
        }
    }
    if (tid == 0) progress = s_bad = 0;
    for (int r = v; r < 64; r += 16) T.m[1][r][lane] = T.m[2][r][lane] = {0.f, 0.f};
    __syncthreads();
    // LDS operations of one wave complete in order: a counter read before the
    // data it covers, and data written before its counter, need no fence.  The
    // multipliers are read with the counter and used if it covers them.
    // (Atomic accesses: a volatile one goes through a flat instruction and waits.)
    for (int c = 0; c < 4 * v;) {
        if (c >= 4 * v - 4)
            __builtin_amdgcn_s_setprio(2);
        else if (c >= 4 * v - 12)
            __builtin_amdgcn_s_setprio(1);
        int avail = __hip_atomic_load(&progress, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        cf l = Lc[c][lane];
        avail = __builtin_amdgcn_readfirstlane(avail);
        if (avail <= c) {
            if (c < 4 * v - 4) __builtin_amdgcn_s_sleep(1);
            continue;
        }
        avail = min(avail, 4 * v);
        for (; c < avail; ++c) {
            const cf cur = l;
            if (c + 1 < avail) l = Lc[c + 1][lane];
#pragma unroll
            for (int q = 0; q < 4; ++q) fms(a[q], cur, cf{rlane(a[q].re, c), rlane(a[q].im, c)});
        }
    }
    __builtin_amdgcn_s_setprio(3);
    // The chain: pivot, reciprocal, multipliers, next own column.  Everything
    // else waits until the four columns are published.
    cf l[4], inv[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int c = 4 * v + q;
        const float pr = rlane(a[q].re, c), pi = rlane(a[q].im, c), rd = __builtin_amdgcn_rcpf(pr * pr + pi * pi);
        inv[q] = {pr * rd, -pi * rd};
        l[q] = cmul(a[q], inv[q]);
        l[q].re = lane > c ? l[q].re : 0.f;
        l[q].im = lane > c ? l[q].im : 0.f;
        Lc[c][lane] = l[q];
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __hip_atomic_store(&progress, c + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
#pragma unroll
        for (int t = q + 1; t < 4; ++t) fms(a[t], l[q], cf{rlane(a[t].re, c), rlane(a[t].im, c)});
    }
    bool bad = false;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int c = 4 * v + q;
        // a zero pivot makes its reciprocal infinite or not a number
        bad |= !(l[q].re * l[q].re + l[q].im * l[q].im <= tau2) || !(fabsf(inv[q].re) + fabsf(inv[q].im) < INFINITY);
        if (lane > c) a[q] = l[q];
        if (lane == 0) dinv[c] = inv[q];
    }
    __builtin_amdgcn_s_setprio(0);
#pragma unroll
    for (int q = 0; q < 2; ++q)
        *(f4 *)&T.m[0][lane][4 * v + 2 * q] = f4{a[2 * q].re, a[2 * q].im, a[2 * q + 1].re, a[2 * q + 1].im};
    if (bad) s_bad = 1;
    __syncthreads();
    if (v == 0)
        inv8<false>(T, dinv, lane);
    else if (v == 1)
        inv8<true>(T, dinv, lane);
    else if (tid >= 128 && tid < 128 + w)
        ipiv[js + tid - 128] = js + tid - 128;
    if (lane < w) {
        cf *Ar = A + (size_t)(js + lane) * lda + js + 4 * v;
        if (w == 64) {
#pragma unroll
            for (int q = 0; q < 2; ++q)
                *(f4_a8 *)(Ar + 2 * q) = f4{a[2 * q].re, a[2 * q].im, a[2 * q + 1].re, a[2 * q + 1].im};
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (4 * v + q < w) Ar[q] = a[q];
        }
    }
    __syncthreads();
    join64(T, 3, v, lane);
    for (int r = v; r < 64; r += 16) {
        uinv[(size_t)r * kNoPivW + lane] = lane >= r ? T.m[2][r][lane] : cf{0.f, 0.f};
        linv[(size_t)r * ldl + lane] = lane <= r ? T.m[1][r][lane] : cf{0.f, 0.f};
    }
    if (tid == 0 && s_bad) flags[2] = 1;
}

// ---------------------------------------------------------------------------
// The two products that follow the diagonal block, in one launch: workgroups
// [0, nl) form 16 rows of L21 = A21 U^-1 (a wave two of the eight column
// tiles), the others 16 columns of U12 = L^-1 A12 (a wave 16 of the 64 rows).
// In place: a workgroup's loads are done before its first store, and the
// workgroups touch disjoint parts of A.  K = 64 throughout: 64 MFMAs per wave
// behind one round of loads.  6.4 us per launch at 1920 unknowns; 17 us as a
// VALU product and substitution through LDS.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_nopiv_rows(cf *__restrict__ A, long long lda, int js, int w, int N,
                                                    const cf *__restrict__ uinv, const cf *__restrict__ linv,
                                                    long long ldl, int *flags, float tau2, int nl, int c0, int c1,
                                                    float *__restrict__ Bt, long long ldbt, Batch bt) {
    A = batch_mat(bt, A);
    uinv = batch_scr(bt, uinv);
    linv = batch_scr(bt, linv);
    flags = batch_scr(bt, flags);
    Bt = batch_scr(bt, Bt);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g = lane >> 4;
    const bool odd = l16 & 1, low = (int)blockIdx.x < nl;
    // rows of the left operand, columns of the right one
    const int r0 = low ? js + w + 16 * (int)blockIdx.x : 16 * wave;
    const int cb = low ? 16 * wave : c0 + 16 * ((int)blockIdx.x - nl);
    const cf *Ar = low ? A + (size_t)min(r0 + l16, N - 1) * lda + js : linv + (size_t)(r0 + l16) * ldl;
    f4 a[8];
    if (w == 64) {
#pragma unroll
        for (int q = 0; q < 8; ++q) a[q] = *(const f4_a8 *)(Ar + 8 * q + 2 * g);
    } else {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int k = 8 * q + 2 * g;
            const cf u = k < w ? Ar[k] : cf{0.f, 0.f}, v = k + 1 < w ? Ar[k + 1] : cf{0.f, 0.f};
            a[q] = f4{u.re, u.im, v.re, v.im};
        }
    }
    f4 acc[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int j = cb + 8 * t + (l16 >> 1);
        const cf *X = low ? uinv + j : A + (size_t)js * lda + min(j, c1 - 1);
        const long long ldx = low ? kNoPivW : lda;
        acc[t] = f4{0.f, 0.f, 0.f, 0.f};
        cf x[16];
#pragma unroll
        for (int q = 0; q < 8; ++q)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int k = 8 * q + 2 * g + h;
                x[2 * q + h] = k < w ? X[k * ldx] : cf{0.f, 0.f};
            }
#pragma unroll
        for (int q = 0; q < 8; ++q) acc[t] = mac2(acc[t], a[q], x[2 * q], x[2 * q + 1], odd);
    }
    __syncthreads();
    bool bad = false;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int j = cb + 8 * t + (l16 >> 1);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float v = acc[t][i], other = __shfl_xor(v, 1);
            const int r = r0 + 4 * g + i;
            if (low) {
                if (r < N && j < w) {
                    ((float *)(A + (size_t)r * lda + js + j))[odd] = v;
                    if (v * v + other * other > tau2) bad = true;
                }
            } else if (r < w && j < c1) {
                ((float *)(A + (size_t)(js + r) * lda + j))[odd] = v;
                // expanded operand: rows 2j {Re, -Im}, 2j + 1 {Im, Re}
                float *b = Bt + (2LL * (j - c0) + odd) * ldbt + 2 * r;
                b[0] = v;
                b[1] = odd ? other : -other;
            }
        }
    }
    if (bad) flags[2] = 1;
}

// ---------------------------------------------------------------------------
// Inverses of 256 x 256 diagonal blocks in three launches: every 64 x 64
// diagonal tile (k_inv_diag), then pairs of 64, then pairs of 128 (k_inv_join,
// one workgroup per 8 columns of a pair's off-diagonal block: the columns are
// independent, so both products of X21 = -X22 (L21 X11) stay in it): 31 us per
// factor whatever its size; 230 us with one VALU workgroup per 64 x 64 tile and
// a launch per sub-diagonal.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kDiagThreads) void k_inv_diag(const cf *__restrict__ F, int N, cf *__restrict__ Dinv,
                                                           int nblk, Batch bf, Batch bd) {
    __shared__ __attribute__((aligned(16))) Tri64 T;
    __shared__ cf dinv[64];
    F = batch_mat(bf, F);
    Dinv = batch_mat(bd, Dinv);
    const int blk = blockIdx.x >> 2, i = blockIdx.x & 3, r0 = blk * kInvB + 64 * i;
    const bool up = blockIdx.y != 0;
    const int tid = threadIdx.x, lane = tid & 63, v = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (r0 >= N) return;
    for (int r = v; r < 64; r += 16) {
        // identity past the matrix
        const cf d = (r0 + r < N && r0 + lane < N) ? F[(size_t)(r0 + r) * N + r0 + lane]
                                                   : cf{r == lane ? 1.f : 0.f, 0.f};
        T.m[0][r][lane] = d;
        T.m[up ? 2 : 1][r][lane] = {0.f, 0.f};
        if (r == lane) {
            const float den = d.re * d.re + d.im * d.im;
            dinv[r] = den > 0.f ? cf{d.re / den, -d.im / den} : cf{0.f, 0.f};
        }
    }
    __syncthreads();
    if (v == 0) {
        if (up)
            inv8<true>(T, dinv, lane);
        else
            inv8<false>(T, dinv, lane);
    }
    __syncthreads();
    join64(T, up ? 2 : 1, v, lane);
    cf *X = Dinv + (up ? (size_t)nblk * kInvB * kInvB : 0) + (size_t)blk * kInvB * kInvB + (size_t)64 * i * kInvB;
    for (int r = v; r < 64; r += 16) {
        X[(size_t)r * kInvB + 64 * i + lane] =
            (up ? lane >= r : lane <= r) ? T.m[up ? 2 : 1][r][lane] : cf{0.f, 0.f};
        for (int j = 0; j < 4; ++j)
            if (up ? j < i : j > i) X[(size_t)r * kInvB + 64 * j + lane] = {0.f, 0.f};
    }
}

template <int B>
__global__ __launch_bounds__(256) void k_inv_join(const cf *__restrict__ F, long long ldf, int N,
                                                  cf *__restrict__ Dinv, int nblk, int scr, Batch bf, Batch bd) {
    constexpr int STRIPS = B / 8, PAIRS = kInvB / (2 * B), RT = B / 64;  // 16-row tiles per wave
    __shared__ cf C[B][12];
    F = batch_mat(bf, F);
    Dinv = scr ? batch_scr(bd, Dinv) : batch_mat(bd, Dinv);
    const int c = 8 * ((int)blockIdx.x % STRIPS), pr = (int)blockIdx.x / STRIPS, blk = pr / PAIRS;
    const int s0 = 2 * B * (pr % PAIRS), s1 = s0 + B, r0 = blk * kInvB;
    const bool up = blockIdx.y != 0;
    if (r0 + s1 >= N) return;
    cf *X = Dinv + (up ? (size_t)nblk * kInvB * kInvB : 0) + (size_t)blk * kInvB * kInvB;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g = lane >> 4;
    const bool odd = l16 & 1;
    // rows fr.. and columns fc.. of F times the strip of X that starts at row xk
    const int fr = r0 + (up ? s0 : s1), fc = r0 + (up ? s1 : s0), xk = up ? s1 : s0;
    const int k0 = up ? 0 : c, k1 = up ? c + 8 : B;  // X's strip is zero outside
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        const int r = 16 * (RT * wave + t), row = fr + r + l16;
        const cf *Ar = F + (size_t)min(row, N - 1) * ldf + fc;
        const cf *Xs = X + (size_t)xk * kInvB + xk + c + (l16 >> 1);
        f4 acc = {0.f, 0.f, 0.f, 0.f};
        if (fr + B <= N && fc + B <= N) {
            // loads ahead of the products, 64 of K at a time; 64 x 64 tiles of X
            // across the diagonal hold nothing
#pragma unroll
            for (int h = 0; h < B; h += 64) {
                if (h >= k1 || h + 64 <= k0) continue;
#pragma unroll
                for (int k = h; k < h + 64; k += 8) {
                    const int ka = k + 2 * g;
                    acc = mac2(acc, *(const f4_a8 *)(Ar + ka), Xs[(size_t)ka * kInvB], Xs[(size_t)(ka + 1) * kInvB],
                               odd);
                }
            }
        } else {
            for (int k = k0; k < k1; k += 8) {
                const int ka = k + 2 * g;
                f4 a = {0.f, 0.f, 0.f, 0.f};
                if (row < N && fc + ka < N) {
                    a.x = Ar[ka].re;
                    a.y = Ar[ka].im;
                }
                if (row < N && fc + ka + 1 < N) {
                    a.z = Ar[ka + 1].re;
                    a.w = Ar[ka + 1].im;
                }
                acc = mac2(acc, a, Xs[(size_t)ka * kInvB], Xs[(size_t)(ka + 1) * kInvB], odd);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) ((float *)&C[r + 4 * g + i][0])[l16] = acc[i];
    }
    __syncthreads();
    const int orow = up ? s0 : s1, ocol = (up ? s1 : s0) + c;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        const int r = 16 * (RT * wave + t);
        const cf *Ar = X + (size_t)(orow + r + l16) * kInvB + orow;
        f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int h = 0; h < B; h += 64) {
            if (up ? h + 64 <= r : h > r) continue;
#pragma unroll
            for (int k = h; k < h + 64; k += 8) {
                const int ka = k + 2 * g;
                acc = mac2(acc, *(const f4 *)(Ar + ka), C[ka][l16 >> 1], C[ka + 1][l16 >> 1], odd);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) ((float *)(X + (size_t)(orow + r + 4 * g + i) * kInvB + ocol))[l16] = -acc[i];
    }
}

// ---------------------------------------------------------------------------
// U rows of a 256-row block: U = L^-1 A on its rows, for 8 CT columns per
// workgroup, in place (the columns go to LDS first).  Wave v takes 16-row
// tiles v and 15 - v, so the triangle's work is even.  Against the blocked
// substitution it replaces (per 64 rows one substitution and one update
// launch, 15 launches and 176 us per 512 rows at 1920 unknowns) it is one
// launch per 256 rows: 50 us with the update between the two.
// ---------------------------------------------------------------------------
template <int CT>
__global__ __launch_bounds__(512) void k_nopiv_urows(cf *__restrict__ A, long long lda, int r0, int wb, int c0,
                                                     int c1, const cf *__restrict__ Li, float *__restrict__ Bt,
                                                     long long ldbt, int kofs, Batch bt) {
    constexpr int S = 8 * CT;
    __shared__ cf Xs[kInvB][S + 4];
    A = batch_mat(bt, A);
    Li = batch_scr(bt, Li);
    Bt = batch_scr(bt, Bt);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g = lane >> 4;
    const bool odd = l16 & 1;
    const int cb = c0 + S * (int)blockIdx.x;
#pragma unroll 4
    for (int e = tid; e < kInvB * S; e += 512) {
        const int k = e / S, j = e % S;
        Xs[k][j] = (k < wb && cb + j < c1) ? A[(size_t)(r0 + k) * lda + cb + j] : cf{0.f, 0.f};
    }
    __syncthreads();
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        const int r = 16 * (half ? 15 - wave : wave);
        if (r >= wb) continue;
        const cf *Ar = Li + (size_t)(r + l16) * kInvB + 2 * g;
        f4 acc[CT], a[4];
#pragma unroll
        for (int t = 0; t < CT; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
        // steps of 32 of K, the next step's rows of L^-1 loaded ahead; the
        // last step may reach past the tile's diagonal, where L^-1 is zero
#pragma unroll
        for (int q = 0; q < 4; ++q) a[q] = *(const f4 *)(Ar + 8 * q);
        for (int k = 0; k < r + 16; k += 32) {
            f4 nx[4];
            const int kn = min(k + 32, kInvB - 32);
#pragma unroll
            for (int q = 0; q < 4; ++q) nx[q] = *(const f4 *)(Ar + kn + 8 * q);
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int t = 0; t < CT; ++t)
                    acc[t] = mac2(acc[t], a[q], Xs[k + 8 * q + 2 * g][8 * t + (l16 >> 1)],
                                  Xs[k + 8 * q + 2 * g + 1][8 * t + (l16 >> 1)], odd);
#pragma unroll
            for (int q = 0; q < 4; ++q) a[q] = nx[q];
        }
#pragma unroll
        for (int t = 0; t < CT; ++t) {
            const int j = cb + 8 * t + (l16 >> 1);
            float o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = __shfl_xor(acc[t][i], 1) * (odd ? 1.f : -1.f);
            if (j >= c1) continue;
            // expanded operand: rows 2j {Re, -Im}, 2j + 1 {Im, Re}
            float *b = Bt + (2LL * (j - c0) + odd) * ldbt + 2 * (kofs + r + 4 * g);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (r + 4 * g + i >= wb) continue;
                ((float *)(A + (size_t)(r0 + r + 4 * g + i) * lda + j))[odd] = acc[t][i];
                *(float2 *)(b + 2 * i) = make_float2(acc[t][i], o[i]);
            }
        }
    }
}

}  // namespace

emfa_status nopiv_diag_launch(hipStream_t s, cf *A, long long lda, int js, int w, int *ipiv, int *flags, float tau2,
                              cf *uinv, cf *linv, long long ldl, const Batch &bt) {
    EMFA_REQUIRE(w >= 1 && w <= kNoPivW && ldl >= kNoPivW, EMFA_E_INVALID, "pivot-free panel of width %d", w);
    k_nopiv_diag<<<dim3(1, 1, bt.count), kDiagThreads, 0, s>>>(A, lda, js, w, ipiv, flags, tau2, uinv, linv, ldl, bt);
    EMFA_HIP_CHECK(hipGetLastError());
    return EMFA_OK;
}

emfa_status nopiv_rows_launch(hipStream_t s, cf *A, long long lda, int js, int w, int N, const cf *uinv,
                              const cf *linv, long long ldl, int *flags, float tau2, int c0, int c1, float *Bt,
                              long long ldbt, const Batch &bt) {
    const int nl = (N - js - w + 15) / 16, nu = std::max(0, (c1 - c0 + 15) / 16);
    if (nl + nu <= 0) return EMFA_OK;
    k_nopiv_rows<<<dim3(nl + nu, 1, bt.count), 256, 0, s>>>(A, lda, js, w, N, uinv, linv, ldl, flags, tau2, nl, c0,
                                                            c1, Bt, ldbt, bt);
    EMFA_HIP_CHECK(hipGetLastError());
    return EMFA_OK;
}

emfa_status nopiv_linv_launch(hipStream_t s, const cf *F, long long ldf, int n, cf *Li, const Batch &bt) {
    const int nblk = (n + kInvB - 1) / kInvB;
    if (n > 64) k_inv_join<64><<<dim3(nblk * 16, 1, bt.count), 256, 0, s>>>(F, ldf, n, Li, nblk, 1, bt, bt);
    if (n > 128) k_inv_join<128><<<dim3(nblk * 16, 1, bt.count), 256, 0, s>>>(F, ldf, n, Li, nblk, 1, bt, bt);
    EMFA_HIP_CHECK(hipGetLastError());
    return EMFA_OK;
}

emfa_status nopiv_urows_launch(hipStream_t s, cf *A, long long lda, int r0, int wb, int c0, int c1, const cf *Li,
                               float *Bt, long long ldbt, int kofs, const Batch &bt) {
    if (c1 <= c0 || wb <= 0) return EMFA_OK;
    EMFA_REQUIRE(wb <= kInvB, EMFA_E_INVALID, "U rows of a block of %d", wb);
    const int nc = c1 - c0;
    // Wider strips read L^-1 fewer times, narrower ones have the shorter chain:
    // 8 columns while they fill the chip at most twice over (1920 unknowns: 15.6
    // us per launch, 16 columns 22.5)
    const long long cols = (long long)nc * bt.count;
    auto go = [&](auto kernel, int strip) {
        kernel<<<dim3((nc + strip - 1) / strip, 1, bt.count), 512, 0, s>>>(A, lda, r0, wb, c0, c1, Li, Bt, ldbt, kofs,
                                                                          bt);
    };
    if (cols >= 16384)
        go(k_nopiv_urows<4>, 32);
    else if (cols >= 4096)
        go(k_nopiv_urows<2>, 16);
    else
        go(k_nopiv_urows<1>, 8);
    EMFA_HIP_CHECK(hipGetLastError());
    return EMFA_OK;
}

emfa_status dinv_f32_launch(hipStream_t s, const cf *F, int N, cf *Dinv, int nblk, const Batch &bf, const Batch &bd) {
    k_inv_diag<<<dim3(nblk * 4, 2, bf.count), kDiagThreads, 0, s>>>(F, N, Dinv, nblk, bf, bd);
    k_inv_join<64><<<dim3(nblk * 16, 2, bf.count), 256, 0, s>>>(F, N, N, Dinv, nblk, 0, bf, bd);
    k_inv_join<128><<<dim3(nblk * 16, 2, bf.count), 256, 0, s>>>(F, N, N, Dinv, nblk, 0, bf, bd);
    EMFA_HIP_CHECK(hipGetLastError());
    return EMFA_OK;
}

}  // namespace emfa
