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

// two complex steps of K: a = {A[.][k], A[.][k+1]}, x0 / x1 = column values.  One
// sum in K's order: in products with the inverse of a block of large multipliers
// neighbouring terms cancel, and two sums of half the terms each made factors 2
// to 3 times less accurate.
__device__ __forceinline__ void mac2(f4 &acc, f4 a, cf x0, cf x1, bool odd) {
    acc = mfma(a.x, odd ? x0.im : x0.re, acc);
    acc = mfma(a.y, odd ? x0.re : -x0.im, acc);
    acc = mfma(a.z, odd ? x1.im : x1.re, acc);
    acc = mfma(a.w, odd ? x1.re : -x1.im, acc);
}

__device__ __forceinline__ float rlane(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// x -= a b, the product formed first: one rounding per part at x's size (two
// fused steps into x, an instruction less, round twice there: 1.4 times the
// error of a diagonal block)
__device__ __forceinline__ void fms(cf &x, cf a, cf b) {
    x.re -= fmaf(a.re, b.re, -(a.im * b.im));
    x.im -= fmaf(a.re, b.im, a.im * b.re);
}

// Orders a wave's own LDS accesses: its lanes read what other lanes of it wrote.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Forward substitution with a unit-lower 64 x 64 block for 8 complex columns by
// one wave, 16 rows at a time: the tiles below the diagonal and the inverses of
// the 16 x 16 diagonal tiles less the identity, as left operands.  Inverses no
// larger than 16 keep the error at |L| |U| as substitution by single rows has
// it; a 256-row inverse in its place (U = L^-1 A) made factors of matrices with
// multipliers of 10 to 90 four to eight times less accurate at 1100 unknowns.
struct Sub64 {
    f4 d[4][2], l[6][2];

    // L: the factored block (w x w), inv: L^-1 - I (64 x 64)
    __device__ __forceinline__ void load(const cf *L, long long ldl, const cf *inv, int w, int lane) {
        const int l16 = lane & 15, g = lane >> 4;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int q = 0; q < 2; ++q)
                d[i][q] = *(const f4 *)(inv + (16 * i + l16) * kNoPivW + 16 * i + 8 * q + 2 * g);
        // rows past the block read its last one and count as zero
#pragma unroll
        for (int b = 1; b < 4; ++b) {
            const cf *Lr = L + min(16 * b + l16, w - 1) * ldl + 2 * g;
#pragma unroll
            for (int i = 0; i < b; ++i)
#pragma unroll
                for (int q = 0; q < 2; ++q) l[b * (b - 1) / 2 + i][q] = *(const f4_a8 *)(Lr + 16 * i + 8 * q);
        }
        if (w < 64) {
#pragma unroll
            for (int b = 1; b < 4; ++b)
#pragma unroll
                for (int i = 0; i < 2 * b; ++i)
                    if (16 * b + l16 >= w) l[b * (b - 1) / 2 + (i >> 1)][i & 1] = f4{0.f, 0.f, 0.f, 0.f};
        }
    }

    // v: the columns, tile i holding rows 16 i + 4 g + r, real column l16; X: 64
    // rows of 8 columns in LDS (row stride ldx), left with the result as v is
    __device__ __forceinline__ void solve(f4 *v, cf *X, int ldx, int lane) const {
        const int l16 = lane & 15, g = lane >> 4;
        const bool odd = l16 & 1;
        f4 p[4];
        cf x[4], y[4];  // a tile's rows and those of the last finished tile, as right operands
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = f4{0.f, 0.f, 0.f, 0.f};
        auto turn = [&](int i, cf *o) {
            cf *Xi = X + 16 * i * ldx;
            wave_sync();
#pragma unroll
            for (int r = 0; r < 4; ++r) ((float *)(Xi + (4 * g + r) * ldx))[l16] = v[i][r];
            wave_sync();
#pragma unroll
            for (int h = 0; h < 4; ++h) o[h] = Xi[(8 * (h >> 1) + 2 * g + (h & 1)) * ldx + (l16 >> 1)];
        };
        auto off = [&](int b, int i) {  // p[b] += L's tile (b, i) times tile i
#pragma unroll
            for (int q = 0; q < 2; ++q) mac2(p[b], l[b * (b - 1) / 2 + i][q], y[2 * q], y[2 * q + 1], odd);
        };
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (i) off(i, i - 1);
            v[i] -= p[i];
            turn(i, x);
            // behind the trip through LDS
#pragma unroll
            for (int b = i + 1; i && b < 4; ++b) off(b, i - 1);
            f4 e = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < 2; ++q) mac2(e, d[i][q], x[2 * q], x[2 * q + 1], odd);
            v[i] += e;
            turn(i, y);
        }
    }
};

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
// tris: 3 both, 1 L only, 2 U only; L's inverse as far as blocks of lmax.  All
// waves call it (it synchronises).
__device__ __forceinline__ void join64(Tri64 &T, int tris, int lmax, int wave, int lane) {
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
        const bool act = (wave >> lt) < 2 && ((tris >> up) & 1) && (up || 2 * b <= lmax);
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
                    mac2(acc, *(const f4 *)(Al + k), Bl[k * kLd], Bl[(k + 1) * kLd], odd);
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
// 22 us per block (LU 15, inverses 6); 39 us with a barrier per four columns
// and one VALU inverse by doubling.
// ---------------------------------------------------------------------------
constexpr int kDiagThreads = 1024;

__global__ __launch_bounds__(kDiagThreads) void k_nopiv_diag(cf *__restrict__ A, long long lda, int js, int w,
                                                             int *__restrict__ ipiv, int *flags, float tau2,
                                                             cf *__restrict__ uinv, cf *__restrict__ linv, Batch bt) {
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
    float corr[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int c = 4 * v + q;
        const float pr = rlane(a[q].re, c), pi = rlane(a[q].im, c), den = pr * pr + pi * pi;
        const float rd = __builtin_amdgcn_rcpf(den);
        corr[q] = fmaf(-den, rd, 1.f);
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
        // the estimate's Newton step: an error here is common to a whole column of L21
        if (lane == 0) dinv[c] = {fmaf(inv[q].re, corr[q], inv[q].re), fmaf(inv[q].im, corr[q], inv[q].im)};
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
    join64(T, 3, 16, v, lane);
    for (int r = v; r < 64; r += 16) {
        uinv[(size_t)r * kNoPivW + lane] = lane >= r ? T.m[2][r][lane] : cf{0.f, 0.f};
        linv[(size_t)r * kNoPivW + lane] = lane < r ? T.m[1][r][lane] : cf{0.f, 0.f};
    }
    if (tid == 0 && s_bad) flags[2] = 1;
}

// ---------------------------------------------------------------------------
// What follows the diagonal block, in one launch: workgroups [0, nu), whose chain
// is the longer one, form 32 columns of U12 by substitution with L (a wave 8
// columns), the others 16 rows of L21 = A21 U^-1 (a wave two of the eight column
// tiles, K = 64: 64 MFMAs behind one round of loads).  In place: a workgroup's
// (U12: a wave's) loads are done before its first store, and they touch disjoint
// parts of A.  8.0 us per launch at 1920 unknowns (6.4 with U12 = L^-1 A12 by an
// explicit inverse, 17 as a VALU product and substitution through LDS).
// ---------------------------------------------------------------------------
constexpr int kSubLd = 10;  // sixteen lanes' rows four apart on different banks

__global__ __launch_bounds__(256) void k_nopiv_rows(cf *__restrict__ A, long long lda, int js, int w, int N,
                                                    const cf *__restrict__ uinv, const cf *__restrict__ linv,
                                                    int *flags, float tau2, int nu, int c0, int c1,
                                                    float *__restrict__ Bt, long long ldbt, Batch bt) {
    __shared__ cf Xs[4][64 * kSubLd];
    A = batch_mat(bt, A);
    uinv = batch_scr(bt, uinv);
    linv = batch_scr(bt, linv);
    flags = batch_scr(bt, flags);
    Bt = batch_scr(bt, Bt);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g = lane >> 4;
    const bool odd = l16 & 1;
    if ((int)blockIdx.x < nu) {
        const int cb = c0 + 32 * (int)blockIdx.x + 8 * wave, j = cb + (l16 >> 1);
        if (cb >= c1) return;
        Sub64 op;
        op.load(A + (size_t)js * lda + js, lda, linv, w, lane);
        f4 v[4];
        const float *Aj = (const float *)(A + (size_t)js * lda + min(j, c1 - 1)) + odd;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * i + 4 * g + r;
                const float x = Aj[2 * min(row, w - 1) * lda];
                v[i][r] = row < w ? x : 0.f;
            }
        op.solve(v, Xs[wave], kSubLd, lane);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * i + 4 * g + r;
                const float x = v[i][r], other = __shfl_xor(x, 1);
                if (row >= w || j >= c1) continue;
                ((float *)(A + (size_t)(js + row) * lda + j))[odd] = x;
                // expanded operand: rows 2j {Re, -Im}, 2j + 1 {Im, Re}
                *(float2 *)(Bt + (2LL * (j - c0) + odd) * ldbt + 2 * row) = make_float2(x, odd ? other : -other);
            }
        return;
    }
    const int r0 = js + w + 16 * ((int)blockIdx.x - nu);
    const cf *Ar = A + (size_t)min(r0 + l16, N - 1) * lda + js;
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
        const cf *X = uinv + 16 * wave + 8 * t + (l16 >> 1);
        acc[t] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int k = 8 * q + 2 * g;
            mac2(acc[t], a[q], X[k * kNoPivW], X[(k + 1) * kNoPivW], odd);
        }
    }
    __syncthreads();
    bool bad = false;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int j = 16 * wave + 8 * t + (l16 >> 1);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float v = acc[t][i], other = __shfl_xor(v, 1);
            const int r = r0 + 4 * g + i;
            if (r >= N || j >= w) continue;
            ((float *)(A + (size_t)r * lda + js + j))[odd] = v;
            if (v * v + other * other > tau2) bad = true;
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
    join64(T, up ? 2 : 1, 64, v, lane);
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
                                                  cf *__restrict__ Dinv, int nblk, Batch bf, Batch bd) {
    constexpr int STRIPS = B / 8, PAIRS = kInvB / (2 * B), RT = B / 64;  // 16-row tiles per wave
    __shared__ cf C[B][12];
    F = batch_mat(bf, F);
    Dinv = batch_mat(bd, Dinv);
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
                    mac2(acc, *(const f4_a8 *)(Ar + ka), Xs[(size_t)ka * kInvB], Xs[(size_t)(ka + 1) * kInvB], odd);
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
                mac2(acc, a, Xs[(size_t)ka * kInvB], Xs[(size_t)(ka + 1) * kInvB], odd);
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
                mac2(acc, *(const f4 *)(Ar + ka), C[ka][l16 >> 1], C[ka + 1][l16 >> 1], odd);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) ((float *)(X + (size_t)(orow + r + 4 * g + i) * kInvB + ocol))[l16] = -acc[i];
    }
}

// ---------------------------------------------------------------------------
// U rows of a 256-row block by substitution with L, for 8 CT columns per
// workgroup, in place (the columns in LDS): per 64 rows a wave and column tile
// substitutes (Sub64) while the other waves take the last 64 rows' part off the
// tiles below.  Wave v owns the 16-row tiles v and 15 - v, so the triangle's
// work is even.
// A chain of four substitutions: 21 us per launch at 1920 unknowns, where the
// product with L's explicit inverse took 15 and that inverse 20 more per block,
// and blocked substitution in launches of 64 rows 176 us per 512 rows.  Strips of
// up to 16 columns run in one round, one workgroup a CU: L's tiles and the
// substitution's operands are loaded a block ahead.  Strips of 32, in several
// rounds, take half the registers instead and come two to a CU: 30720 unknowns 121
// -> 105 us per launch, 8321 44 -> 48.
// ---------------------------------------------------------------------------
template <int CT>
__global__ __launch_bounds__(512, CT == 4 ? 4 : 2) void k_nopiv_urows(cf *__restrict__ A, long long lda, int r0, int wb, int c0,
                                                     int c1, const cf *__restrict__ linv, float *__restrict__ Bt,
                                                     long long ldbt, int kofs, Batch bt) {
    constexpr int S = 8 * CT, LD = S + 2;
    constexpr bool kAhead = CT < 4;
    __shared__ cf Xs[kURows * LD];
    A = batch_mat(bt, A);
    linv = batch_scr(bt, linv);
    Bt = batch_scr(bt, Bt);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15,
              g = lane >> 4;
    const bool odd = l16 & 1;
    const int cb = c0 + S * (int)blockIdx.x, nc = min(S, c1 - cb);
    const cf *L = A + (size_t)r0 * lda + r0;
    const int tile[2] = {wave, 15 - wave}, solver = wave - (8 - CT);  // column tile that the wave substitutes
    const int nst = (wb + 63) / 64;
    f4 l[kAhead ? 2 : 1][8];
    Sub64 op;
    // L's tile in block column s
    auto load_l = [&](int h, int s) {
        const cf *Lr = L + (size_t)min(16 * tile[h] + l16, wb - 1) * lda + 64 * s + 2 * g;
#pragma unroll
        for (int q = 0; q < 8; ++q) l[kAhead ? h : 0][q] = *(const f4_a8 *)(Lr + 8 * q);
    };
    auto load_op = [&](int s) {
        op.load(L + (size_t)64 * s * lda + 64 * s, lda, linv + (size_t)s * kNoPivW * kNoPivW,
                min(64, wb - 64 * s), lane);
    };
    // the tile's columns less L's tile times the rows of block s
    auto update = [&](int h, int s) {
        const cf *X = Xs + (64 * s + 2 * g) * LD + (l16 >> 1);
        if (!kAhead) load_l(h, s);
#pragma unroll
        for (int t = 0; t < CT; ++t) {
            f4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < 8; ++q) mac2(p, l[kAhead ? h : 0][q], X[8 * q * LD + 8 * t], X[(8 * q + 1) * LD + 8 * t], odd);
#pragma unroll
            for (int i = 0; i < 4; ++i) ((float *)(Xs + (16 * tile[h] + 4 * g + i) * LD + 8 * t))[l16] -= p[i];
        }
    };
    if (kAhead && solver >= 0) load_op(0);
    {
        cf x[kURows * S / 512];
#pragma unroll
        for (int i = 0; i < kURows * S / 512; ++i) {
            const int e = tid + 512 * i;
            x[i] = A[(size_t)(r0 + min(e / S, wb - 1)) * lda + cb + min(e % S, nc - 1)];
        }
#pragma unroll
        for (int i = 0; i < kURows * S / 512; ++i) {
            const int e = tid + 512 * i;
            Xs[e / S * LD + e % S] = (e / S < wb && e % S < nc) ? x[i] : cf{0.f, 0.f};
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
        if (kAhead && tile[h] >= 4 && 16 * tile[h] < wb) load_l(h, 0);
    __syncthreads();
    for (int s = 0; s < nst; ++s) {
        if (s) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (tile[h] >> 2 == s && 16 * tile[h] < wb) update(h, s - 1);
            __syncthreads();
        }
        if (solver >= 0) {
            if (!kAhead) load_op(s);
            cf *X = Xs + 64 * s * LD + 8 * solver;
            f4 v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) v[i][r] = ((const float *)(X + (16 * i + 4 * g + r) * LD))[l16];
            op.solve(v, X, LD, lane);
            if (kAhead && s + 1 < nst) load_op(s + 1);
        }
        // beside it, the tiles of later blocks
        if (s) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (tile[h] >> 2 > s && 16 * tile[h] < wb) {
                    update(h, s - 1);
                    if (kAhead) load_l(h, s);
                }
        }
        __syncthreads();
    }
    for (int e = tid; e < wb * S; e += 512) {
        const int k = e / S, j = e % S;
        if (j < nc) A[(size_t)(r0 + k) * lda + cb + j] = Xs[k * LD + j];
    }
    // expanded operand: rows 2j {Re, -Im}, 2j + 1 {Im, Re}
    for (int j = wave; j < nc; j += 8)
        for (int k = lane; k < wb; k += 64) {
            const cf x = Xs[k * LD + j];
            float *b = Bt + 2LL * (cb - c0 + j) * ldbt + 2 * (kofs + k);
            *(float2 *)b = make_float2(x.re, -x.im);
            *(float2 *)(b + ldbt) = make_float2(x.im, x.re);
        }
}

}  // namespace

emfa_status nopiv_diag_launch(hipStream_t s, cf *A, long long lda, int js, int w, int *ipiv, int *flags, float tau2,
                              cf *uinv, cf *linv, const Batch &bt) {
    EMFA_REQUIRE(w >= 1 && w <= kNoPivW, EMFA_E_INVALID, "pivot-free panel of width %d", w);
    k_nopiv_diag<<<dim3(1, 1, bt.count), kDiagThreads, 0, s>>>(A, lda, js, w, ipiv, flags, tau2, uinv, linv, bt);
    EMFA_HIP_CHECK(hipGetLastError());
    return EMFA_OK;
}

emfa_status nopiv_rows_launch(hipStream_t s, cf *A, long long lda, int js, int w, int N, const cf *uinv,
                              const cf *linv, int *flags, float tau2, int c0, int c1, float *Bt, long long ldbt,
                              const Batch &bt) {
    const int nl = (N - js - w + 15) / 16, nu = std::max(0, (c1 - c0 + 31) / 32);
    if (nl + nu <= 0) return EMFA_OK;
    k_nopiv_rows<<<dim3(nl + nu, 1, bt.count), 256, 0, s>>>(A, lda, js, w, N, uinv, linv, flags, tau2, nu, c0, c1, Bt,
                                                            ldbt, bt);
    EMFA_HIP_CHECK(hipGetLastError());
    return EMFA_OK;
}

emfa_status nopiv_urows_launch(hipStream_t s, cf *A, long long lda, int r0, int wb, int c0, int c1, const cf *linv,
                               float *Bt, long long ldbt, int kofs, int cus, const Batch &bt) {
    if (c1 <= c0 || wb <= 0) return EMFA_OK;
    EMFA_REQUIRE(wb <= kURows, EMFA_E_INVALID, "U rows of a block of %d", wb);
    const int nc = c1 - c0;
    // A strip's time is its chain's (8, 16, 32 columns 21, 29, 48 us alone), and a
    // CU holds one workgroup (two of the widest): the narrowest strips that run in
    // one round.  In factorisations of 1920 / 8321 / 30720 unknowns all strips of 8 columns take
    // 2.20 / 19.2 / 388 ms, of 16 2.26 / 19.0 / 382, of 32 2.28 / 18.9 / 381.
    const long long cols = (long long)nc * bt.count;
    auto go = [&](auto kernel, int strip) {
        kernel<<<dim3((nc + strip - 1) / strip, 1, bt.count), 512, 0, s>>>(A, lda, r0, wb, c0, c1, linv, Bt, ldbt, kofs,
                                                                          bt);
    };
    if (cols > 16LL * cus)
        go(k_nopiv_urows<4>, 32);
    else if (cols > 8LL * cus)
        go(k_nopiv_urows<2>, 16);
    else
        go(k_nopiv_urows<1>, 8);
    EMFA_HIP_CHECK(hipGetLastError());
    return EMFA_OK;
}

emfa_status dinv_f32_launch(hipStream_t s, const cf *F, int N, cf *Dinv, int nblk, const Batch &bf, const Batch &bd) {
    k_inv_diag<<<dim3(nblk * 4, 2, bf.count), kDiagThreads, 0, s>>>(F, N, Dinv, nblk, bf, bd);
    k_inv_join<64><<<dim3(nblk * 16, 2, bf.count), 256, 0, s>>>(F, N, N, Dinv, nblk, bf, bd);
    k_inv_join<128><<<dim3(nblk * 16, 2, bf.count), 256, 0, s>>>(F, N, N, Dinv, nblk, bf, bd);
    EMFA_HIP_CHECK(hipGetLastError());
    return EMFA_OK;
}

}  // namespace emfa
