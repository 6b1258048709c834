// Complex products with few columns on the matrix cores: the steps of a
// triangular solve with few right-hand sides and the refinement residual.
//
//   C (M x m) = beta C + sign A (M x K) X (K x m)      (P == null)
//   plane z of P = A X over K slice [z kc, (z + 1) kc)  (P given)
//
// A workgroup forms 16 RT rows x 8 CT columns.  Its four waves split K: in a
// chunk of 16 KL, wave w and 16-lane group g hold KL consecutive complex
// values of their row (straight from memory, A is read once per column
// group), so MFMA t of a chunk multiplies the t-th real of each lane's run.  The
// complex product is a real one with X's columns expanded in registers: real
// column 2j + p takes (p ? Im : Re) against Re A and (p ? Re : -Im) against
// Im A.  Partial tiles are added through LDS in wave order.  An entry's sum
// depends on K and the slice only, never on m or the tile, so a column has the
// same bits in every block of right-hand sides that takes this route with the
// same slices (a residual's are the same up to 64 columns).  A second job shares the launch
// (workgroups from tiles0 on) when it writes other rows and reads nothing
// that the first one writes.
//
// These products are latency chains, not throughput: at 256 x 256 x 32 FP32
// (one diagonal block of a 32-column solve) the time is the loads' latency
// plus 32 MFMAs per column tile and wave; K split over waves and column tiles
// over workgroups keep that chain short.  Against the VALU product through
// LDS that it replaced (19 us per launch whatever the size): a refined FP32
// factorisation of 1920 unknowns with 24 right-hand sides 4.57 -> 3.70 ms,
// of 8321 with 49 36.7 -> 26.3 ms (its FP64 residual 2.8 -> 1.1 ms, with two
// row tiles and more slices 0.8), eight of 1920 unknowns 22.0 -> 11.4 ms.
#include <algorithm>
#include <type_traits>

#include "gemm.h"

namespace emfa {

namespace {

template <typename T>
struct Vec4;
template <>
struct Vec4<float> {
    typedef float type __attribute__((ext_vector_type(4)));
};
template <>
struct Vec4<double> {
    typedef double type __attribute__((ext_vector_type(4)));
};

// 16 bytes of FP32 at 8-byte alignment (rows of an odd-sized matrix)
typedef float float4_a8 __attribute__((ext_vector_type(4), aligned(8)));

__device__ __forceinline__ void mfma4(Vec4<float>::type &acc, float a, float b) {
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
}
__device__ __forceinline__ void mfma4(Vec4<double>::type &acc, double a, double b) {
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
}
// row of result element v in lane group g: V_MFMA_F32_16X16X4_F32 holds
// 4 g + v, V_MFMA_F64_16X16X4_F64 g + 4 v
__device__ __forceinline__ int mfma4_row(float, int g, int v) { return 4 * g + v; }
__device__ __forceinline__ int mfma4_row(double, int g, int v) { return g + 4 * v; }

template <typename TA, typename TC, int RT, int CT>
__global__ __launch_bounds__(256) void k_skinny(SkinnyJob<TA, TC> job0, SkinnyJob<TA, TC> job1, int tiles0, int m,
                                                int kc, cx<TC> *P) {
    constexpr int KL = sizeof(TC) == 4 ? 16 / RT : 8 / RT;  // complex values of K per lane and step
    constexpr int KC = sizeof(TC) == 4 ? 16 : 8;            // ... and chunk
    constexpr int NR = 16 * RT, NC = 16 * CT;               // rows and real columns of the tile
    constexpr int OUT = 16 * NC / 256;                      // outputs per thread and 16 rows
    __shared__ TC red[4][16][NC + 1];
    using V4 = typename Vec4<TC>::type;
    const bool second = (int)blockIdx.x >= tiles0;
    const SkinnyJob<TA, TC> &g = second ? job1 : job0;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, grp = lane >> 4;
    const int r0 = ((int)blockIdx.x - (second ? tiles0 : 0)) * NR, j0 = blockIdx.y * 8 * CT, z = blockIdx.z;
    const int M = g.M, kb = z * kc, ke = min(g.K, kb + kc);
    const long long ldx = g.ldx;
    const cx<TA> *__restrict__ Ar[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) Ar[rt] = g.A + (long long)min(r0 + 16 * rt + l16, M - 1) * g.lda;
    const bool odd = l16 & 1;
    // the outputs' old values are on their way during the product
    TC old[RT][OUT];
    if (!P) {
#pragma unroll
        for (int i = 0; i < RT * OUT; ++i) {
            const int e = tid + 256 * i, r = r0 + e / NC, c = 2 * j0 + e % NC;
            old[i / OUT][i % OUT] = (g.beta && r < M && c < 2 * m) ? ((const TC *)(g.C + (long long)r * g.ldc))[c] : TC(0);
        }
    }
    V4 acc[RT][CT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = V4{TC(0), TC(0), TC(0), TC(0)};
    for (int k0 = kb; k0 < ke; k0 += 16 * KC) {
        if (k0 + 4 * wave * KC >= ke) break;  // uniform in the wave
        const bool full = k0 + 4 * (wave + 1) * KC <= ke;
#pragma unroll
        for (int st = 0; st < RT; ++st) {
            const int kw = k0 + (4 * wave + grp) * KC + st * KL;  // this lane's run of K
            cx<TA> a[RT][KL];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                if (full && sizeof(TA) == 4) {
#pragma unroll
                    for (int i = 0; i < KL / 2; ++i) {
                        const float4_a8 v = ((const float4_a8 *)(Ar[rt] + kw))[i];
                        a[rt][2 * i] = {(TA)v.x, (TA)v.y};
                        a[rt][2 * i + 1] = {(TA)v.z, (TA)v.w};
                    }
                } else if (full) {
#pragma unroll
                    for (int i = 0; i < KL; ++i) a[rt][i] = Ar[rt][kw + i];
                } else {
#pragma unroll
                    for (int i = 0; i < KL; ++i) a[rt][i] = kw + i < ke ? Ar[rt][kw + i] : cx<TA>{TA(0), TA(0)};
                }
            }
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                const cx<TC> *__restrict__ Xj = g.X + min(j0 + 8 * ct + (l16 >> 1), m - 1);
                cx<TC> x[KL];
#pragma unroll
                for (int i = 0; i < KL; ++i) {
                    const bool in = full || kw + i < ke;
                    x[i] = in ? Xj[(long long)(kw + i) * ldx] : cx<TC>{TC(0), TC(0)};
                }
#pragma unroll
                for (int i = 0; i < KL; ++i)
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt) {
                        mfma4(acc[rt][ct], (TC)a[rt][i].re, odd ? x[i].im : x[i].re);
                        mfma4(acc[rt][ct], (TC)a[rt][i].im, odd ? x[i].re : -x[i].im);
                    }
            }
        }
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        if (rt) __syncthreads();
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int v = 0; v < 4; ++v) red[wave][mfma4_row(TC(0), grp, v)][16 * ct + l16] = acc[rt][ct][v];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < OUT; ++i) {
            const int e = tid + 256 * i, rr = e / NC, cc = e % NC, r = r0 + 16 * rt + rr, c = 2 * j0 + cc;
            if (r >= M || c >= 2 * m) continue;
            const TC v = ((red[0][rr][cc] + red[1][rr][cc]) + red[2][rr][cc]) + red[3][rr][cc];
            if (P)
                ((TC *)(P + (long long)z * M * m + (long long)r * m))[c] = v;
            else
                ((TC *)(g.C + (long long)r * g.ldc))[c] = old[rt][i] + g.sign * v;
        }
    }
}

template <typename TA, typename TC>
emfa_status launch(hipStream_t s, const SkinnyJob<TA, TC> &j0, const SkinnyJob<TA, TC> *second, int m, int slices,
                   int kc, cx<TC> *P) {
    SkinnyJob<TA, TC> j1 = second ? *second : SkinnyJob<TA, TC>();
    EMFA_REQUIRE(m > 0 && j0.M >= 0 && j1.M >= 0 && j0.K > 0, EMFA_E_INVALID, "skinny product: bad shape");
    EMFA_REQUIRE(slices >= 1 && slices <= 65535 && kc > 0 && (long long)slices * kc >= std::max(j0.K, j1.K) &&
                     (P ? !second : slices == 1),
                 EMFA_E_INVALID, "skinny product: bad slices %d x %d for K=%d", slices, kc, j0.K);
    if (j0.M + j1.M == 0) return EMFA_OK;
    auto wgs = [&](int rt, int ct) {
        return (long long)((j0.M + 16 * rt - 1) / (16 * rt) + (j1.M + 16 * rt - 1) / (16 * rt)) *
               ((m + 8 * ct - 1) / (8 * ct)) * slices;
    };
    // The widest column tile that gives each of 256 CUs a workgroup (A is read
    // once per column group), then two row tiles where that leaves two per CU (X
    // is read half as often).  Counted on the whole chip also for a context with a
    // share of it: its products run in what the others leave.  Refined factorisation of 8321 unknowns, 49 columns:
    // 20.2 ms with one row tile, 19.5 with two, 21.4 with four; 64 columns per
    // tile instead of 32: 20.7.
    int ct = 1;
    while (ct < 4 && 8 * ct < m) ct *= 2;
    while (ct > 1 && wgs(1, ct) < 256) ct /= 2;
    const bool tall = ct >= 2 && wgs(2, ct) >= 512;
    auto go = [&](auto r, auto c) {
        constexpr int RT = decltype(r)::value, CT = decltype(c)::value;
        const int t0 = (j0.M + 16 * RT - 1) / (16 * RT), t1 = (j1.M + 16 * RT - 1) / (16 * RT);
        const dim3 grid(t0 + t1, (m + 8 * CT - 1) / (8 * CT), slices);
        k_skinny<TA, TC, RT, CT><<<grid, 256, 0, s>>>(j0, j1, t0, m, kc, P);
    };
    using std::integral_constant;
    const integral_constant<int, 1> one;
    const integral_constant<int, 2> two;
    const integral_constant<int, 4> four;
    if (ct == 4)
        tall ? go(two, four) : go(one, four);
    else if (ct == 2)
        tall ? go(two, two) : go(one, two);
    else
        go(one, one);
    EMFA_HIP_CHECK(hipGetLastError());
    return EMFA_OK;
}

}  // namespace

emfa_status skinny_mm(hipStream_t s, const SkinnyJob<float, float> &j, int m, const SkinnyJob<float, float> *second) {
    return launch<float, float>(s, j, second, m, 1, std::max(j.K, second ? second->K : 0), nullptr);
}
emfa_status skinny_mm(hipStream_t s, const SkinnyJob<double, double> &j, int m,
                      const SkinnyJob<double, double> *second) {
    return launch<double, double>(s, j, second, m, 1, std::max(j.K, second ? second->K : 0), nullptr);
}
emfa_status skinny_mm_slices(hipStream_t s, const SkinnyJob<float, double> &j, int m, int slices, int kc,
                             cx<double> *P) {
    return launch<float, double>(s, j, nullptr, m, slices, kc, P);
}
emfa_status skinny_mm_slices(hipStream_t s, const SkinnyJob<double, double> &j, int m, int slices, int kc,
                             cx<double> *P) {
    return launch<double, double>(s, j, nullptr, m, slices, kc, P);
}

}  // namespace emfa
