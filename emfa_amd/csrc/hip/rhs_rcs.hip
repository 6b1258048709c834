// Excitation columns (K3) and far-field RCS (K9), plus small matrix utilities.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "em_device.h"
#include "internal.h"

namespace emfa {

struct tri_abs {
    double v[3][3];
    double n[3];
};

__device__ __forceinline__ void load_tri(const double *__restrict__ tg, int T, int t, tri_abs *o) {
    for (int i = 0; i < 3; ++i)
        for (int c = 0; c < 3; ++c) o->v[i][c] = tg[(size_t)c * T + t] + tg[(size_t)(3 + 3 * i + c) * T + t];
    for (int c = 0; c < 3; ++c) o->n[c] = tg[(size_t)(12 + c) * T + t];
}

// V(u, j) = 1/2 l_u sum_{+,-} sum_a w_a rho . [alpha e + (1-alpha) n x h] exp(-jk k.r)
// EFIE (kind 0): 7-point rule, e only (EMSolver/EFIE.cpp:568-601,698-722).
// CFIE (kind 1): 3-point rule (EMSolver/Miscellaneous.cpp:152-189).
// MFIE (kind 2): 7-point rule, n x h part only (EMSolver/MFIE.cpp:289-322,
// 435-436 without its 1/Z0, matching the Z0-scaled MFIE operator of the fill).
//
// Up to 2048 values per CU (524288 on 256 CUs: 8321 x 49 still): one thread per
// (u, j), j fastest so the row-major writes coalesce.  A launch's latency mostly
// (122880 x 1 columns 15 us, 10 as k_rhs with one column per thread); it keeps the
// library's sincos and absolute points, and so the bits that an iterative solver's
// step count can hang on.  A column's last bits differ from k_rhs's.
template <typename R>
__global__ __launch_bounds__(256) void k_rhs_few(const double *__restrict__ tg, const int *__restrict__ rtp,
                                             const int *__restrict__ rtm, const int *__restrict__ rap,
                                             const int *__restrict__ ram, const double *__restrict__ rlen, int T,
                                             int N, int nrhs, const double *__restrict__ inc, int kind, double k,
                                             double alpha, cx<R> *__restrict__ B) {
    long long id = (long long)blockIdx.x * 256 + threadIdx.x;
    if (id >= (long long)N * nrhs) return;
    int u = (int)(id / nrhs), j = (int)(id % nrhs);
    const double *c = inc + 9 * j;
    double kv[3] = {c[0], c[1], c[2]}, ev[3] = {c[3], c[4], c[5]}, hv[3] = {c[6], c[7], c[8]};
    double vr = 0, vi = 0, mr = 0, mi = 0;
    for (int side = 0; side < 2; ++side) {
        int t = side == 0 ? rtp[u] : rtm[u];
        int a = side == 0 ? rap[u] : ram[u];
        tri_abs ta;
        load_tri(tg, T, t, &ta);
        double sg = side == 0 ? 1.0 : -1.0;
        double nxh[3] = {ta.n[1] * hv[2] - ta.n[2] * hv[1], ta.n[2] * hv[0] - ta.n[0] * hv[2],
                         ta.n[0] * hv[1] - ta.n[1] * hv[0]};
        int Q = kind == EMFA_CFIE ? 3 : 7;
        for (int p = 0; p < Q; ++p) {
            const double *rw = Q == 7 ? c_rule7[p] : c_rule3[p];
            double r[3];
            for (int cc = 0; cc < 3; ++cc) r[cc] = rw[0] * ta.v[0][cc] + rw[1] * ta.v[1][cc] + rw[2] * ta.v[2][cc];
            double rho[3];
            for (int cc = 0; cc < 3; ++cc) rho[cc] = sg * (r[cc] - ta.v[a][cc]);
            double ph = k * (r[0] * kv[0] + r[1] * kv[1] + r[2] * kv[2]);
            double s, co;
            sincos(ph, &s, &co);
            double w = rw[3];
            double de = rho[0] * ev[0] + rho[1] * ev[1] + rho[2] * ev[2];
            vr += w * de * co;
            vi -= w * de * s;
            if (kind != EMFA_EFIE) {
                double dm = rho[0] * nxh[0] + rho[1] * nxh[1] + rho[2] * nxh[2];
                mr += w * dm * co;
                mi -= w * dm * s;
            }
        }
    }
    double outr, outi;
    if (kind == EMFA_EFIE) {
        outr = vr;
        outi = vi;
    } else if (kind == EMFA_MFIE) {
        outr = mr;
        outi = mi;
    } else {
        outr = alpha * vr + (1.0 - alpha) * mr;
        outi = alpha * vi + (1.0 - alpha) * mi;
    }
    double h = 0.5 * rlen[u];
    B[(size_t)u * nrhs + j] = {(R)(h * outr), (R)(h * outi)};
}

// Many values: one thread per u and JB consecutive j, for which the points and
// rho are formed once.  VALU-bound: Q sines and cosines per side and value.  7680
// unknowns x 181 CFIE columns: 72 -> 36 us against k_rhs_few.
template <typename R, int Q, int JB>
__global__ __launch_bounds__(256) void k_rhs(const double *__restrict__ tg, const int *__restrict__ rtp,
                                             const int *__restrict__ rtm, const int *__restrict__ rap,
                                             const int *__restrict__ ram, const double *__restrict__ rlen, int T,
                                             int N, int nrhs, const double *__restrict__ inc, double we, double wh,
                                             double kq, double kl, cx<R> *__restrict__ B) {
    const int nj = (nrhs + JB - 1) / JB;
    const long long id = (long long)blockIdx.x * 256 + threadIdx.x;
    if (id >= (long long)N * nj) return;
    const int u = (int)(id / nj), j0 = (int)(id % nj) * JB;
    double vr[JB], vi[JB];
#pragma unroll
    for (int i = 0; i < JB; ++i) vr[i] = vi[i] = 0;
#pragma unroll 1
    for (int side = 0; side < 2; ++side) {
        const int t = side == 0 ? rtp[u] : rtm[u], a = side == 0 ? rap[u] : ram[u];
        const double sg = side == 0 ? 1.0 : -1.0;
        double cen[3], v[3][3], n[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            cen[c] = tg[(size_t)c * T + t];
            n[c] = tg[(size_t)(12 + c) * T + t];
#pragma unroll
            for (int i = 0; i < 3; ++i) v[i][c] = tg[(size_t)(3 + 3 * i + c) * T + t];
        }
        double x[Q][3];
#pragma unroll
        for (int p = 0; p < Q; ++p)
#pragma unroll
            for (int c = 0; c < 3; ++c) x[p][c] = rule<Q>(p, 0) * v[0][c] + rule<Q>(p, 1) * v[1][c] + rule<Q>(p, 2) * v[2][c];
        double va[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) va[c] = a == 0 ? v[0][c] : a == 1 ? v[1][c] : v[2][c];
#pragma unroll
        for (int i = 0; i < JB; ++i) {
            const double *w = inc + 9 * min(j0 + i, nrhs - 1);
            // the field that rho is dotted with, sign included (a field the
            // formulation does not use may hold anything)
            double f[3] = {0, 0, 0};
            if (we != 0)
                for (int c = 0; c < 3; ++c) f[c] = sg * we * w[3 + c];
            if (wh != 0) {
                f[0] += sg * wh * (n[1] * w[8] - n[2] * w[7]);
                f[1] += sg * wh * (n[2] * w[6] - n[0] * w[8]);
                f[2] += sg * wh * (n[0] * w[7] - n[1] * w[6]);
            }
            const double kc = cen[0] * w[0] + cen[1] * w[1] + cen[2] * w[2];
#pragma unroll
            for (int p = 0; p < Q; ++p) {
                double s, co;
                sincos_kr(kc + (x[p][0] * w[0] + x[p][1] * w[1] + x[p][2] * w[2]), kq, kl, &s, &co);
                const double d = rule<Q>(p, 3) * ((x[p][0] - va[0]) * f[0] + (x[p][1] - va[1]) * f[1] +
                                                  (x[p][2] - va[2]) * f[2]);
                vr[i] += d * co;
                vi[i] -= d * s;
            }
        }
    }
    const double h = 0.5 * rlen[u];
#pragma unroll
    for (int i = 0; i < JB; ++i)
        if (j0 + i < nrhs) B[(size_t)u * nrhs + j0 + i] = {(R)(h * vr[i]), (R)(h * vi[i])};
}

// Far field per direction: Es = sum_u I_u L_u sum_7 w rho exp(+jk s.r), summed by
// triangles: with c_a = +-I L of the edge opposite vertex a, a triangle adds
//   sum_p w_p exp(jk s.r_p) (C x_p - D),  C = sum_a c_a,  D = sum_a c_a A_a
// (points x_p and vertices A_a relative to the centroid), so each of its seven
// exponentials is formed once instead of once per edge and side, and x_p =
// sum_i b_pi A_i leaves sums over b_pi exp for each vertex.
// Grid (directions, slices of the triangles); part[d][slice] = {Es re, im}.
// VALU-bound: 7 sines and cosines per triangle and direction.  5120 triangles x
// 181 directions 168 -> 43 us, 81920 x 361 3.41 -> 0.67 ms against one
// workgroup per direction and 14 library sincos per edge.
template <typename R>
__global__ __launch_bounds__(256) void k_rcs_part(const double *__restrict__ tg, const int *__restrict__ t2r,
                                                  const double *__restrict__ rlen, int T,
                                                  const cx<R> *__restrict__ X, int ldx,
                                                  const double *__restrict__ dirs, const int *__restrict__ cols,
                                                  double kq, double kl, double *__restrict__ part) {
    const int d = blockIdx.x, ns = gridDim.y;
    const double s[3] = {dirs[3 * d], dirs[3 * d + 1], dirs[3 * d + 2]};
    const int col = cols ? cols[d] : 0;
    double acc[6] = {0, 0, 0, 0, 0, 0};
    for (int t = blockIdx.y * 256 + threadIdx.x; t < T; t += ns * 256) {
        double A[3][3], sA[3], Cr = 0, Ci = 0, Dr[3] = {0, 0, 0}, Di[3] = {0, 0, 0}, sc = 0;
#pragma unroll
        for (int c = 0; c < 3; ++c) sc += s[c] * tg[(size_t)c * T + t];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
#pragma unroll
            for (int c = 0; c < 3; ++c) A[a][c] = tg[(size_t)(3 + 3 * a + c) * T + t];
            sA[a] = s[0] * A[a][0] + s[1] * A[a][1] + s[2] * A[a][2];
            const int code = t2r[(size_t)a * T + t];
            if (code == 0) continue;
            const int u = (code > 0 ? code : -code) - 1;
            const cx<R> x = X[(size_t)u * ldx + col];
            const double L = code > 0 ? rlen[u] : -rlen[u];
            const double cr = (double)x.re * L, ci = (double)x.im * L;
            Cr += cr;
            Ci += ci;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                Dr[c] += cr * A[a][c];
                Di[c] += ci * A[a][c];
            }
        }
        double er[3] = {0, 0, 0}, ei[3] = {0, 0, 0};  // sum_p w b_pi exp per vertex; their sum is sum_p w exp
#pragma unroll
        for (int p = 0; p < 7; ++p) {
            double sn, co;
            sincos_kr(sc + (rule<7>(p, 0) * sA[0] + rule<7>(p, 1) * sA[1] + rule<7>(p, 2) * sA[2]), kq, kl, &sn, &co);
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                er[i] += rule<7>(p, 3) * rule<7>(p, i) * co;
                ei[i] += rule<7>(p, 3) * rule<7>(p, i) * sn;
            }
        }
        const double e0r = er[0] + er[1] + er[2], e0i = ei[0] + ei[1] + ei[2];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double vr = er[0] * A[0][c] + er[1] * A[1][c] + er[2] * A[2][c];
            const double vi = ei[0] * A[0][c] + ei[1] * A[1][c] + ei[2] * A[2][c];
            acc[2 * c] += Cr * vr - Ci * vi - (Dr[c] * e0r - Di[c] * e0i);
            acc[2 * c + 1] += Cr * vi + Ci * vr - (Dr[c] * e0i + Di[c] * e0r);
        }
    }
    __shared__ double red[6][4];
#pragma unroll
    for (int i = 0; i < 6; ++i) {
#pragma unroll
        for (int o = 1; o < 64; o *= 2) acc[i] += __shfl_xor(acc[i], o);
        if ((threadIdx.x & 63) == 0) red[i][threadIdx.x >> 6] = acc[i];
    }
    __syncthreads();
    if (threadIdx.x < 6)
        part[((size_t)d * ns + blockIdx.y) * 6 + threadIdx.x] =
            (red[threadIdx.x][0] + red[threadIdx.x][1]) + (red[threadIdx.x][2] + red[threadIdx.x][3]);
}

// sigma = Z0^2 k^2 |1/2 s x (s x Es)|^2 / 4 pi  (EMSolver/EFIE.cpp:788-832), in dB;
// one thread per direction, its slices added in order.
__global__ __launch_bounds__(64) void k_rcs_db(const double *__restrict__ part, int ns, int ndir,
                                               const double *__restrict__ dirs, double k, double *__restrict__ out) {
    const int d = blockIdx.x * 64 + threadIdx.x;
    if (d >= ndir) return;
    double e[6] = {0, 0, 0, 0, 0, 0};
    for (int i = 0; i < ns; ++i)
        for (int c = 0; c < 6; ++c) e[c] += part[((size_t)d * ns + i) * 6 + c];
    const double s[3] = {dirs[3 * d], dirs[3 * d + 1], dirs[3 * d + 2]};
    const double Er[3] = {e[0], e[2], e[4]}, Ei[3] = {e[1], e[3], e[5]};
    // c = s x E ; f = 0.5 s x c
    const double cr[3] = {s[1] * Er[2] - s[2] * Er[1], s[2] * Er[0] - s[0] * Er[2], s[0] * Er[1] - s[1] * Er[0]};
    const double ci[3] = {s[1] * Ei[2] - s[2] * Ei[1], s[2] * Ei[0] - s[0] * Ei[2], s[0] * Ei[1] - s[1] * Ei[0]};
    const double fr[3] = {0.5 * (s[1] * cr[2] - s[2] * cr[1]), 0.5 * (s[2] * cr[0] - s[0] * cr[2]),
                          0.5 * (s[0] * cr[1] - s[1] * cr[0])};
    const double fi[3] = {0.5 * (s[1] * ci[2] - s[2] * ci[1]), 0.5 * (s[2] * ci[0] - s[0] * ci[2]),
                          0.5 * (s[0] * ci[1] - s[1] * ci[0])};
    double nrm = 0;
    for (int c = 0; c < 3; ++c) nrm += fr[c] * fr[c] + fi[c] * fi[c];
    out[d] = 10.0 * log10(kZ0 * kZ0 * k * k * nrm / (4.0 * kPi));
}

// Precision conversion / copy of interleaved complex buffers.
template <typename S, typename D>
__global__ __launch_bounds__(256) void k_convert(const S *__restrict__ src, D *__restrict__ dst, size_t n) {
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    size_t stride = (size_t)gridDim.x * 256;
    for (; i < n; i += stride) dst[i] = (D)src[i];
}

// X += D  (X double, D float or double), element-wise over interleaved reals
template <typename S>
__global__ __launch_bounds__(256) void k_axpy(double *__restrict__ x, const S *__restrict__ d, size_t n) {
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    size_t stride = (size_t)gridDim.x * 256;
    for (; i < n; i += stride) x[i] += (double)d[i];
}

emfa_status convert_copy(emfa_ctx *ctx, const emfa_mat *src, emfa_mat *dst) {
    size_t n = 2 * (size_t)src->rows * src->cols;
    if (src->prec == dst->prec) {
        EMFA_HIP_CHECK(hipMemcpyAsync(dst->d, src->d, src->bytes, hipMemcpyDeviceToDevice, ctx->stream));
        return EMFA_OK;
    }
    int blocks = (int)std::min<size_t>((n + 255) / 256, 65536);
    if (src->prec == EMFA_F32)
        k_convert<float, double><<<blocks, 256, 0, ctx->stream>>>((const float *)src->d, (double *)dst->d, n);
    else
        k_convert<double, float><<<blocks, 256, 0, ctx->stream>>>((const double *)src->d, (float *)dst->d, n);
    EMFA_HIP_CHECK(hipGetLastError());
    return EMFA_OK;
}

emfa_status axpy_f64(emfa_ctx *ctx, emfa_mat *X, const emfa_mat *D) {
    size_t n = 2 * (size_t)X->rows * X->cols;
    int blocks = (int)std::min<size_t>((n + 255) / 256, 65536);
    if (D->prec == EMFA_F32)
        k_axpy<float><<<blocks, 256, 0, ctx->stream>>>((double *)X->d, (const float *)D->d, n);
    else
        k_axpy<double><<<blocks, 256, 0, ctx->stream>>>((double *)X->d, (const double *)D->d, n);
    EMFA_HIP_CHECK(hipGetLastError());
    return EMFA_OK;
}

}  // namespace emfa

using namespace emfa;

extern "C" emfa_status emfa_rhs_fill(emfa_ctx *ctx, const emfa_mesh *M, int kind, double k, double alpha, int nrhs,
                                     const double *inc, emfa_mat *B) {
    EMFA_REQUIRE(ctx && M && inc && B, EMFA_E_INVALID, "emfa_rhs_fill: null argument");
    EMFA_REQUIRE(nrhs > 0 && B->rows == M->n && B->cols == nrhs, EMFA_E_INVALID,
                 "emfa_rhs_fill: B is %dx%d, expected %dx%d", B->rows, B->cols, M->n, nrhs);
    EMFA_REQUIRE(kind == EMFA_EFIE || kind == EMFA_CFIE || kind == EMFA_MFIE, EMFA_E_INVALID,
                 "emfa_rhs_fill: bad kind");
    EMFA_HIP_CHECK(hipSetDevice(ctx->device));
    void *dinc = nullptr;
    EMFA_HIP_CHECK(ctx_alloc(ctx, &dinc, 9 * sizeof(double) * nrhs));
    EMFA_HIP_CHECK(hipMemcpyAsync(dinc, inc, 9 * sizeof(double) * nrhs, hipMemcpyHostToDevice, ctx->stream));
    {
        ProfScope ps(ctx, "rhs", 0);
        double kq, kl;
        quarter_turns(k, &kq, &kl);
        const double we = kind == EMFA_EFIE ? 1.0 : kind == EMFA_MFIE ? 0.0 : alpha;
        const double wh = kind == EMFA_EFIE ? 0.0 : kind == EMFA_MFIE ? 1.0 : 1.0 - alpha;
        auto go = [&](auto q, auto jb) {
            constexpr int Q = decltype(q)::value, JB = decltype(jb)::value;
            const unsigned blocks = (unsigned)(((long long)M->n * ((nrhs + JB - 1) / JB) + 255) / 256);
            if (B->prec == EMFA_F32)
                k_rhs<float, Q, JB><<<blocks, 256, 0, ctx->stream>>>(M->tg64, M->rtp, M->rtm, M->rap, M->ram,
                                                                     M->rlen64, M->nt, M->n, nrhs,
                                                                     (const double *)dinc, we, wh, kq, kl,
                                                                     (cx<float> *)B->d);
            else
                k_rhs<double, Q, JB><<<blocks, 256, 0, ctx->stream>>>(M->tg64, M->rtp, M->rtm, M->rap, M->ram,
                                                                      M->rlen64, M->nt, M->n, nrhs,
                                                                      (const double *)dinc, we, wh, kq, kl,
                                                                      (cx<double> *)B->d);
        };
        using std::integral_constant;
        // four columns per thread once that still gives every CU eight waves
        if ((long long)M->n * nrhs >= 4LL * 512 * ctx->num_cu) {
            if (kind == EMFA_CFIE)
                go(integral_constant<int, 3>{}, integral_constant<int, 4>{});
            else
                go(integral_constant<int, 7>{}, integral_constant<int, 4>{});
        } else {
            const unsigned blocks = (unsigned)(((long long)M->n * nrhs + 255) / 256);
            if (B->prec == EMFA_F32)
                k_rhs_few<float><<<blocks, 256, 0, ctx->stream>>>(M->tg64, M->rtp, M->rtm, M->rap, M->ram, M->rlen64,
                                                                  M->nt, M->n, nrhs, (const double *)dinc, kind, k,
                                                                  alpha, (cx<float> *)B->d);
            else
                k_rhs_few<double><<<blocks, 256, 0, ctx->stream>>>(M->tg64, M->rtp, M->rtm, M->rap, M->ram, M->rlen64,
                                                                   M->nt, M->n, nrhs, (const double *)dinc, kind, k,
                                                                   alpha, (cx<double> *)B->d);
        }
    }
    hipError_t e = hipGetLastError();
    (void)hipStreamSynchronize(ctx->stream);
    ctx_free(ctx, dinc, 9 * sizeof(double) * nrhs);
    EMFA_HIP_CHECK(e);
    return EMFA_OK;
}

extern "C" emfa_status emfa_rcs(emfa_ctx *ctx, const emfa_mesh *M, double k, const emfa_mat *X, int ndir,
                                const double *dirs, const int *cols, double *out_db) {
    EMFA_REQUIRE(ctx && M && X && dirs && out_db, EMFA_E_INVALID, "emfa_rcs: null argument");
    EMFA_REQUIRE(X->rows == M->n && ndir > 0, EMFA_E_INVALID, "emfa_rcs: X has %d rows, mesh %d RWGs", X->rows, M->n);
    if (cols)
        for (int d = 0; d < ndir; ++d)
            EMFA_REQUIRE(cols[d] >= 0 && cols[d] < X->cols, EMFA_E_INVALID, "emfa_rcs: column %d out of range",
                         cols[d]);
    EMFA_HIP_CHECK(hipSetDevice(ctx->device));
    // about four workgroups per CU over the directions and triangle slices
    const int ns = std::max(1, std::min((M->nt + 255) / 256, (4 * ctx->num_cu + ndir - 1) / ndir));
    // one upload: directions, then columns; behind them the values and the slices' sums
    const size_t nd = (size_t)ndir, in_b = nd * 3 * sizeof(double) + (cols ? (nd * sizeof(int) + 7) / 8 * 8 : 0);
    const size_t bytes = in_b + nd * sizeof(double) + nd * ns * 6 * sizeof(double);
    std::vector<char> in(in_b);
    std::memcpy(in.data(), dirs, nd * 3 * sizeof(double));
    if (cols) std::memcpy(in.data() + nd * 3 * sizeof(double), cols, nd * sizeof(int));
    void *buf = nullptr;
    EMFA_HIP_CHECK(ctx_alloc(ctx, &buf, bytes));
    const double *ddirs = (const double *)buf;
    const int *dcols = cols ? (const int *)(ddirs + 3 * nd) : nullptr;
    double *dout = (double *)((char *)buf + in_b), *part = dout + nd;
    EMFA_HIP_CHECK(hipMemcpyAsync(buf, in.data(), in_b, hipMemcpyHostToDevice, ctx->stream));
    {
        ProfScope ps(ctx, "rcs", 0);
        double kq, kl;
        quarter_turns(k, &kq, &kl);
        const dim3 grid(ndir, ns);
        if (X->prec == EMFA_F32)
            k_rcs_part<float><<<grid, 256, 0, ctx->stream>>>(M->tg64, M->t2r, M->rlen64, M->nt, (const cx<float> *)X->d,
                                                             X->cols, ddirs, dcols, kq, kl, part);
        else
            k_rcs_part<double><<<grid, 256, 0, ctx->stream>>>(M->tg64, M->t2r, M->rlen64, M->nt,
                                                              (const cx<double> *)X->d, X->cols, ddirs, dcols, kq, kl,
                                                              part);
        k_rcs_db<<<(ndir + 63) / 64, 64, 0, ctx->stream>>>(part, ns, ndir, ddirs, k, dout);
    }
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(out_db, dout, ndir * sizeof(double), hipMemcpyDeviceToHost, ctx->stream);
    (void)hipStreamSynchronize(ctx->stream);
    ctx_free(ctx, buf, bytes);
    EMFA_HIP_CHECK(e);
    return EMFA_OK;
}
