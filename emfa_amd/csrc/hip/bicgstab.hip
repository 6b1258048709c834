// BiCGSTAB on the device over any operator y = A x on vectors of n complex
// FP64 values: the dense matrix (K7 matvec) or the MLFMA operator.
//
// Two forms, as the reference has them:
//   variant 0  EMIterative/iml.cpp:3-39 (the overload EMSolver/CFIE.cpp:76
//              calls with eps 0.01 and 500 steps; MLFMA.cpp:402-452 runs the
//              same steps): x0 = 0, stop when ||s|| / ||b|| < eps after the
//              alpha step; "not converged" when all max_iter steps ran.
//   variant 1  EMIterative/iml.cpp:88-154 (the matrix-free overload): stop
//              when ||r||^2 / ||b||^2 <= eps^2; when |rho| falls below
//              eps_f^2 ||r0||^2 (eps_f = float epsilon) the shadow residual
//              restarts at r and the first restart resets the step count.
// The vector updates are fused elementwise kernels; the inner products of a
// step are formed together in one launch (deterministic chunked sums, FP64)
// and read back with one copy.
#include <algorithm>
#include <cmath>
#include <complex>
#include <functional>
#include <vector>

#include "internal.h"

namespace emfa {

namespace {

constexpr int kBiChunks = 64;
constexpr int kMaxPairs = 5;  // per right-hand side

struct DotPairs {
    const double2 *a[kMaxPairs * kGemvCols];  // conj(a) . b
    const double2 *b[kMaxPairs * kGemvCols];
};

// partial sums part[pair][chunk] of conj(a_pair) . b_pair over row chunks
__global__ __launch_bounds__(256) void k_bi_dots(DotPairs d, int n, double2 *__restrict__ part) {
    const int pr = blockIdx.y, c = blockIdx.x, nc = gridDim.x;
    const double2 *a = d.a[pr], *b = d.b[pr];
    const int per = (n + nc - 1) / nc;
    const int t0 = c * per, t1 = min(n, t0 + per);
    double sr = 0, si = 0;
    for (int t = t0 + threadIdx.x; t < t1; t += 256) {
        const double2 x = a[t], y = b[t];
        sr += x.x * y.x + x.y * y.y;
        si += x.x * y.y - x.y * y.x;
    }
    __shared__ double rr[256], ri[256];
    rr[threadIdx.x] = sr;
    ri[threadIdx.x] = si;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (threadIdx.x < st) {
            rr[threadIdx.x] += rr[threadIdx.x + st];
            ri[threadIdx.x] += ri[threadIdx.x + st];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) part[(size_t)pr * nc + c] = make_double2(rr[0], ri[0]);
}

// the chunks of each pair added in chunk order
__global__ __launch_bounds__(64) void k_bi_dots_sum(const double2 *__restrict__ part, int np, int nc,
                                                    double2 *__restrict__ out) {
    const int i = threadIdx.x;
    if (i >= np) return;
    double sr = 0, si = 0;
    for (int c = 0; c < nc; ++c) {
        sr += part[(size_t)i * nc + c].x;
        si += part[(size_t)i * nc + c].y;
    }
    out[i] = make_double2(sr, si);
}

__device__ __forceinline__ double2 cmad(double2 acc, double2 a, double2 x) {  // acc + a x
    return make_double2(acc.x + a.x * x.x - a.y * x.y, acc.y + a.x * x.y + a.y * x.x);
}

// The group's columns that a step still works on (blockIdx.y picks one): column
// c[i] of the group's vectors, ld apart, with its scalars.
struct BiCols {
    int n, m;  // columns listed
    long long ld;
    int c[kGemvCols];
    double2 s[kGemvCols], w[kGemvCols];
};

// p = r + beta (p - w v), beta = s
__global__ __launch_bounds__(256) void k_bi_p(const double2 *__restrict__ r, const double2 *__restrict__ v, BiCols g,
                                              double2 *__restrict__ p) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= g.n) return;
    const long long o = g.c[blockIdx.y] * g.ld + t;
    const double2 w = g.w[blockIdx.y];
    const double2 d = cmad(p[o], make_double2(-w.x, -w.y), v[o]);
    p[o] = cmad(r[o], g.s[blockIdx.y], d);
}

// x += alpha p ; s = r - alpha v
__global__ __launch_bounds__(256) void k_bi_xs(const double2 *__restrict__ p, const double2 *__restrict__ r,
                                               const double2 *__restrict__ v, BiCols g, double2 *__restrict__ x,
                                               double2 *__restrict__ s) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= g.n) return;
    const long long o = g.c[blockIdx.y] * g.ld + t;
    const double2 alpha = g.s[blockIdx.y];
    x[o] = cmad(x[o], alpha, p[o]);
    s[o] = cmad(r[o], make_double2(-alpha.x, -alpha.y), v[o]);
}

// s = r - alpha v
__global__ __launch_bounds__(256) void k_bi_s(const double2 *__restrict__ r, const double2 *__restrict__ v, BiCols g,
                                              double2 *__restrict__ s) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= g.n) return;
    const long long o = g.c[blockIdx.y] * g.ld + t;
    const double2 alpha = g.s[blockIdx.y];
    s[o] = cmad(r[o], make_double2(-alpha.x, -alpha.y), v[o]);
}

// x += a p + w s ; r = s - w t   (a = 0 drops the p term)
__global__ __launch_bounds__(256) void k_bi_xr(const double2 *__restrict__ p, const double2 *__restrict__ s,
                                               const double2 *__restrict__ tv, BiCols g, double2 *__restrict__ x,
                                               double2 *__restrict__ r) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= g.n) return;
    const long long o = g.c[blockIdx.y] * g.ld + t;
    const double2 a = g.s[blockIdx.y], w = g.w[blockIdx.y];
    double2 xv = x[o];
    if (a.x != 0.0 || a.y != 0.0) xv = cmad(xv, a, p[o]);
    x[o] = cmad(xv, w, s[o]);
    r[o] = cmad(s[o], make_double2(-w.x, -w.y), tv[o]);
}

// column col0 + c of M (n x m) into b, r and the shadow residual; x, p, v = 0
__global__ __launch_bounds__(256) void k_bi_start(const double2 *__restrict__ M, int col0, BiCols g,
                                                  double2 *__restrict__ b, double2 *__restrict__ r,
                                                  double2 *__restrict__ rs, double2 *__restrict__ x,
                                                  double2 *__restrict__ p, double2 *__restrict__ v) {
    const int t = blockIdx.x * 256 + threadIdx.x, c = g.c[blockIdx.y];
    if (t >= g.n) return;
    const long long o = c * g.ld + t;
    b[o] = r[o] = rs[o] = M[(size_t)t * g.m + col0 + c];
    x[o] = p[o] = v[o] = make_double2(0.0, 0.0);
}

__global__ __launch_bounds__(256) void k_bi_put(const double2 *__restrict__ x, int col0, BiCols g,
                                                double2 *__restrict__ M) {
    const int t = blockIdx.x * 256 + threadIdx.x, c = g.c[blockIdx.y];
    if (t < g.n) M[(size_t)t * g.m + col0 + c] = x[c * g.ld + t];
}

__global__ __launch_bounds__(256) void k_bi_copy(const double2 *__restrict__ a, BiCols g, double2 *__restrict__ b) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= g.n) return;
    const long long o = g.c[blockIdx.y] * g.ld + t;
    b[o] = a[o];
}

// b - y into y
__global__ __launch_bounds__(256) void k_bi_resid(const double2 *__restrict__ b, BiCols g, double2 *__restrict__ y) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= g.n) return;
    const long long o = g.c[blockIdx.y] * g.ld + t;
    y[o] = make_double2(b[o].x - y[o].x, b[o].y - y[o].y);
}

}  // namespace

// Device bytes the solver's vectors and partial sums take for n unknowns and
// groups of `group` right-hand sides.
size_t bicgstab_work_bytes(int n, int group) {
    const int nchunk = std::max(1, std::min(kBiChunks, (n + 2047) / 2048));
    const size_t vb = ((size_t)n * sizeof(double2) + 255) & ~(size_t)255;
    return (size_t)group * (9 * vb + (size_t)kMaxPairs * (nchunk + 1) * sizeof(double2)) + 512;
}

// The right-hand sides of a group step together: one product reads the matrix
// for all of them and one read-back brings all their inner products; a column
// that is done drops out.  Each column's operations and their order are those
// of a solve of its own.  7680 unknowns, FP32, to 1e-2: one column 3.03 -> 2.68
// ms, two 6.63 -> 3.28, four 12.57 -> 3.53; 1920 unknowns, two: 1.63 -> 0.79.
emfa_status bicgstab_impl(emfa_ctx *ctx, int n, const BicgstabOp &matvec, const emfa_mat *B, emfa_mat *X, double tol,
                          int max_iter, int variant, emfa_bicgstab_report *rep, int group, void *work,
                          size_t work_bytes) {
    const int nr = B->cols;
    EMFA_REQUIRE(B->rows == n && X->rows == n && X->cols == nr && B->prec == EMFA_F64 && X->prec == EMFA_F64,
                 EMFA_E_INVALID, "bicgstab: B and X must be F64 n x nrhs");
    EMFA_REQUIRE(max_iter >= 1 && tol > 0 && (variant == 0 || variant == 1), EMFA_E_INVALID,
                 "bicgstab: max_iter >= 1, tol > 0, variant 0 or 1");
    EMFA_HIP_CHECK(hipSetDevice(ctx->device));
    const int G = std::max(1, std::min({group, kGemvCols, nr}));
    const int nchunk = std::max(1, std::min(kBiChunks, (n + 2047) / 2048));
    const size_t vb = ((size_t)n * sizeof(double2) + 255) & ~(size_t)255;
    void *scr = work;
    emfa_status st = EMFA_OK;
    if (scr) {
        EMFA_REQUIRE(work_bytes >= bicgstab_work_bytes(n, G), EMFA_E_INVALID,
                     "bicgstab: workspace of %zu bytes, %zu needed", work_bytes, bicgstab_work_bytes(n, G));
    } else if ((st = ctx_scratch(ctx, bicgstab_work_bytes(n, G), &scr))) {
        return st;
    }
    char *q = (char *)scr;
    auto take = [&](size_t b) {
        char *o = q;
        q += (b + 255) & ~(size_t)255;
        return (double2 *)o;
    };
    // each holds the group's columns, ld apart
    const long long ld = (long long)(vb / sizeof(double2));
    double2 *bv = take(G * vb), *x = take(G * vb), *r = take(G * vb), *rs = take(G * vb), *p = take(G * vb),
            *v = take(G * vb), *s = take(G * vb), *tv = take(G * vb), *w = take(G * vb);
    double2 *part = take((size_t)G * kMaxPairs * nchunk * sizeof(double2));
    double2 *dsum = take((size_t)G * kMaxPairs * sizeof(double2));
    hipStream_t stm = ctx->stream;
    using cd = std::complex<double>;
    struct Column {
        cd rho0 = 1, rho1 = 1, alpha = 1, omega = 1;
        double bn2 = 0, r0_sq = 0;
        int steps = 0, restarts = 0;
        bool conv = false;
    } col[kGemvCols];
    std::vector<int> act;  // columns of the group at work
    BiCols g{};
    g.n = n;
    g.m = nr;
    g.ld = ld;
    auto d2 = [](cd z) { return make_double2(z.real(), z.imag()); };
    // the working columns with their scalars
    auto cols = [&](auto scalar, auto second) {
        for (size_t i = 0; i < act.size(); ++i) {
            g.c[i] = act[i];
            g.s[i] = d2(scalar(col[act[i]]));
            g.w[i] = d2(second(col[act[i]]));
        }
        return dim3((n + 255) / 256, (unsigned)act.size());
    };
    auto none = [](const Column &) { return cd(0); };
    double2 hd[kMaxPairs * kGemvCols];
    // conj(a_i) . b_i of every working column for the given pairs of vectors,
    // read back to the host: hd[column's place * pairs + pair]
    auto dots = [&](std::initializer_list<std::pair<const double2 *, const double2 *>> pr) -> emfa_status {
        DotPairs d{};
        int i = 0;
        for (int c : act)
            for (auto &ab : pr) {
                d.a[i] = ab.first + c * ld;
                d.b[i] = ab.second + c * ld;
                ++i;
            }
        k_bi_dots<<<dim3(nchunk, i), 256, 0, stm>>>(d, n, part);
        k_bi_dots_sum<<<1, 64, 0, stm>>>(part, i, nchunk, dsum);
        EMFA_HIP_CHECK(hipGetLastError());
        EMFA_HIP_CHECK(hipMemcpyAsync(hd, dsum, i * sizeof(double2), hipMemcpyDeviceToHost, stm));
        EMFA_HIP_CHECK(hipStreamSynchronize(stm));
        return EMFA_OK;
    };
    auto dot = [&](size_t place, int pairs, int pair) {
        const double2 z = hd[place * pairs + pair];
        return cd(z.x, z.y);
    };
    auto apply = [&](const double2 *in, double2 *out) -> emfa_status {
        const double2 *pi[kGemvCols];
        double2 *po[kGemvCols];
        for (size_t i = 0; i < act.size(); ++i) {
            pi[i] = in + act[i] * ld;
            po[i] = out + act[i] * ld;
        }
        return matvec((int)act.size(), pi, po);
    };
    // drops the columns for which done(column, place) holds
    auto drop = [&](auto done) {
        std::vector<int> keep;
        for (size_t i = 0; i < act.size(); ++i)
            if (!done(col[act[i]], i)) keep.push_back(act[i]);
        act.swap(keep);
    };
    auto all_columns = [&](int m) {
        act.clear();
        for (int c = 0; c < m; ++c) act.push_back(c);
    };
    int total = 0, worst_steps = 0;
    double worst = 0;
    bool all_conv = true;
    for (int c0 = 0; c0 < nr; c0 += G) {
        const int m = std::min(G, nr - c0);
        for (int c = 0; c < m; ++c) col[c] = Column();
        all_columns(m);
        // b, r = b (x0 = 0), shadow residual = b, x = p = v = 0
        k_bi_start<<<cols(none, none), 256, 0, stm>>>((const double2 *)B->d, c0, g, bv, r, rs, x, p, v);
        EMFA_HIP_CHECK(hipGetLastError());
        if ((st = dots({{bv, bv}}))) return st;
        for (int c = 0; c < m; ++c) col[c].bn2 = dot(c, 1, 0).real();
        drop([](Column &z, size_t) { return z.conv = z.bn2 == 0; });  // b = 0: x = 0
        if (variant == 0 && !act.empty()) {
            if ((st = dots({{rs, r}}))) return st;
            for (size_t i = 0; i < act.size(); ++i) col[act[i]].rho1 = dot(i, 1, 0);
            for (int it = 0; it < max_iter && !act.empty(); ++it) {
                for (int c : act) ++col[c].steps;
                k_bi_p<<<cols([](const Column &z) { return (z.rho1 / z.rho0) * (z.alpha / z.omega); },
                              [](const Column &z) { return z.omega; }),
                         256, 0, stm>>>(r, v, g, p);
                EMFA_HIP_CHECK(hipGetLastError());
                if ((st = apply(p, v))) return st;
                if ((st = dots({{rs, v}}))) return st;
                for (size_t i = 0; i < act.size(); ++i) col[act[i]].alpha = col[act[i]].rho1 / dot(i, 1, 0);
                k_bi_xs<<<cols([](const Column &z) { return z.alpha; }, none), 256, 0, stm>>>(p, r, v, g, x, s);
                EMFA_HIP_CHECK(hipGetLastError());
                if ((st = dots({{s, s}}))) return st;
                drop([&](Column &z, size_t i) {
                    return std::sqrt(std::max(0.0, dot(i, 1, 0).real())) / std::sqrt(std::max(0.0, z.bn2)) < tol;
                });
                if (act.empty()) break;
                if ((st = apply(s, tv))) return st;
                // t^H s, t^H t; and for the next step's rho: rs^H s, rs^H t
                if ((st = dots({{tv, s}, {tv, tv}, {rs, s}, {rs, tv}}))) return st;
                for (size_t i = 0; i < act.size(); ++i) col[act[i]].omega = dot(i, 4, 0) / dot(i, 4, 1);
                k_bi_xr<<<cols(none, [](const Column &z) { return z.omega; }), 256, 0, stm>>>(nullptr, s, tv, g, x, r);
                EMFA_HIP_CHECK(hipGetLastError());
                // the second test of iml.cpp:33-34 reads the same ||s||
                for (size_t i = 0; i < act.size(); ++i) {
                    Column &z = col[act[i]];
                    z.rho0 = z.rho1;
                    z.rho1 = dot(i, 4, 2) - z.omega * dot(i, 4, 3);  // rs^H (s - omega t)
                }
            }
            // iml.cpp:38: success unless every step ran
            for (int c = 0; c < m; ++c)
                if (col[c].bn2 != 0) col[c].conv = col[c].steps != max_iter;
        } else if (variant == 1) {
            const double epsf = 1.1920928955078125e-07, eps2 = epsf * epsf, tol2 = tol * tol;
            for (int c : act) col[c].r0_sq = col[c].bn2;
            while (!act.empty()) {
                if ((st = dots({{r, r}, {rs, r}}))) return st;
                std::vector<int> restart;
                drop([&](Column &z, size_t i) {
                    const double rr = dot(i, 2, 0).real();
                    if (!(rr / z.bn2 > tol2 && z.steps < max_iter)) return true;
                    z.rho0 = z.rho1;
                    z.rho1 = dot(i, 2, 1);
                    if (std::abs(z.rho1) < eps2 * z.r0_sq) {
                        restart.push_back((int)(&z - col));
                        z.rho1 = z.r0_sq = rr;
                        if (z.restarts++ == 0) z.steps = 0;
                    }
                    return false;
                });
                if (act.empty()) break;
                if (!restart.empty()) {
                    act.swap(restart);
                    k_bi_copy<<<cols(none, none), 256, 0, stm>>>(r, g, rs);
                    EMFA_HIP_CHECK(hipGetLastError());
                    act.swap(restart);
                }
                k_bi_p<<<cols([](const Column &z) { return (z.rho1 / z.rho0) * (z.alpha / z.omega); },
                              [](const Column &z) { return z.omega; }),
                         256, 0, stm>>>(r, v, g, p);
                EMFA_HIP_CHECK(hipGetLastError());
                if ((st = apply(p, v))) return st;
                if ((st = dots({{rs, v}}))) return st;
                for (size_t i = 0; i < act.size(); ++i) col[act[i]].alpha = col[act[i]].rho1 / dot(i, 1, 0);
                k_bi_s<<<cols([](const Column &z) { return z.alpha; }, none), 256, 0, stm>>>(r, v, g, s);
                EMFA_HIP_CHECK(hipGetLastError());
                if ((st = apply(s, tv))) return st;
                if ((st = dots({{tv, tv}, {tv, s}}))) return st;
                for (size_t i = 0; i < act.size(); ++i) {
                    const double tt = dot(i, 2, 0).real();
                    col[act[i]].omega = tt > 0 ? dot(i, 2, 1) / tt : cd(0);
                }
                k_bi_xr<<<cols([](const Column &z) { return z.alpha; }, [](const Column &z) { return z.omega; }), 256, 0,
                          stm>>>(p, s, tv, g, x, r);
                EMFA_HIP_CHECK(hipGetLastError());
                for (int c : act) ++col[c].steps;
            }
            // the overload always reports success (iml.cpp:147-153)
            for (int c = 0; c < m; ++c) col[c].conv = true;
        }
        // true residual of the returned x
        all_columns(m);
        if ((st = apply(x, w))) return st;
        k_bi_resid<<<cols(none, none), 256, 0, stm>>>(bv, g, w);
        EMFA_HIP_CHECK(hipGetLastError());
        if ((st = dots({{w, w}}))) return st;
        k_bi_put<<<cols(none, none), 256, 0, stm>>>(x, c0, g, (double2 *)X->d);
        EMFA_HIP_CHECK(hipGetLastError());
        for (int c = 0; c < m; ++c) {
            const double rel =
                col[c].bn2 > 0 ? std::sqrt(std::max(0.0, dot(c, 1, 0).real()) / col[c].bn2) : 0.0;
            total += col[c].steps;
            worst_steps = std::max(worst_steps, col[c].steps);
            worst = std::max(worst, rel);
            all_conv = all_conv && col[c].conv;
        }
    }
    EMFA_HIP_CHECK(hipStreamSynchronize(stm));
    if (rep) {
        rep->iterations = total;
        rep->max_steps = worst_steps;
        rep->relres = worst;
    }
    if (!all_conv) {
        set_error("bicgstab: a right-hand side used all %d steps (relative residual %.3e)", max_iter, worst);
        return EMFA_E_NOCONV;
    }
    return EMFA_OK;
}

}  // namespace emfa

using namespace emfa;

extern "C" emfa_status emfa_bicgstab(emfa_ctx *ctx, const emfa_mat *Z, const emfa_mat *B, emfa_mat *X, double tol,
                                     int max_iter, int variant, emfa_bicgstab_report *rep) {
    EMFA_REQUIRE(ctx && Z && B && X, EMFA_E_INVALID, "emfa_bicgstab: null argument");
    EMFA_REQUIRE(Z->cols == Z->rows, EMFA_E_INVALID, "emfa_bicgstab: Z must be square");
    return bicgstab_impl(
        ctx, Z->rows,
        [&](int nc, const double2 *const *in, double2 *const *out) { return gemv(ctx, Z, nc, in, out); }, B, X, tol,
        max_iter, variant, rep, kGemvCols);
}
