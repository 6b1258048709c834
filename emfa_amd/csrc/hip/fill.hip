// Impedance fill on gfx950: triangle-pair formulation.
//
// Every RWG-pair entry of EMFA's fill (EMSolver/EFIE.cpp:603-696,
// EMSolver/CFIE.cpp:485-568) is a sum over the 4 triangle pairs the two RWGs
// span of  s_f s_s l_f l_s * Z_tri(tf, a; ts, b), where a (b) is the local
// index of the RWG's free vertex in tf (ts) and s = +1 on the RWG's plus
// triangle, -1 on its minus triangle: every term of the reference kernels is
// bilinear in rho_f, rho_s, so the RWG signs factor out.  Z_tri is computed
// once per triangle pair (9 values) instead of once per RWG pair (the
// reference evaluates each triangle pair 9 times), then gathered.
//
//   K1 k_fill_pairs     one wavefront per (test triangle, 64 source triangles),
//                       source geometry staged in LDS, one lane per source
//                       triangle, quadrature moments accumulated in registers
//   K2 k_fill_singular  FP64 self terms (tf == ts) of all triangles, EFIE.cpp:231-542,
//                       Miscellaneous.cpp:32-77
//   K1b k_fill_gather   Z(m,n) = sum over sides of l_m l_n s_m (Ztri(n+) - Ztri(n-))
#include <cmath>

#include "em_device.h"
#include "internal.h"

namespace emfa {

// ---------------------------------------------------------------------------
// K1: regular triangle pairs.
//   KIND 0 (EFIE):  Ztri = cE * sum w (1/4 rho_f.rho_s - 1/k^2) G
//   KIND 1 (CFIE):  Ztri = cE * (same) + cM * sum w rho_f.(n_f x (u x rho_s)) (1+jkR) G/R^2
// with G = exp(-jkR)/R, u = r_p - r_q, rho_f = r_p - v_a, rho_s = r_q - v_b.
// Points are kept relative to each triangle's centroid (x_p, y_q) and the
// integrand is accumulated as moments, from which the 9 (a, b) values follow:
//   rho_f.rho_s = x.y - x.B - A.y + A.B          (A = v_a - c_f, B = v_b - c_s)
//   rho_f.(n x (u x rho_s)) = (rho_f.u)(n.rho_s) - (rho_f.rho_s)(n.u)
// Everything but x_p.y_q depends on p or q alone: with e_p = c_f - c_s + x_p,
// u = e_p - y_q and, since n.x_p = 0, n.u = n.(c_f - c_s) - n.y_q.  So an
// evaluation adds w G and the magnetic kernel to sums per p, sums per q and sums
// weighted with x_p.y_q and n.y_q, and the vector moments are formed once per p
// and per q.
// VALU-bound: instructions per evaluation.  26.2M CFIE pairs (5120 triangles,
// 3 points, FP32) 1.23 -> 0.95 ms (2.5e11 evaluations/s, 2 TB/s of scratch
// written); EFIE, 7 points, FP64, 3042 triangles 4.0 -> 1.28 ms, against
// library roots, divisions and sincos and moments formed per evaluation.
// ---------------------------------------------------------------------------
template <typename R>
__device__ __forceinline__ void axpy3(R *v, R s, const R *x) {
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] += s * x[c];
}

template <typename R, int Q, int KIND>
__global__ __launch_bounds__(256) void k_fill_pairs(const R *__restrict__ tg, int T, int t0, int tcount, R k, R kq,
                                                    R kl, R ik2, R cE, R cM, cx<R> *__restrict__ Ztri) {
    __shared__ R s_src[12][64];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int tsb = blockIdx.x * 64;
    for (int i = threadIdx.x; i < 12 * 64; i += 256) {
        int f = i >> 6, l = i & 63, ts = tsb + l;
        s_src[f][l] = ts < T ? tg[(size_t)f * T + ts] : R(0);
    }
    __syncthreads();
    const int tfl = blockIdx.y * 4 + wave;
    if (tfl >= tcount) return;
    const int tf = __builtin_amdgcn_readfirstlane(t0 + tfl);
    const int ts = tsb + lane;
    if (ts >= T || ts == tf) return;  // self terms: K2

    R Af[3][3], nf[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) nf[c] = tg[(size_t)(12 + c) * T + tf];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int c = 0; c < 3; ++c) Af[i][c] = tg[(size_t)(3 + 3 * i + c) * T + tf];
    R Bs[3][3], d0[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) d0[c] = tg[(size_t)c * T + tf] - s_src[c][lane];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int c = 0; c < 3; ++c) Bs[i][c] = s_src[3 + 3 * i + c][lane];

    R y[Q][3], ny[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
#pragma unroll
        for (int c = 0; c < 3; ++c)
            y[q][c] = (R)rule<Q>(q, 0) * Bs[0][c] + (R)rule<Q>(q, 1) * Bs[1][c] + (R)rule<Q>(q, 2) * Bs[2][c];
        if (KIND == 1) ny[q] = dot3(nf, y[q]);
    }
    const R nd = KIND == 1 ? dot3(nf, d0) : R(0);

    // EFIE: sums of w G; per q; weighted with x.y; with x
    R gqr[Q], gqi[Q], Sxyr = 0, Sxyi = 0, Sxr[3] = {0, 0, 0}, Sxi[3] = {0, 0, 0};
    // CFIE: sums of the magnetic kernel per q, and per q weighted with x.y; Q1,
    // Q2 (weights n.y u, u), P1, P2 (n.y x.u, x.u), Tx and the totals
    R kqr[Q], kqi[Q], aqr[Q], aqi[Q];
    R P1r = 0, P1i = 0, P2r = 0, P2i = 0, Kr = 0, Ki = 0, Nr = 0, Ni = 0;
    R Q1r[3] = {0, 0, 0}, Q1i[3] = {0, 0, 0}, Q2r[3] = {0, 0, 0}, Q2i[3] = {0, 0, 0};
    R Txr[3] = {0, 0, 0}, Txi[3] = {0, 0, 0};
#pragma unroll
    for (int q = 0; q < Q; ++q) gqr[q] = gqi[q] = kqr[q] = kqi[q] = aqr[q] = aqi[q] = 0;

#pragma unroll(Q == 3 ? 3 : 1)
    for (int p = 0; p < Q; ++p) {
        R x[3], e[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            x[c] = (R)rule<Q>(p, 0) * Af[0][c] + (R)rule<Q>(p, 1) * Af[1][c] + (R)rule<Q>(p, 2) * Af[2][c];
            e[c] = d0[c] + x[c];
        }
        const R wp2 = R(2) * (R)rule<Q>(p, 3);  // root() gives 1 / 2R
        R gpr = 0, gpi = 0, kpr = 0, kpi = 0, npr = 0, npi = 0;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            R u[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) u[c] = e[c] - y[q][c];
            R r, h, sn, cs;
            root(dot3(u, u), &r, &h);
            sincos_kr(r, kq, kl, &sn, &cs);
            const R wir = wp2 * (R)rule<Q>(q, 3) * h;
            const R gr = wir * cs, gi = -wir * sn;  // w * exp(-jkR)/R
            const R xy = dot3(x, y[q]);
            gpr += gr;
            gpi += gi;
            gqr[q] += gr;
            gqi[q] += gi;
            Sxyr += gr * xy;
            Sxyi += gi * xy;
            if (KIND == 1) {
                // w (1 + jkR) G / R^2
                const R kr = k * r, ir2 = R(4) * h * h;
                const R kcr = (gr - kr * gi) * ir2, kci = (gi + kr * gr) * ir2;
                kpr += kcr;
                kpi += kci;
                npr += kcr * ny[q];
                npi += kci * ny[q];
                kqr[q] += kcr;
                kqi[q] += kci;
                aqr[q] += kcr * xy;
                aqi[q] += kci * xy;
            }
        }
        axpy3(Sxr, gpr, x);
        axpy3(Sxi, gpi, x);
        if (KIND == 1) {
            const R xe = dot3(x, e);
            P1r += xe * npr;
            P1i += xe * npi;
            P2r += xe * kpr;
            P2i += xe * kpi;
            axpy3(Q1r, npr, e);
            axpy3(Q1i, npi, e);
            axpy3(Q2r, kpr, e);
            axpy3(Q2i, kpi, e);
            axpy3(Txr, nd * kpr - npr, x);
            axpy3(Txi, nd * kpi - npi, x);
            Kr += kpr;
            Ki += kpi;
            Nr += npr;
            Ni += npi;
        }
    }
    R S0r = 0, S0i = 0, Syr[3] = {0, 0, 0}, Syi[3] = {0, 0, 0}, Tyr[3] = {0, 0, 0}, Tyi[3] = {0, 0, 0};
    R Txyr = 0, Txyi = 0;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        S0r += gqr[q];
        S0i += gqi[q];
        axpy3(Syr, gqr[q], y[q]);
        axpy3(Syi, gqi[q], y[q]);
        if (KIND == 1) {
            const R nu = nd - ny[q];
            axpy3(Tyr, nu * kqr[q], y[q]);
            axpy3(Tyi, nu * kqi[q], y[q]);
            axpy3(Q2r, -kqr[q], y[q]);
            axpy3(Q2i, -kqi[q], y[q]);
            axpy3(Q1r, -ny[q] * kqr[q], y[q]);
            axpy3(Q1i, -ny[q] * kqi[q], y[q]);
            P2r -= aqr[q];
            P2i -= aqi[q];
            P1r -= ny[q] * aqr[q];
            P1i -= ny[q] * aqi[q];
            Txyr += nu * aqr[q];
            Txyi += nu * aqi[q];
        }
    }
    const R T0r = nd * Kr - Nr, T0i = nd * Ki - Ni;

    cx<R> *out = Ztri + (size_t)(tfl * 9) * T + ts;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            const R *A = Af[a];
            const R *B = Bs[b];
            R AB = dot3(A, B);
            R Ir = R(0.25) * (Sxyr - dot3(Sxr, B) - dot3(A, Syr) + AB * S0r) - ik2 * S0r;
            R Ii = R(0.25) * (Sxyi - dot3(Sxi, B) - dot3(A, Syi) + AB * S0i) - ik2 * S0i;
            R zr = -cE * Ii;  // the electric part's factor is imaginary
            R zi = cE * Ir;
            if (KIND == 1) {
                R nB = dot3(nf, B);
                R mr = (P1r - nB * P2r - dot3(A, Q1r) + nB * dot3(A, Q2r)) -
                       (Txyr - dot3(Txr, B) - dot3(A, Tyr) + AB * T0r);
                R mi = (P1i - nB * P2i - dot3(A, Q1i) + nB * dot3(A, Q2i)) -
                       (Txyi - dot3(Txi, B) - dot3(A, Tyi) + AB * T0i);
                zr += cM * mr;
                zi += cM * mi;
            }
            out[(size_t)(a * 3 + b) * T] = {zr, zi};
        }
    }
}

// ---------------------------------------------------------------------------
// K2: self terms in FP64 (EFIE.cpp:231-542, Miscellaneous.cpp:32-77), one lane
// per triangle and point p: a group of G lanes forms the nine (a, b) values of
// a triangle, point by point, and adds them over its lanes.  All triangles in
// one launch: it is a chain of logarithms and divisions, 18 us whatever the
// count as one thread per (a, b) looping over the points.
// ---------------------------------------------------------------------------
template <typename R, int Q>
__global__ __launch_bounds__(64) void k_fill_singular(const double *__restrict__ tg, int T, int kind, double k,
                                                      double alpha, double sig_re, double sig_im, int cfie_mode,
                                                      cx<R> *__restrict__ Zself, double *__restrict__ Zsig) {
    constexpr int G = Q == 3 ? 4 : 8;
    const int p = threadIdx.x % G, tf = blockIdx.x * (64 / G) + threadIdx.x / G;
    double zr[9], zi[9], gs[9];
#pragma unroll
    for (int ab = 0; ab < 9; ++ab) zr[ab] = zi[ab] = gs[ab] = 0;
    if (tf < T && p < Q) {
        d3 t[3];
        for (int i = 0; i < 3; ++i)
            t[i] = mk3(tg[(size_t)(3 + 3 * i) * T + tf], tg[(size_t)(4 + 3 * i) * T + tf],
                       tg[(size_t)(5 + 3 * i) * T + tf]);
        const double area = tg[(size_t)15 * T + tf], ik2 = 1.0 / (k * k), wp = rule<Q>(p, 3);
        auto point = [&](int q) { return t[0] * rule<Q>(q, 0) + t[1] * rule<Q>(q, 1) + t[2] * rule<Q>(q, 2); };
        const d3 r = point(p);
        // Taylor part (exp(-jkR)-1)/R ~ -jk - k^2 R/2 + j k^3 R^2/6 (EFIE.cpp:251-256)
        double er[9], ei[9];
#pragma unroll
        for (int ab = 0; ab < 9; ++ab) er[ab] = ei[ab] = 0;
#pragma unroll 1
        for (int q = 0; q < Q; ++q) {
            const d3 rq = point(q);
            const double Rd = normd(r - rq), f = wp * rule<Q>(q, 3);
            const double cr = -0.5 * k * k * Rd * f, ci = (k / 6.0) * (k * k * Rd * Rd - 6.0) * f;
#pragma unroll
            for (int ab = 0; ab < 9; ++ab) {
                const double g = 0.25 * dotd(r - t[ab / 3], rq - t[ab % 3]) - ik2;
                er[ab] += g * cr;
                ei[ab] += g * ci;
            }
        }
        const bool quirk = kind == EMFA_CFIE && cfie_mode == 0;
        d3 Is1 = mk3(0, 0, 0);
        double pot = 0;
        if (quirk) {
            // Miscellaneous.cpp:53-66: in-plane log terms with the last inner rho_s
#pragma unroll 1
            for (int i = 0; i < 3; ++i) {
                const d3 va = t[i], vb = t[i == 2 ? 0 : i + 1], Li = unitd(vb - va);
                const double Lp = dotd(vb - r, Li), Lm = dotd(va - r, Li), Rp = normd(vb - r), Rm = normd(va - r);
                const double P0 = normd(va + Li * dotd(r - va, Li) - r);
                if (P0 > 1e-10) pot += P0 * log((Rp + Lp) / (Rm + Lm));
            }
        } else {
            potentials(t, r, &Is1, &pot);
        }
        const double ce = k * kZ0 / (4.0 * kPi);
        const d3 last = point(Q - 1);
#pragma unroll
        for (int ab = 0; ab < 9; ++ab) {
            const d3 rf = r - t[ab / 3], rs = r - t[ab % 3];
            const double same = wp * dotd(rf, rs);
            const double e2 = quirk ? wp * (0.25 * dotd(rf, last - t[ab % 3]) - ik2) * pot
                                    : wp * (0.25 * dotd(rf, Is1 + rs * pot) - pot * ik2);
            // coefE = j k Z0 / 4 pi applied to (Ze1 + Ze2 / area)
            const double vr = -ce * ei[ab], vi = ce * (er[ab] + e2 / area);
            if (kind == EMFA_EFIE) {
                zr[ab] = vr;
                zi[ab] = vi;
                // Sigma term (EFIE.cpp:297-306), coefE included: 1 / (4 S)
                gs[ab] = same / (4.0 * area);
            } else {
                zr[ab] = alpha * vr + (1.0 - alpha) * kZ0 * same / (8.0 * area);
                zi[ab] = alpha * vi;
            }
        }
    }
#pragma unroll
    for (int ab = 0; ab < 9; ++ab) {
#pragma unroll
        for (int o = 1; o < G; o *= 2) {
            zr[ab] += __shfl_xor(zr[ab], o);
            zi[ab] += __shfl_xor(zi[ab], o);
            if (Zsig) gs[ab] += __shfl_xor(gs[ab], o);
        }
        if (tf < T && p == ab % G) {
            Zself[(size_t)tf * 9 + ab] = {(R)zr[ab], (R)zi[ab]};
            if (Zsig) {
                Zsig[2 * ((size_t)tf * 9 + ab)] = gs[ab] * sig_re;
                Zsig[2 * ((size_t)tf * 9 + ab) + 1] = gs[ab] * sig_im;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Gather: for rows m with a triangle in the chunk,
//   Z(m,n) (+)= l_m l_n s_m [Ztri(tf,a_m; n+, b_n+) - Ztri(tf,a_m; n-, b_n-)]
//               + l_m l_n [Zsig(tf,a_m,b) for the source triangle equal to tf]
// summed over the row's sides in the chunk, plus side first.  A row with both
// triangles in the chunk is written once, by its plus side; one that spans two
// chunks is written with the first and added to with the second, so every
// entry is written and none is cleared beforehand.  A workgroup takes
// kGatherRows half functions (tf, a) on 256 columns and reads the columns'
// tables once.
// HBM: the scratch once, Z once.  5120 triangles, FP32: 0.51 ms, 4.6 TB/s
// (clearing Z and adding each side in a launch of its own: 0.88 ms).  Gathering
// a chunk on a second stream during the next one's pairs gained nothing.
// ---------------------------------------------------------------------------
constexpr int kGatherRows = 4;

template <typename R>
__global__ __launch_bounds__(256) void k_fill_gather(const int *__restrict__ t2r, const int *__restrict__ rtp,
                                                     const int *__restrict__ rtm, const int *__restrict__ rap,
                                                     const int *__restrict__ ram, const R *__restrict__ rlen, int T,
                                                     int N, int t0, int tcount, const cx<R> *__restrict__ Ztri,
                                                     const cx<R> *__restrict__ Zself,
                                                     const double *__restrict__ Zsig, cx<R> *__restrict__ Z) {
    const int n = blockIdx.x * 256 + threadIdx.x;
    if (n >= N) return;
    const int tp = rtp[n], tm = rtm[n], bp = rap[n], bm = ram[n];
    const size_t op = (size_t)bp * T + tp, om = (size_t)bm * T + tm;
    const R ln = rlen[n];
    // the side of row m on half function h = 3 tfl + a of the chunk
    auto side = [&](int h, R s, R *vr, R *vi) {
        const cx<R> *row = Ztri + (size_t)h * 3 * T;
        const int tf = t0 + h / 3;
        const cx<R> *own = Zself + 9 * (size_t)t0 + 3 * (size_t)h;
        const cx<R> zp = tp == tf ? own[bp] : row[op], zm = tm == tf ? own[bm] : row[om];
        *vr = s * (zp.re - zm.re);
        *vi = s * (zp.im - zm.im);
        if (Zsig) {
            const double *zs = Zsig + 18 * (size_t)t0 + 6 * (size_t)h;
            if (tp == tf) {
                *vr += (R)zs[2 * bp];
                *vi += (R)zs[2 * bp + 1];
            }
            if (tm == tf) {
                *vr += (R)zs[2 * bm];
                *vi += (R)zs[2 * bm + 1];
            }
        }
    };
#pragma unroll
    for (int i = 0; i < kGatherRows; ++i) {
        const int e = blockIdx.y * kGatherRows + i;
        if (e >= 3 * tcount) return;
        const int tf = t0 + e / 3, a = e % 3, code = t2r[(size_t)a * T + tf];
        if (code == 0) continue;
        const bool plus = code > 0;
        const int m = (plus ? code : -code) - 1;
        const int other = plus ? rtm[m] : rtp[m];
        const bool both = other >= t0 && other < t0 + tcount;
        if (both && !plus) continue;
        R vr, vi;
        side(e, plus ? R(1) : R(-1), &vr, &vi);
        const R ll = rlen[m] * ln;
        cx<R> *z = Z + (size_t)m * N + n;
        cx<R> old = {R(0), R(0)};
        if (other < t0) old = *z;
        cx<R> v = {old.re + ll * vr, old.im + ll * vi};
        if (both) {
            side(3 * (other - t0) + ram[m], R(-1), &vr, &vi);
            v = {v.re + ll * vr, v.im + ll * vi};
        }
        *z = v;
    }
}

template <typename R>
static emfa_status fill_impl(emfa_ctx *ctx, const emfa_mesh *M, const emfa_fill_params *p, emfa_mat *Zm) {
    const int T = M->nt, N = M->n;
    const R *tg = nullptr;
    const R *rlen = nullptr;
    if constexpr (sizeof(R) == 4) {
        tg = (const R *)M->tg32;
        rlen = (const R *)M->rlen32;
    } else {
        tg = (const R *)M->tg64;
        rlen = (const R *)M->rlen64;
    }
    const bool sigma = p->kind == EMFA_EFIE && std::hypot(p->sigma_re, p->sigma_im) > 1e-8;
    const size_t per_tri = 9 * (size_t)T * sizeof(cx<R>);
    size_t budget = (size_t)2 << 30;
    if (const char *s = getenv("EMFA_FILL_SCRATCH_MB")) budget = (size_t)atol(s) << 20;
    int chunk = (int)std::min<size_t>((size_t)T, std::max<size_t>(4, budget / per_tri));
    chunk = std::min(chunk, 16384);
    chunk = (chunk + 3) & ~3;
    const size_t buf_b = ((size_t)chunk * per_tri + 255) & ~(size_t)255;
    const size_t self_b = (9 * (size_t)T * sizeof(cx<R>) + 255) & ~(size_t)255;
    void *scr = nullptr;
    emfa_status st = ctx_scratch(ctx, buf_b + self_b + (sigma ? 18 * (size_t)T * sizeof(double) : 0), &scr);
    if (st != EMFA_OK) return st;
    cx<R> *Ztri = (cx<R> *)scr;
    cx<R> *Zself = (cx<R> *)((char *)scr + buf_b);
    double *Zsig = sigma ? (double *)((char *)Zself + self_b) : nullptr;
    cx<R> *Z = (cx<R> *)Zm->d;

    const double k = p->k;
    const double ce = k * kZ0 / (4.0 * kPi);  // |j k Z0 / 4 pi|
    R cE = (R)ce, cM = 0;  // the electric part's factor is j cE
    if (p->kind == EMFA_CFIE) {
        cE = (R)(p->alpha * ce);
        cM = (R)((1.0 - p->alpha) * kZ0 / (16.0 * kPi));
    }
    const R kr = (R)k, ik2 = (R)(1.0 / (k * k));
    R kq, kl;
    quarter_turns(k, &kq, &kl);
    {
        constexpr int per7 = 64 / 8, per3 = 64 / 4;  // triangles per workgroup
        if (p->quad == 7)
            k_fill_singular<R, 7><<<(T + per7 - 1) / per7, 64, 0, ctx->stream>>>(
                M->tg64, T, p->kind, k, p->alpha, p->sigma_re, p->sigma_im, p->cfie_mode, Zself, Zsig);
        else
            k_fill_singular<R, 3><<<(T + per3 - 1) / per3, 64, 0, ctx->stream>>>(
                M->tg64, T, p->kind, k, p->alpha, p->sigma_re, p->sigma_im, p->cfie_mode, Zself, Zsig);
        EMFA_HIP_CHECK(hipGetLastError());
    }
    for (int t0 = 0; t0 < T; t0 += chunk) {
        int tc = std::min(chunk, T - t0);
        {
            ProfScope ps(ctx, "fill_pairs", (double)tc * T * p->quad * p->quad);
            dim3 grid((T + 63) / 64, (tc + 3) / 4);
#define LAUNCH_PAIRS(Q, KIND) \
    k_fill_pairs<R, Q, KIND><<<grid, 256, 0, ctx->stream>>>(tg, T, t0, tc, kr, kq, kl, ik2, cE, cM, Ztri)
            if (p->quad == 7) {
                if (p->kind == EMFA_EFIE)
                    LAUNCH_PAIRS(7, 0);
                else
                    LAUNCH_PAIRS(7, 1);
            } else {
                if (p->kind == EMFA_EFIE)
                    LAUNCH_PAIRS(3, 0);
                else
                    LAUNCH_PAIRS(3, 1);
            }
#undef LAUNCH_PAIRS
            EMFA_HIP_CHECK(hipGetLastError());
        }
        {
            ProfScope ps(ctx, "fill_gather", 0);
            dim3 grid((N + 255) / 256, (tc * 3 + kGatherRows - 1) / kGatherRows);
            k_fill_gather<R><<<grid, 256, 0, ctx->stream>>>(M->t2r, M->rtp, M->rtm, M->rap, M->ram, rlen, T, N, t0,
                                                            tc, Ztri, Zself, Zsig, Z);
            EMFA_HIP_CHECK(hipGetLastError());
        }
    }
    return EMFA_OK;
}

}  // namespace emfa

using namespace emfa;

extern "C" emfa_status emfa_fill(emfa_ctx *ctx, const emfa_mesh *mesh, const emfa_fill_params *p, emfa_mat *Z) {
    EMFA_REQUIRE(ctx && mesh && p && Z, EMFA_E_INVALID, "emfa_fill: null argument");
    EMFA_REQUIRE(Z->rows == mesh->n && Z->cols == mesh->n, EMFA_E_INVALID, "emfa_fill: Z is %dx%d, mesh has %d RWGs",
                 Z->rows, Z->cols, mesh->n);
    EMFA_REQUIRE(p->kind == EMFA_EFIE || p->kind == EMFA_CFIE, EMFA_E_INVALID, "emfa_fill: bad kind %d", p->kind);
    EMFA_REQUIRE(p->quad == 3 || p->quad == 7, EMFA_E_INVALID, "emfa_fill: quadrature must be 3 or 7 (got %d)",
                 p->quad);
    EMFA_REQUIRE(p->k > 0, EMFA_E_INVALID, "emfa_fill: wave number must be positive");
    EMFA_HIP_CHECK(hipSetDevice(ctx->device));
    if (Z->prec == EMFA_F32) return fill_impl<float>(ctx, mesh, p, Z);
    return fill_impl<double>(ctx, mesh, p, Z);
}
