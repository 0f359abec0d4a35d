// mgs_tail_dev.h -- device side of the single-workgroup tails of the plain FP64
// cycles and of the mixed nDGP inner cycle (mgs_tail.hip), shared with the
// batched serving kernels.
#pragma once

#include "mgs_dgp_dev.h"
#include "mgs_fr_dev.h"

namespace mgs {

// A cell in the tail's LDS arrays, which are lexicographic (x fastest): its
// place and the steps to its periodic neighbours (an edge neighbour's step is
// the sum of two).
struct LexCell {
    int me, xp, xm, yp, ym, zp, zm;
};

__device__ __forceinline__ LexCell lex_cell(const Geo& g, int i, int j, int k)
{
    const int n = g.n, nn = n * n;
    LexCell q;
    q.me = k * nn + j * n + i;
    q.xp = i == n - 1 ? 1 - n : 1;
    q.xm = i == 0 ? n - 1 : -1;
    q.yp = j == n - 1 ? n - nn : n;
    q.ym = j == 0 ? nn - n : -n;
    q.zp = k == n - 1 ? nn - n * nn : nn;
    q.zm = k == 0 ? n * nn - nn : -nn;
    return q;
}

// entry t of colour c's half
__device__ __forceinline__ LexCell lex_half(const Geo& g, int c, int t)
{
    int m, j, k;
    half_mjk(g, t, m, j, k);
    return lex_cell(g, 2 * m + ((c + j + k) & 1), j, k);
}

template <typename T>
__device__ __forceinline__ S19<T> lex_s19(const T* u, const LexCell& q)
{
    const T* p = u + q.me;
    S19<T> s;
    s.c0 = p[0];
    s.xp = p[q.xp];
    s.xm = p[q.xm];
    s.yp = p[q.yp];
    s.ym = p[q.ym];
    s.zp = p[q.zp];
    s.zm = p[q.zm];
    s.xy_pp = p[q.xp + q.yp];
    s.xy_mm = p[q.xm + q.ym];
    s.xy_pm = p[q.xp + q.ym];
    s.xy_mp = p[q.xm + q.yp];
    s.xz_pp = p[q.xp + q.zp];
    s.xz_mm = p[q.xm + q.zm];
    s.xz_pm = p[q.xp + q.zm];
    s.xz_mp = p[q.xm + q.zp];
    s.yz_pp = p[q.yp + q.zp];
    s.yz_mm = p[q.ym + q.zm];
    s.yz_pm = p[q.yp + q.zm];
    s.yz_mp = p[q.ym + q.zp];
    return s;
}

// What differs between the three cycles: the element type, the new value and
// the residual of a cell, whether a colour pass reads its own colour (JACOBI:
// every cell from the values before the pass), the correction's sum and
// guard, and the coarsest level's sweeps.
template <int FRN>
struct TailFr64 {
    using T = double;
    using Coef = FrCoef;
    static constexpr bool JACOBI = false, BASE = false, WRITE_BACK = true;
    static constexpr int COARSEST_PAIRS = 2;
    static __device__ __forceinline__ double update(const Coef& c, const double* u, const double*, const LexCell& q,
                                                    double rho, double f, bool)
    {
        double v;
        const FrSmoothOp<FRN, true, false> op{&v, nullptr, nullptr, c};
        const double* p = u + q.me;
        op.update(0u, 0u, typename FrSmoothOp<FRN, true, false>::Own{rho, f}, 0.0, p[q.xp], p[q.xm], p[q.yp], p[q.ym],
                  p[q.zp], p[q.zm]);
        return v;
    }
    static __device__ __forceinline__ double resid(const Coef& c, const double* u, const double*, const LexCell& q,
                                                   double rho, double sub)
    {
        const FrResOp<FRN, true> op{nullptr, nullptr, nullptr, nullptr, c};
        const double* p = u + q.me;
        return op.cell(0u, typename FrResOp<FRN, true>::Own{rho, sub}, p[0], p[q.xp], p[q.xm], p[q.yp], p[q.ym], p[q.zp],
                       p[q.zm]);
    }
    static __device__ __forceinline__ void add(double& P, double w, double vh, double vr)
    {
        P = P + w * vh;
        P = P - w * vr;
    }
    static __device__ __forceinline__ bool keep(double v) { return v > 0.0; }
};

struct TailDgp64 {
    using T = double;
    using Coef = DgpCoef;
    static constexpr bool JACOBI = true, BASE = false, WRITE_BACK = true;
    static constexpr int COARSEST_PAIRS = 2;
    static __device__ __forceinline__ double resid(const Coef& c, const double* u, const double*, const LexCell& q,
                                                   double rho, double sub)
    {
        return dgp_L19(lex_s19(u, q), rho, c) - sub;
    }
    static __device__ __forceinline__ double update(const Coef& c, const double* u, const double* pb, const LexCell& q,
                                                    double rho, double f, bool)
    {
        const double dLphi = -6.0 / c.dx2;
        return u[q.me] - resid(c, u, pb, q, rho, f) / dLphi;
    }
    static __device__ __forceinline__ void add(double& P, double w, double vh, double vr)
    {
        P = P + w * vh;
        P = P - w * vr;
    }
    static __device__ __forceinline__ bool keep(double) { return true; }
};

struct TailDgpm {
    using T = float;
    using Coef = DgpF;
    static constexpr bool JACOBI = true, BASE = true, WRITE_BACK = false;
    static constexpr int COARSEST_PAIRS = 8;
    static __device__ __forceinline__ float resid(const Coef& c, const float* e, const float* pb, const LexCell& q,
                                                  float rho, float sub)
    {
        return dgp_dop(d2_of(lex_s19(pb, q)), d2_of(lex_s19(e, q)), rho, c) - sub;
    }
    static __device__ __forceinline__ float update(const Coef& c, const float* e, const float* pb, const LexCell& q,
                                                   float rho, float f, bool coarsest)
    {
        const D2f de = d2_of(lex_s19(e, q)), db = d2_of(lex_s19(pb, q));
        if (coarsest) {  // the update in FP64 (dgpm_coarsest_block)
            const double D = (double)dgp_dop(db, de, rho, c) - (double)f;
            return (float)((double)de.c0 + D / (6.0 * (double)c.inv_dx2));
        }
        const float D = dgp_dop(db, de, rho, c) - f;
        return de.c0 + over_six(D, c);
    }
    static __device__ __forceinline__ void add(float& P, float w, float vh, float vr) { P += w * (vh - vr); }
    static __device__ __forceinline__ bool keep(float) { return true; }
};

template <class MD>
struct PTailLevel {
    Geo g;
    typename MD::T *u, *f, *res, *rres, *ru;
    const double* rho;
    const float* pb;
    typename MD::Coef c;
};

constexpr int PTAIL_MAXL = 4;  // 16^3, 8^3, 4^3, 2^3

template <class MD>
struct PTailDesc {
    int nl;  // levels below the first
    PTailLevel<MD> L[PTAIL_MAXL];
};

// LDS arrays of a level: u, rho, f, res and the base of the mixed form; below
// the first level also R r and R u
template <class MD>
struct PTailArrays {
    typename MD::T *u, *rho, *f, *res, *pb, *rres, *ru;
};

template <class MD>
constexpr int ptail_arrays(int i)
{
    return (i == 0 ? 4 : 6) + (MD::BASE ? 1 : 0);
}

// elements for 16^3 down to 2^3
template <class MD>
constexpr int PTAIL_LDS = ptail_arrays<MD>(0) * 4096 + ptail_arrays<MD>(1) * (512 + 64 + 8);

template <class MD>
__device__ __forceinline__ PTailArrays<MD> ptail_level(const PTailDesc<MD>& G, int i, typename MD::T* lds)
{
    int off = 0;
    for (int q = 0; q < i; q++) off += ptail_arrays<MD>(q) * 2 * (int)G.L[q].g.half;
    const int cells = 2 * (int)G.L[i].g.half;
    typename MD::T* p = lds + off;
    PTailArrays<MD> a;
    a.u = p;
    a.rho = p + cells;
    a.f = p + 2 * cells;
    a.res = p + 3 * cells;
    p += 4 * cells;
    a.pb = MD::BASE ? p : nullptr;
    if (MD::BASE) p += cells;
    a.rres = i > 0 ? p : nullptr;
    a.ru = i > 0 ? p + cells : nullptr;
    return a;
}

template <class MD, bool WAVE>
__device__ __forceinline__ void ptail_smooth(const PTailLevel<MD>& L, const PTailArrays<MD>& l, int pairs, bool coarsest)
{
    using T = typename MD::T;
    const int tid = threadIdx.x, nthr = WAVE ? 64 : TAIL_THREADS, half = (int)L.g.half;
    for (int pair = 0; pair < pairs; pair++)
        for (int c = 0; c < 2; c++) {
            T v[TAIL_CELLS];
            int me[TAIL_CELLS];
#pragma unroll
            for (int r = 0; r < TAIL_CELLS; r++) {
                const int t = tid + r * nthr;
                if (t >= half) continue;
                const LexCell q = lex_half(L.g, c, t);
                me[r] = q.me;
                v[r] = MD::update(L.c, l.u, l.pb, q, l.rho[q.me], l.f[q.me], coarsest);
                if (!MD::JACOBI) l.u[q.me] = v[r];
            }
            group_sync<WAVE>();
            if (MD::JACOBI) {
#pragma unroll
                for (int r = 0; r < TAIL_CELLS; r++)
                    if (tid + r * nthr < half) l.u[me[r]] = v[r];
                group_sync<WAVE>();
            }
        }
}

// out = L(u) - sub on a whole level
template <class MD, bool WAVE>
__device__ __forceinline__ void ptail_resid(const PTailLevel<MD>& L, const PTailArrays<MD>& l, const typename MD::T* u,
                                            const typename MD::T* sub, typename MD::T* out)
{
    const int nthr = WAVE ? 64 : TAIL_THREADS;
    for (int t = threadIdx.x; t < 2 * (int)L.g.half; t += nthr) {
        int i, j, k;
        coarse_ijk(L.g, t, i, j, k);
        const LexCell q = lex_cell(L.g, i, j, k);
        out[q.me] = MD::resid(L.c, u, l.pb, q, l.rho[q.me], sub[q.me]);
    }
    group_sync<WAVE>();
}

// the 8-child average in restrict8_cell's order
template <typename T>
__device__ __forceinline__ T lex_mean8(const T* a, int n, int o)
{
    T P = a[o];
    P = P + a[o + 1];
    P = P + a[o + n];
    P = P + a[o + n + 1];
    P = P + a[o + n * n];
    P = P + a[o + n * n + 1];
    P = P + a[o + n * n + n];
    P = P + a[o + n * n + n + 1];
    return P / (T)8.0;
}

template <class MD, bool WAVE>
__device__ void ptail_cycle(const PTailDesc<MD>& G, int i0, typename MD::T* lds)
{
    using T = typename MD::T;
    const int tid = threadIdx.x, nthr = WAVE ? 64 : TAIL_THREADS;
    int bottom = G.nl;
    for (int i = i0; i < G.nl; i++) {
        const PTailLevel<MD>&L = G.L[i], &C = G.L[i + 1];
        if (!WAVE && L.g.half <= TAIL_WAVE_HALF) {
            bottom = i;
            break;
        }
        const PTailArrays<MD> l = ptail_level(G, i, lds), c = ptail_level(G, i + 1, lds);
        ptail_smooth<MD, WAVE>(L, l, 2, false);
        ptail_resid<MD, WAVE>(L, l, l.u, l.f, l.res);
        const int n = L.g.n;
        for (int t = tid; t < 2 * (int)C.g.half; t += nthr) {
            int I, J, K;
            coarse_ijk(C.g, t, I, J, K);
            const int o = (2 * K * n + 2 * J) * n + 2 * I;
            c.rres[t] = lex_mean8(l.res, n, o);
            const T v = lex_mean8(l.u, n, o);
            c.ru[t] = v;
            c.u[t] = v;
        }
        group_sync<WAVE>();
        ptail_resid<MD, WAVE>(C, c, c.ru, c.rres, c.f);
    }
    if (bottom < G.nl) {
        if constexpr (!WAVE) {
            if (tid < 64) ptail_cycle<MD, true>(G, bottom, lds);
            __syncthreads();
        }
    } else {
        ptail_smooth<MD, WAVE>(G.L[G.nl], ptail_level(G, G.nl, lds), MD::COARSEST_PAIRS, true);
    }
    for (int i = bottom - 1; i >= i0; i--) {
        const PTailLevel<MD>&L = G.L[i], &C = G.L[i + 1];
        const PTailArrays<MD> l = ptail_level(G, i, lds), c = ptail_level(G, i + 1, lds);
        // u += P (u_H - R u), a thread per fine cell; weights and order of
        // correct64_sons_apply / dgpm_sons_new
        for (int t = tid; t < 2 * (int)L.g.half; t += nthr) {
            int x, y, z;
            coarse_ijk(L.g, t, x, y, z);
            const LexCell q = lex_cell(C.g, x >> 1, y >> 1, z >> 1);
            const int sx = (x & 1) ? q.xp : q.xm, sy = (y & 1) ? q.yp : q.ym, sz = (z & 1) ? q.zp : q.zm;
            const T a = (T)(1.0 / 64.0), b = (T)3.0 * a, c9 = (T)9.0 * a, d = (T)27.0 * a;
            const T wt[8] = {a, b, b, c9, b, c9, c9, d};
            T P = (T)0.0;
#pragma unroll
            for (int ind = 0; ind < 8; ind++) {
                const int o = q.me + ((ind & 1) ? 0 : sx) + ((ind & 2) ? 0 : sy) + ((ind & 4) ? 0 : sz);
                MD::add(P, wt[ind], c.u[o], c.ru[o]);
            }
            const T v = l.u[t] + P;
            if (MD::keep(v)) l.u[t] = v;
        }
        group_sync<WAVE>();
        ptail_smooth<MD, WAVE>(L, l, 2, false);
    }
}

// split <-> lexicographic: entry t of a split level
__device__ __forceinline__ int lex_of_split(const Geo& g, int t)
{
    const int c = t >= (int)g.half ? 1 : 0;
    int m, j, k;
    half_mjk(g, t - c * (int)g.half, m, j, k);
    return (k * g.n + j) * g.n + 2 * m + ((c + j + k) & 1);
}

// the cycle of the levels in G by one workgroup of TAIL_THREADS, out of lds
// (PTAIL_LDS<MD> elements)
template <class MD>
__device__ __forceinline__ void ptail_run(const PTailDesc<MD>& G, typename MD::T* lds)
{
    using T = typename MD::T;
    const int tid = threadIdx.x;
    {
        // the first level's R u, R r and density and every density below, all
        // loads issued before the first is used
        constexpr int NR = 2 * TAIL_CELLS;
        const Geo g = G.L[0].g;
        const PTailArrays<MD> a = ptail_level(G, 0, lds);
        T v[3][NR];
        float b[NR];
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const int t = tid + r * TAIL_THREADS;
            if (t >= 2 * (int)g.half) continue;
            v[0][r] = G.L[0].ru[t];
            v[1][r] = (T)G.L[0].rho[t];
            v[2][r] = G.L[0].rres[t];
            if (MD::BASE) b[r] = G.L[0].pb[t];
        }
        T rc[PTAIL_MAXL];
        float bc[PTAIL_MAXL];
#pragma unroll
        for (int i = 1; i < PTAIL_MAXL; i++)  // at most 8^3 cells
            if (i <= G.nl && tid < 2 * (int)G.L[i].g.half) {
                rc[i] = (T)G.L[i].rho[tid];
                if (MD::BASE) bc[i] = G.L[i].pb[tid];
            }
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const int t = tid + r * TAIL_THREADS;
            if (t >= 2 * (int)g.half) continue;
            const int q = lex_of_split(g, t);
            a.u[q] = v[0][r];
            a.rho[q] = v[1][r];
            a.f[q] = v[2][r];
            if (MD::BASE) a.pb[q] = (T)b[r];
        }
#pragma unroll
        for (int i = 1; i < PTAIL_MAXL; i++)
            if (i <= G.nl && tid < 2 * (int)G.L[i].g.half) {
                const PTailArrays<MD> c = ptail_level(G, i, lds);
                const int q = lex_of_split(G.L[i].g, tid);
                c.rho[q] = rc[i];
                if (MD::BASE) c.pb[q] = (T)bc[i];
            }
        __syncthreads();
        // f = L(R u) - R r in R r's place (a cell reads only its own)
        ptail_resid<MD, false>(G.L[0], a, a.u, a.f, a.f);
    }
    ptail_cycle<MD, false>(G, 0, lds);
    for (int i = 0; i <= G.nl; i++) {
        const PTailLevel<MD>& L = G.L[i];
        const PTailArrays<MD> l = ptail_level(G, i, lds);
        for (int t = tid; t < 2 * (int)L.g.half; t += TAIL_THREADS) {
            const int q = lex_of_split(L.g, t);
            L.u[t] = l.u[q];
            if (!MD::WRITE_BACK) continue;
            L.f[t] = l.f[q];
            if (i < G.nl) L.res[t] = l.res[q];
            if (i > 0) {
                L.rres[t] = l.rres[q];
                L.ru[t] = l.ru[q];
            }
        }
        if (!MD::WRITE_BACK) break;
    }
}

// the chain of levels from n cells a side (nlev of them) is the tail's
inline bool ptail_fits(int n, int nlev) { return nlev >= 2 && nlev <= PTAIL_MAXL && n <= 16; }

}  // namespace mgs
