// mgs_dgp_dev.h -- device-side nDGP operators shared by the standalone
// kernels (mgs_dgp.hip) and the batched serving kernels (mgs_serve.hip):
// the FP64 19-point operator L(phi) of PMP2MGsolver_DGP.f90 and the FP32
// delta-form operator D(e) of the mixed solve, and per-cell bodies of the
// mixed solve's kernels.  The same bodies run in both places, so a request
// served in a batch is bit-identical to mgs_solve.
#pragma once

#include <cmath>

#include "mgs_device.h"
#include "mgs_fr_dev.h"
#include "mgs_internal.h"
#include "mgs_stencil.h"

namespace mgs {

// The 19 points of the stencil at a cell: centre, 6 faces and 12 edges
// (the edges named by their offsets, e.g. pp_xy = (i+1, j+1, k)).  Both the
// per-cell gathers and the z-marching register windows fill one, and the
// operators below read it, so every path adds the same values in the same
// order.
template <typename T>
struct S19 {
    T c0, xp, xm, yp, ym, zp, zm;
    T xy_pp, xy_mm, xy_pm, xy_mp;  // (i+-1, j+-1, k)
    T xz_pp, xz_mm, xz_pm, xz_mp;  // (i+-1, j, k+-1)
    T yz_pp, yz_mm, yz_pm, yz_mp;  // (i, j+-1, k+-1)
};

// the stencil of cell (i, j, k) from a field's colour halves
template <typename T>
__device__ __forceinline__ S19<T> s19_halves(const T* __restrict__ h0, const T* __restrict__ h1, const Geo& g, int i,
                                             int j, int k)
{
    const int n = g.n;
    const int im = wrap_dec(i, n), ip = wrap_inc(i, n);
    const int jm = wrap_dec(j, n), jp = wrap_inc(j, n);
    const int km = wrap_dec(k, n), kp = wrap_inc(k, n);
    // the cell's own colour and the other (n is even: a wrap keeps the parity)
    const bool c = (i + j + k) & 1;
    const T *a = c ? h1 : h0, *b = c ? h0 : h1;
    auto at = [&](const T* h, int x, int y, int z) { return h[row_base(g, y, z) + (unsigned)(x >> 1)]; };
    S19<T> s;
    s.c0 = at(a, i, j, k);
    s.xp = at(b, ip, j, k);
    s.xm = at(b, im, j, k);
    s.yp = at(b, i, jp, k);
    s.ym = at(b, i, jm, k);
    s.zp = at(b, i, j, kp);
    s.zm = at(b, i, j, km);
    s.xy_pp = at(a, ip, jp, k);
    s.xy_mm = at(a, im, jm, k);
    s.xy_pm = at(a, ip, jm, k);
    s.xy_mp = at(a, im, jp, k);
    s.xz_pp = at(a, ip, j, kp);
    s.xz_mm = at(a, im, j, km);
    s.xz_pm = at(a, ip, j, km);
    s.xz_mp = at(a, im, j, kp);
    s.yz_pp = at(a, i, jp, kp);
    s.yz_mm = at(a, i, jm, km);
    s.yz_pm = at(a, i, jp, km);
    s.yz_mp = at(a, i, jm, kp);
    return s;
}

template <typename T>
__device__ __forceinline__ S19<T> s19_at(const T* __restrict__ u, const Geo& g, int i, int j, int k)
{
    return s19_halves(u, u + g.half, g, i, j, k);
}

// Sigma's stencil sums and the Laplacian numerator
__device__ __forceinline__ void dgp_sums(const S19<double>& u, double& se0, double& se1, double& se2, double& lap)
{
    const double dxx = u.xp + u.xm - 2.0 * u.c0;
    const double dyy = u.yp + u.ym - 2.0 * u.c0;
    const double dzz = u.zp + u.zm - 2.0 * u.c0;
    const double cxy = u.xy_pp + u.xy_mm - u.xy_pm - u.xy_mp;
    const double cxz = u.xz_pp + u.xz_mm - u.xz_pm - u.xz_mp;
    const double cyz = u.yz_pp + u.yz_mm - u.yz_pm - u.yz_mp;
    se0 = dxx * dxx + dyy * dyy + dzz * dzz;
    se1 = dxx * dyy + dxx * dzz + dyy * dzz;
    se2 = cxy * cxy + cxz * cxz + cyz * cyz;
    const double s6 = u.xp + u.xm + u.yp + u.ym + u.zp + u.zm;
    lap = s6 - u.c0 * 6.0;
}

// L(phi) at a cell from its stencil values (without the FAS right-hand side)
__device__ __forceinline__ double dgp_L19(const S19<double>& u, double rho, const DgpCoef& c)
{
    const double TWOOVERTHREE = 2.0 / 3.0, ONEOVEREIGHT = 0.125, THREEOVERFOUR = 0.75, EIGHTOVERTHREE = 8.0 / 3.0;
    double se0, se1, se2, lap;
    dgp_sums(u, se0, se1, se2, lap);
    double Sigma = c.fct1 * rho;
    // the reference divides by dx^4 and dx^2; dx is a power of two, so the
    // products with the exact reciprocals are the same numbers
    Sigma = Sigma + se0 * TWOOVERTHREE * c.inv_dx4 - se1 * TWOOVERTHREE * c.inv_dx4 + se2 * ONEOVEREIGHT * c.inv_dx4;
    return lap * c.inv_dx2 - (copysign(1.0, c.alpha) * sqrt(c.alpha * c.alpha + EIGHTOVERTHREE * Sigma) - c.alpha) *
                                 THREEOVERFOUR;
}

// L(phi) at absolute cell (i, j, k); c0: the cell's value
__device__ __forceinline__ double dgp_L(const double* __restrict__ u, const Geo& g, int i, int j, int k, double rho,
                                        const DgpCoef& c, double& c0)
{
    const S19<double> s = s19_at(u, g, i, j, k);
    c0 = s.c0;
    return dgp_L19(s, rho, c);
}

// second differences, face sum and centre of a field at a cell
struct D2f {
    float xx, yy, zz, xy, xz, yz, s6, c0;
};

__device__ __forceinline__ D2f d2_of(const S19<float>& u)
{
    D2f d;
    d.c0 = u.c0;
    d.xx = u.xp + u.xm - 2.0f * d.c0;
    d.yy = u.yp + u.ym - 2.0f * d.c0;
    d.zz = u.zp + u.zm - 2.0f * d.c0;
    d.xy = u.xy_pp + u.xy_mm - u.xy_pm - u.xy_mp;
    d.xz = u.xz_pp + u.xz_mm - u.xz_pm - u.xz_mp;
    d.yz = u.yz_pp + u.yz_mm - u.yz_pm - u.yz_mp;
    d.s6 = u.xp + u.xm + u.yp + u.ym + u.zp + u.zm;
    return d;
}

__device__ __forceinline__ D2f d2_at(const float* __restrict__ u, const Geo& g, int i, int j, int k)
{
    return d2_of(s19_at(u, g, i, j, k));
}

struct DgpF {
    float alpha, fct1, inv_dx2, inv_dx4, sgn;
    float six, rsix;  // 6 / dx^2 and its reciprocal
};

inline DgpF dgpf(const DgpCoef& c)
{
    const float inv_dx2 = (float)(1.0 / c.dx2), six = 6.0f * inv_dx2;
    return DgpF{(float)c.alpha, (float)c.fct1, inv_dx2, (float)(1.0 / c.dx4), (float)std::copysign(1.0, c.alpha),
                six,            1.0f / six};
}

// The passes of the large levels are bound by the vector ALU (a cell is some
// 200 instructions), so the quotient and the roots come without the scaling
// steps that general ones carry for results or operands near the ends of the
// FP32 range.

// x / c.six, correctly rounded where |x| >= 2^-100: two corrections by the exact
// remainder with the correctly rounded reciprocal (the first leaves q within an
// ulp, where the second is exact rounding); below, where the remainder itself is
// rounded, within 2^-149 / c.six of that.  An infinity, a NaN
// and an overflow of the first product (for c.six < 1, where the quotient
// overflows too, but for its last place) pass through, as in a division.
__host__ __device__ __forceinline__ float over_six(float x, const DgpF& c)
{
    const float p = x * c.rsix;
    float q = fmaf(fmaf(-p, c.six, x), c.rsix, p);
    q = fmaf(fmaf(-q, c.six, x), c.rsix, q);
    return fabsf(p) <= __FLT_MAX__ ? q : p;
}

// sqrt(x), x >= 0, correctly rounded for x >= 2^-100 and infinite x (below, to an
// ulp; dgp_dop's operands are 0 or at least 2^-25 alpha^2): the hardware's root
// is within an ulp, and the signs of the fused remainders x - lo s and x - hi s
// with its two neighbours lo and hi, the usual correction, pick the right one
__device__ __forceinline__ float sqrt_pos(float x)
{
    const float s = __builtin_amdgcn_sqrtf(x);
    const float lo = __int_as_float(__float_as_int(s) - 1), hi = __int_as_float(__float_as_int(s) + 1);
    const float rl = fmaf(-lo, s, x), rh = fmaf(-hi, s, x);
    const float t = rl <= 0.0f ? lo : s;
    return rh > 0.0f ? hi : t;
}

// D(e) at a cell from the base's and the increment's second differences
__device__ __forceinline__ float dgp_dop(const D2f& b, const D2f& e, float rho, const DgpF& c)
{
    const float Qb = b.xx * b.xx + b.yy * b.yy + b.zz * b.zz - b.xx * b.yy - b.xx * b.zz - b.yy * b.zz;
    const float Cb = b.xy * b.xy + b.xz * b.xz + b.yz * b.yz;
    const float Sig = c.fct1 * rho + ((2.0f / 3.0f) * Qb + 0.125f * Cb) * c.inv_dx4;
    const float Bx = 2.0f * b.xx - b.yy - b.zz, By = 2.0f * b.yy - b.xx - b.zz, Bz = 2.0f * b.zz - b.xx - b.yy;
    const float Qe = e.xx * e.xx + e.yy * e.yy + e.zz * e.zz - e.xx * e.yy - e.xx * e.zz - e.yy * e.zz;
    const float lin = Bx * e.xx + By * e.yy + Bz * e.zz;
    const float cross = 2.0f * (b.xy * e.xy + b.xz * e.xz + b.yz * e.yz) + e.xy * e.xy + e.xz * e.xz + e.yz * e.yz;
    const float dSig = ((2.0f / 3.0f) * (lin + Qe) + 0.125f * cross) * c.inv_dx4;
    const float a2 = c.alpha * c.alpha;
    const float So = sqrt_pos(fmaxf(a2 + (8.0f / 3.0f) * Sig, 0.0f));
    const float Sn = sqrt_pos(fmaxf(a2 + (8.0f / 3.0f) * (Sig + dSig), 0.0f));
    const float den = So + Sn;
    const bool ok = den > 0.0f;  // (a division per lane rather than a branch around it)
    const float q = 2.0f * c.sgn * dSig / (ok ? den : 1.0f), nl = ok ? q : 0.0f;
    return (e.s6 - 6.0f * e.c0) * c.inv_dx2 - nl;
}

// ---------------------------------------------------------------------------
// per-cell bodies of the mixed nDGP kernels
// ---------------------------------------------------------------------------

// one colour pass of the inner smoother at the cell (m, row = j + n k) of
// colour `colour`: the increment's halves e0, e1 in, the colour's new half out
__device__ __forceinline__ void dgpm_smooth_cell(const float* __restrict__ e0, const float* __restrict__ e1,
                                                 const float* __restrict__ pb, const double* __restrict__ rho,
                                                 const float* __restrict__ rhs, float* __restrict__ out, const Geo& g,
                                                 int colour, const DgpF& c, int m, unsigned row)
{
    const int j = (int)(row % (unsigned)g.n), k = (int)(row / (unsigned)g.n);
    const int i = 2 * m + ((colour + j + k) & 1);
    const size_t me = (size_t)colour * g.half + row_base(g, j, k) + m;
    const D2f de = d2_of(s19_halves(e0, e1, g, i, j, k)), db = d2_at(pb, g, i, j, k);
    const float D = dgp_dop(db, de, (float)rho[me], c) - rhs[me];
    out[row_base(g, j, k) + m] = de.c0 + over_six(D, c);
}

// out = D(e) - rhs at the cell (m, row2) of both colours (row2 < n^2:
// colour 0, else colour 1)
__device__ __forceinline__ void dgpm_residual_cell(const float* __restrict__ e, const float* __restrict__ pb,
                                                   const double* __restrict__ rho, const float* __restrict__ rhs,
                                                   float* __restrict__ out, const Geo& g, const DgpF& c, int m,
                                                   unsigned row2)
{
    const unsigned nn = (unsigned)g.n * (unsigned)g.n;
    const int col = row2 >= nn ? 1 : 0;
    const unsigned r2 = row2 - (unsigned)col * nn;
    const int j = (int)(r2 % (unsigned)g.n), k = (int)(r2 / (unsigned)g.n);
    const int i = 2 * m + ((col + j + k) & 1);
    const size_t me = (size_t)col * g.half + row_base(g, j, k) + m;
    out[me] = dgp_dop(d2_at(pb, g, i, j, k), d2_at(e, g, i, j, k), (float)rho[me], c) - rhs[me];
}

// The increment of a colour-0 cell after the inner smoother's first pass from
// e = 0 (where D(0) = 0): 0 + (0 - rhs) / (6 / dx^2), as dgpm_smooth_cell
// would form it.  The outer residual writes it, which saves that pass.
__device__ __forceinline__ float dgpm_first(float rhs, float inv_dx2) { return (0.0f - rhs) / (6.0f * inv_dx2); }

// FP64 outer residual r = L(phi) at the cell (m, row2) of both colours, and
// the inner problem's data there: g = -r, phi_b = phi in FP32, and the
// increment after its first colour-0 pass from zero, as the ping-pong has it
// then: colour 0 in e0 (the second array's half), colour 1 of e zero; r^2
__device__ __forceinline__ double dgpm_outer_cell(const double* __restrict__ u, const double* __restrict__ rho,
                                                  float* __restrict__ g32, float* __restrict__ pb,
                                                  float* __restrict__ e, float* __restrict__ e0, const Geo& g,
                                                  const DgpCoef& c, int m, unsigned row2)
{
    const unsigned nn = (unsigned)g.n * (unsigned)g.n;
    const int col = row2 >= nn ? 1 : 0;
    const unsigned r2 = row2 - (unsigned)col * nn;
    const int j = (int)(r2 % (unsigned)g.n), k = (int)(r2 / (unsigned)g.n);
    const int i = 2 * m + ((col + j + k) & 1);
    const size_t me = (size_t)col * g.half + row_base(g, j, k) + m;
    double c0;
    const double OP = dgp_L(u, g, i, j, k, rho[me], c, c0);
    const float gv = (float)(-OP);
    g32[me] = gv;
    pb[me] = (float)c0;
    if (col == 0)
        e0[me] = dgpm_first(gv, (float)c.inv_dx2);
    else
        e[me] = 0.0f;
    return OP * OP;
}

// coarsest level: sweeps of the inner smoother by one workgroup, the update
// evaluated in FP64 (the level holds at most a few thousand cells)
__device__ __forceinline__ void dgpm_coarsest_block(float* __restrict__ e, const float* __restrict__ pb,
                                                    const double* __restrict__ rho, const float* __restrict__ rhs,
                                                    float* __restrict__ tmp, const Geo& g, int sweeps, const DgpF& c)
{
    for (int sw = 0; sw < sweeps; sw++) {
        for (int colour = 0; colour < 2; colour++) {
            for (int t = threadIdx.x; t < (int)g.half; t += blockDim.x) {
                const int m = t % g.h, row = t / g.h;
                const int j = row % g.n, k = row / g.n;
                const int i = 2 * m + ((colour + j + k) & 1);
                const size_t me = (size_t)colour * g.half + t;
                const D2f de = d2_at(e, g, i, j, k);
                const double D = (double)dgp_dop(d2_at(pb, g, i, j, k), de, (float)rho[me], c) - (double)rhs[me];
                tmp[t] = (float)((double)de.c0 + D / (6.0 * (double)c.inv_dx2));
            }
            __syncthreads();
            for (int t = threadIdx.x; t < (int)g.half; t += blockDim.x) e[(size_t)colour * g.half + t] = tmp[t];
            __syncthreads();
        }
    }
}

// ---------------------------------------------------------------------------
// z-marching with 19-point register windows (levels with n/2 >= 64, so that
// a wave is 64 consecutive m of one row)
// ---------------------------------------------------------------------------
// A thread owns column (m, j) and marches over a run of DGP_KC planes.  Its
// window (DWin2) holds, for planes k-1, k, k+1 and rows j-1, j, j+1, the
// pair at x = 2m, 2m+1; with x = 2m-1 and 2m+2 at the five slots the
// stencil reaches off the column (taken from the neighbouring lanes by a
// shift; past the wave's edge by a scalar load), that is every point of the
// 19-point stencil of the cell of either colour at (m, j, k).  A step loads
// the pair at m of plane k+2 in the three rows (both colour halves at one
// offset) and the next cell's own data before plane k is computed, the next
// side values as soon as the present ones are in the stencils.  The stencil
// values go through S19 like the per-cell kernels', so every result is
// bit-identical to theirs.
//
// Bound by the vector ALU and by memory about equally, so the march itself
// costs no vector instructions: planes move scalar base pointers, a row's
// 32-bit offset stays in its register, and the value past the edge is the
// shift's own operand for the lane that has no neighbour.  The barriers to the
// scheduler keep it from raising every address sum of the unrolled run, which
// spills scalar registers into vector lanes.  Instructions per cell: FP32 pass
// 239 -> 177, FP32 residual 238 -> 160, FP64 residual 162 -> 111.  At 512^3, by
// where the arrays lie in memory (each process keeps its times): FP32 pass
// 456-484 -> 399-445 us, in one process 524; FP32 residual 718-850 ->
// 669-705, FP64 outer residual 880-921 -> 730-745 (5.1 TB/s), FP64 pass 632 ->
// 460.  Side values of
// the FP32 pass by vector loads: 467 where scalar ones take 444; of the FP32
// residual by scalar loads: 610 in the one run, 910 in the other; of the FP64
// residual by vector loads: 1043.
//
// The field is read through its two colour halves (h0, h1) and the pass
// writes the new values of its colour to `out`, a half of a second array: a
// pair of passes (colour 0, then colour 1 reading the new colour 0) moves
// the field into the second array without the per-cell kernels' copy.
struct DCol {
    unsigned plane;
    unsigned off[3];    // (m, row j-1..j+1) in a plane of a colour half
    unsigned left[3];   // (first lane's m - 1, ...): wave-uniform
    unsigned right[3];  // (last lane's m + 1, ...)
};

__device__ __forceinline__ DCol dcol_of(const Geo& g, int m, int j)
{
    DCol d;
    d.plane = (unsigned)g.n * (unsigned)g.h;
    // a wave is 64 consecutive m of one row
    const int ma = __builtin_amdgcn_readfirstlane(m), mz = ma + 63, ju = __builtin_amdgcn_readfirstlane(j);
    const unsigned mm = (unsigned)(ma == 0 ? g.h - 1 : ma - 1), mp = (unsigned)(mz + 1 == g.h ? 0 : mz + 1);
    const int jr[3] = {wrap_dec(ju, g.n), ju, wrap_inc(ju, g.n)};
#pragma unroll
    for (int R = 0; R < 3; R++) {
        const unsigned row = (unsigned)jr[R] * (unsigned)g.h;
        d.off[R] = row + (unsigned)m;
        d.left[R] = row + mm;
        d.right[R] = row + mp;
    }
    return d;
}

// Single-colour passes hold only x = 2m and 2m+1 of the window (DWin2).
// The cell of parity s needs the third x at five (plane, row) slots, q =
// 0..4: (1,1), (1,0), (1,2), (0,1), (2,1): x = 2m-1 when s = 0 (the o value
// of lane m-1) and x = 2m+2 when s = 1 (the e value of lane m+1), taken by a
// shift at use.  A wave is 64 consecutive m of one row and plane, so s is the
// same for all its lanes, and so are the five values its edge lane on that
// side needs (DSide).
template <typename T>
struct DWin2 {
    T e[3][3], o[3][3];  // [plane k-1, k, k+1][row j-1, j, j+1]: x = 2m, 2m+1
};

template <typename T>
struct DRaw2 {
    T ev[3], ov[3];
};

template <typename T>
struct DSide {
    T v[5];
};

__device__ __forceinline__ int side_plane(int q) { return q == 3 ? 0 : (q == 4 ? 2 : 1); }
__device__ __forceinline__ int side_row(int q) { return q == 1 ? 0 : (q == 2 ? 2 : 1); }

// The two colour halves of a field seen from the columns of one wave: the
// value at x = 2m of row jr, plane K lies in p[0] when jr + K has the parity
// par0 of j + k0 (the wave's row and first plane), else in p[1]; the value at
// x = 2m+1 in the other.  A wave is 64 consecutive m of one row and plane
// run, so par0 and both pointers are wave-uniform (scalar registers), and
// with the plane offset dk = K - k0 known when the z-march is unrolled, the
// half of every load is chosen at compile time: (jr + K) & 1 =
// par0 ^ ((R + 1 + dk) & 1) for row jr = j + R - 1 (n even, so the wrap
// keeps the parity).
template <typename T>
struct DHalves {
    const T* p[2];
};

template <typename T>
__device__ __forceinline__ DHalves<T> dhalves(const T* h0, const T* h1, int par0)
{
    DHalves<T> H;
    H.p[0] = par0 ? h1 : h0;
    H.p[1] = par0 ? h0 : h1;
    return H;
}

// the pair at (m, rows j-1..j+1) of plane K (dk = K - k0 modulo 2)
template <typename T>
__device__ __forceinline__ void draw2_load(const DHalves<T>& H, const DCol& d, int K, int dk, DRaw2<T>& r)
{
    const size_t kp = (size_t)((unsigned)K * d.plane);
#pragma unroll
    for (int R = 0; R < 3; R++) {
        const int f = (R + 1 + dk) & 1;
        r.ev[R] = ld_at(plane_ptr(H.p[f], kp), d.off[R]);
        r.ov[R] = ld_at(plane_ptr(H.p[f ^ 1], kp), d.off[R]);
    }
}

// the five side values of the cell at plane k (dk = k - k0) with parity s:
// x = 2m+2 has the colour of x = 2m, x = 2m-1 that of 2m+1.  Scalar loads, or
// with VECTOR one address in every lane: for the residual of two fields, whose
// twenty values a plane crowd the scalar registers and the scalar cache.
template <bool VECTOR = false, typename T>
__device__ __forceinline__ void dside_load(const DHalves<T>& H, const DCol& d, int k, int dk, int n, bool s,
                                           DSide<T>& sd)
{
#pragma unroll
    for (int q = 0; q < 5; q++) {
        const int P = side_plane(q), R = side_row(q);
        const unsigned kp = (unsigned)(P == 0 ? wrap_dec(k, n) : (P == 2 ? wrap_inc(k, n) : k)) * d.plane;
        const int f = ((R + P + dk) & 1) ^ (s ? 0 : 1);
        unsigned o = s ? d.right[R] : d.left[R];
        if constexpr (VECTOR) {
            asm("" : "+v"(o));
            sd.v[q] = ld_at(plane_ptr(H.p[f], kp), o);
        } else {
            sd.v[q] = ld_scalar(H.p[f], (size_t)kp + o);
        }
    }
}

template <typename T>
__device__ __forceinline__ void dwin2_set(DWin2<T>& w, int P, const DRaw2<T>& r)
{
#pragma unroll
    for (int R = 0; R < 3; R++) {
        w.e[P][R] = r.ev[R];
        w.o[P][R] = r.ov[R];
    }
}

template <typename T>
__device__ __forceinline__ void dwin2_shift(DWin2<T>& w)
{
#pragma unroll
    for (int R = 0; R < 3; R++) {
        w.e[0][R] = w.e[1][R];
        w.o[0][R] = w.o[1][R];
        w.e[1][R] = w.e[2][R];
        w.o[1][R] = w.o[2][R];
    }
}

template <typename T>
__device__ __forceinline__ void dwin2_init(DWin2<T>& w, const DHalves<T>& H, const DCol& d, int k0, int n)
{
    DRaw2<T> r0, r1, r2;
    draw2_load(H, d, wrap_dec(k0, n), -1, r0);
    draw2_load(H, d, k0, 0, r1);
    draw2_load(H, d, wrap_inc(k0, n), 1, r2);
    dwin2_set(w, 0, r0);
    dwin2_set(w, 1, r1);
    dwin2_set(w, 2, r2);
}

// the value of lane + 1 (FROM_RIGHT) or lane - 1 of the wave, by a DPP
// whole-wave shift (wave_shl:1 / wave_shr:1); the last / first lane, which has
// no such neighbour, takes its own `edge`
template <bool FROM_RIGHT>
__device__ __forceinline__ int wave_shift1(int edge, int v)
{
    return __builtin_amdgcn_update_dpp(edge, v, FROM_RIGHT ? 0x130 : 0x138, 0xf, 0xf, false);
}

template <bool FROM_RIGHT>
__device__ __forceinline__ float wave_shift1(float edge, float v)
{
    return __int_as_float(wave_shift1<FROM_RIGHT>(__float_as_int(edge), __float_as_int(v)));
}

template <bool FROM_RIGHT>
__device__ __forceinline__ double wave_shift1(double edge, double v)
{
    const unsigned long long a = (unsigned long long)__double_as_longlong(edge);
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)wave_shift1<FROM_RIGHT>((int)(unsigned)a, (int)(unsigned)u);
    const unsigned hi = (unsigned)wave_shift1<FROM_RIGHT>((int)(unsigned)(a >> 32), (int)(unsigned)(u >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// the 19 stencil values of the cell of parity s (all lanes of the wave
// execute the shifts)
template <typename T>
__device__ __forceinline__ S19<T> s19_win2(const DWin2<T>& w, bool s, const DSide<T>& sd)
{
    T v[5];
#pragma unroll
    for (int q = 0; q < 5; q++) {
        const int P = side_plane(q), R = side_row(q);
        v[q] = s ? wave_shift1<true>(sd.v[q], w.e[P][R]) : wave_shift1<false>(sd.v[q], w.o[P][R]);
    }
    // x = i + dx at slot (P, R), i = 2m + s; q: the side slot of (P, R)
    auto X = [&](int P, int R, int dx, int q) -> T {
        if (dx == 0) return s ? w.o[P][R] : w.e[P][R];
        if (dx < 0) return s ? w.e[P][R] : v[q];
        return s ? v[q] : w.o[P][R];
    };
    S19<T> u;
    u.c0 = X(1, 1, 0, 0);
    u.xp = X(1, 1, 1, 0);
    u.xm = X(1, 1, -1, 0);
    u.yp = X(1, 2, 0, 0);
    u.ym = X(1, 0, 0, 0);
    u.zp = X(2, 1, 0, 0);
    u.zm = X(0, 1, 0, 0);
    u.xy_pp = X(1, 2, 1, 2);
    u.xy_mm = X(1, 0, -1, 1);
    u.xy_pm = X(1, 0, 1, 1);
    u.xy_mp = X(1, 2, -1, 2);
    u.xz_pp = X(2, 1, 1, 4);
    u.xz_mm = X(0, 1, -1, 3);
    u.xz_pm = X(0, 1, 1, 3);
    u.xz_mp = X(2, 1, -1, 4);
    u.yz_pp = X(2, 2, 0, 0);
    u.yz_mm = X(0, 0, 0, 0);
    u.yz_pm = X(0, 2, 0, 0);
    u.yz_mp = X(2, 0, 0, 0);
    return u;
}

// Both cells of the pair at (m, j) over the run [k0, k0 + DGP_KC), from one
// window per field (OP::NF fields of type OP::T, colour halves
// op.half(f, 0/1)).  Per plane the cell at x = 2m comes first, then x = 2m+1;
// OP::load(colour, b, i) loads a cell's own data from element b + i of its
// colour's half, OP::cell(colour, b, i, own, stencils) returns a value whose square is accumulated (the sum is returned).  The
// next plane's window values and own data are loaded before a plane is
// evaluated.
template <bool PAR0, class OP>
__device__ __forceinline__ double dgp_both_run(const OP& op, const Geo& g, DCol d, int k0)
{
    // (32-bit offsets made in this block: the compiler then knows them as such)
#pragma unroll
    for (int R = 0; R < 3; R++) asm("" : "+v"(d.off[R]));
    using T = typename OP::T;
    using Own = typename OP::Own;
    constexpr int NF = OP::NF;
    DHalves<T> H[NF];
    DWin2<T> w[NF];
    DSide<T> sl[NF], sr[NF];  // of the cells at x = 2m and 2m+1
#pragma unroll
    for (int f = 0; f < NF; f++) {
        H[f] = dhalves(op.half(f, 0), op.half(f, 1), PAR0);
        dwin2_init(w[f], H[f], d, k0, g.n);
        dside_load<(NF > 1)>(H[f], d, k0, 0, g.n, false, sl[f]);
        dside_load<(NF > 1)>(H[f], d, k0, 0, g.n, true, sr[f]);
    }
    const unsigned i = d.off[1];
    size_t b = (size_t)((unsigned)k0 * d.plane);
    Own o0 = op.load(PAR0, b, i), o1 = op.load(!PAR0, b, i);
    double acc = 0.0;
#pragma unroll
    for (int t = 0; t < DGP_KC; t++) {
        const int k = k0 + t, kn = wrap_inc(k, g.n);
        const bool par = PAR0 ^ ((t & 1) != 0);  // colour of x = 2m
        const bool more = t + 1 < DGP_KC;
        DRaw2<T> r[NF];
        Own n0 = o0, n1 = o1;
        if (more) {
#pragma unroll
            for (int f = 0; f < NF; f++) draw2_load(H[f], d, wrap_inc(k + 1, g.n), t + 2, r[f]);
            n0 = op.load(!par, b + d.plane, i);
            n1 = op.load(par, b + d.plane, i);
        }
        // one cell's stencils at a time (fewer live values); its side values
        // are reloaded for the next plane once they are in the stencils
        double r0, r1;
        {
            S19<T> s0[NF];
#pragma unroll
            for (int f = 0; f < NF; f++) {
                s0[f] = s19_win2(w[f], false, sl[f]);
                if (more) dside_load<(NF > 1)>(H[f], d, kn, t + 1, g.n, false, sl[f]);
            }
            r0 = op.cell(par, b, i, o0, s0);
        }
        __builtin_amdgcn_sched_barrier(0);
        {
            S19<T> s1[NF];
#pragma unroll
            for (int f = 0; f < NF; f++) {
                s1[f] = s19_win2(w[f], true, sr[f]);
                if (more) dside_load<(NF > 1)>(H[f], d, kn, t + 1, g.n, true, sr[f]);
            }
            r1 = op.cell(!par, b, i, o1, s1);
        }
        acc += r0 * r0 + r1 * r1;
        if (more) {
#pragma unroll
            for (int f = 0; f < NF; f++) {
                dwin2_shift(w[f]);
                dwin2_set(w[f], 2, r[f]);
            }
            b += d.plane;
            o0 = n0;
            o1 = n1;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    return acc;
}

template <class OP>
__device__ __forceinline__ double dgp_both_zcol(const OP& op, const Geo& g, int m, int j, int k0)
{
    const DCol d = dcol_of(g, m, j);
    const int k = __builtin_amdgcn_readfirstlane(k0);
    return (__builtin_amdgcn_readfirstlane(j) + k) & 1 ? dgp_both_run<true>(op, g, d, k)
                                                       : dgp_both_run<false>(op, g, d, k);
}

// FP64 residual L(phi) (- f on coarse levels), stored in res when non-null
template <bool COARSE, bool NT = false>
struct DgpRes64Op {
    using T = double;
    static constexpr int NF = 1;
    struct Own {
        double rho, f;
    };
    const double* u;
    const double* rho;
    const double* f;
    double* res;
    DgpCoef c;
    unsigned hf;
    __device__ const double* half(int, int colour) const { return u + (colour ? hf : 0u); }
    __device__ __forceinline__ Own load(bool colour, size_t b, unsigned i) const
    {
        if (colour) b += hf;
        return Own{ld_at<NT>(plane_ptr(rho, b), i), COARSE ? ld_at<NT>(plane_ptr(f, b), i) : 0.0};
    }
    __device__ __forceinline__ double cell(bool colour, size_t b, unsigned i, const Own& o, const S19<double>* s) const
    {
        if (colour) b += hf;
        double OP = dgp_L19(s[0], o.rho, c);
        if constexpr (COARSE) OP = OP - o.f;
        if (res) st_at<NT>(plane_ptr(res, b), i, OP);
        return OP;
    }
};

// the mixed solve's FP64 outer residual r = L(phi), with the inner problem's
// data g = -r, phi_b = phi (FP32) and e after its first pass (as dgpm_outer_cell)
template <bool NT = false>
struct DgpmOuterOp {
    using T = double;
    static constexpr int NF = 1;
    struct Own {
        double rho;
    };
    const double* u;
    const double* rho;
    float* g32;
    float* pb;
    float* e;
    float* e0;
    DgpCoef c;
    unsigned hf;
    __device__ const double* half(int, int colour) const { return u + (colour ? hf : 0u); }
    __device__ __forceinline__ Own load(bool colour, size_t b, unsigned i) const
    {
        if (colour) b += hf;
        return Own{ld_at<NT>(plane_ptr(rho, b), i)};
    }
    __device__ __forceinline__ double cell(bool colour, size_t b, unsigned i, const Own& o, const S19<double>* s) const
    {
        if (colour) b += hf;
        const double OP = dgp_L19(s[0], o.rho, c);
        const float gv = (float)(-OP);
        st_at<NT>(plane_ptr(g32, b), i, gv);
        st_at<NT>(plane_ptr(pb, b), i, (float)s[0].c0);
        if (colour)
            st_at<NT>(plane_ptr(e, b), i, 0.0f);
        else
            st_at<NT>(plane_ptr(e0, b), i, dgpm_first(gv, (float)c.inv_dx2));
        return OP;
    }
};

// the mixed inner residual out = D(e) - rhs (as dgpm_residual_cell, which
// rounds the FP64 density to FP32: rho holds those values, or the FP64 ones);
// no norm
template <bool NT = false, typename R = float>
struct DgpmResOp {
    using T = float;
    static constexpr int NF = 2;  // e, phi_b
    struct Own {
        float rho, rhs;
    };
    const float* e;
    const float* pb;
    const R* rho;
    const float* rhs;
    float* out;
    DgpF c;
    unsigned hf;
    __device__ const float* half(int f, int colour) const { return (f ? pb : e) + (colour ? hf : 0u); }
    __device__ __forceinline__ Own load(bool colour, size_t b, unsigned i) const
    {
        if (colour) b += hf;
        return Own{(float)ld_at<NT>(plane_ptr(rho, b), i), ld_at<NT>(plane_ptr(rhs, b), i)};
    }
    __device__ __forceinline__ double cell(bool colour, size_t b, unsigned i, const Own& o, const S19<float>* s) const
    {
        if (colour) b += hf;
        st_at<NT>(plane_ptr(out, b), i, dgp_dop(d2_of(s[1]), d2_of(s[0]), o.rho, c) - o.rhs);
        return 0.0;
    }
};

// one colour of the mixed inner smoother (as dgpm_smooth_cell), z-marching from
// plane k0.  S0: parity of the column's first cell (the same for a whole wave);
// with the run unrolled the parity of every step is a constant, so the
// stencil values are the window's registers themselves.  R: the density's
// type (rounded to FP32 as it is used).
template <bool S0, bool NT, typename R>
__device__ __forceinline__ void dgpm_zsmooth_run(const float* __restrict__ e0, const float* __restrict__ e1,
                                                 float* __restrict__ out, const float* __restrict__ pb,
                                                 const R* __restrict__ rho, const float* __restrict__ rhs,
                                                 const Geo& g, int colour, const DgpF& c, const DCol& d, int k0v)
{
    const int k0 = __builtin_amdgcn_readfirstlane(k0v);
    // (j + k0) & 1 = S0 ^ colour: wave-uniform
    const int par0 = (S0 ? 1 : 0) ^ (colour & 1);
    const DHalves<float> He = dhalves(e0, e1, par0), Hb = dhalves(pb, pb + g.half, par0);
    const R* rhoc = rho + (size_t)colour * g.half;
    const float* rhsc = rhs + (size_t)colour * g.half;
    DWin2<float> we, wb;
    dwin2_init(we, He, d, k0, g.n);
    dwin2_init(wb, Hb, d, k0, g.n);
    DSide<float> se, sb;
    dside_load(He, d, k0, 0, g.n, S0, se);
    dside_load(Hb, d, k0, 0, g.n, S0, sb);
    const unsigned i = d.off[1];
    size_t b = (size_t)((unsigned)k0 * d.plane);
    float rh = (float)ld_at<NT>(plane_ptr(rhoc, b), i);
    float fv = ld_at<NT>(plane_ptr(rhsc, b), i);
#pragma unroll
    for (int t = 0; t < DGP_KC; t++) {
        const int k = k0 + t;
        const bool s = S0 ^ ((t & 1) != 0);
        DRaw2<float> re, rb;
        float rhn = 0.0f, fvn = 0.0f;
        const size_t bn = b + d.plane;
        if (t + 1 < DGP_KC) {
            const int kn = wrap_inc(k + 1, g.n);
            draw2_load(He, d, kn, t + 2, re);
            draw2_load(Hb, d, kn, t + 2, rb);
            rhn = (float)ld_at<NT>(plane_ptr(rhoc, bn), i);
            fvn = ld_at<NT>(plane_ptr(rhsc, bn), i);
        }
        const D2f de = d2_of(s19_win2(we, s, se)), db = d2_of(s19_win2(wb, s, sb));
        if (t + 1 < DGP_KC) {
            dside_load(He, d, wrap_inc(k, g.n), t + 1, g.n, !s, se);
            dside_load(Hb, d, wrap_inc(k, g.n), t + 1, g.n, !s, sb);
        }
        const float D = dgp_dop(db, de, rh, c) - fv;
        st_at<NT>(plane_ptr(out, b), i, de.c0 + over_six(D, c));
        if (t + 1 < DGP_KC) {
            dwin2_shift(we);
            dwin2_shift(wb);
            dwin2_set(we, 2, re);
            dwin2_set(wb, 2, rb);
            b = bn;
            rh = rhn;
            fv = fvn;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// e_h += P(e_H - R e_h) (no guard for DGP), z-marching over coarse columns, as
// k_df_correct: planes of e = e_H - R e_h in registers (x-neighbours from the
// adjacent lanes), all 8 sons of a coarse cell, software-pipelined (plane K's
// sons computed, the loads of plane K+1 issued, then plane K's sons stored).
// A son's sum runs over its 8 contributors with x fastest, the coarse cell last.
template <int S3, bool NT>
__device__ __forceinline__ void dgpm_sons_load(const float* __restrict__ ef, const Geo& gf, int I, int J, int K,
                                               float* old)
{
#pragma unroll
    for (int t = 0; t < 4; t++) old[t] = ld_once<NT>(elem(ef, son_index(gf, I, J, K, t & 1, t >> 1, S3)));
}

template <int S3>
__device__ __forceinline__ void dgpm_sons_new(const float* ez, const float* ek, const float* old, float* nv)
{
    const float a = 1.0f / 64.0f, b = 3.0f * a, c9 = 9.0f * a, dd = 27.0f * a;
    const float wt[8] = {a, b, b, c9, b, c9, c9, dd};
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int s1 = t & 1, s2 = t >> 1;
        float P = 0.0f;
#pragma unroll
        for (int ind = 0; ind < 8; ind++) {
            const int x = (ind & 1) ? 1 : (s1 ? 2 : 0);
            const int y = (ind & 2) ? 1 : (s2 ? 2 : 0);
            P += wt[ind] * ((ind & 4) ? ek[x + 3 * y] : ez[x + 3 * y]);
        }
        nv[t] = old[t] + P;
    }
}

template <int S3, bool NT>
__device__ __forceinline__ void dgpm_sons_store(float* __restrict__ ef, const Geo& gf, int I, int J, int K,
                                                const float* nv)
{
#pragma unroll
    for (int t = 0; t < 4; t++) st_once<NT>(elem(ef, son_index(gf, I, J, K, t & 1, t >> 1, S3)), nv[t]);
}

template <bool SHFL, bool NT>
__device__ __forceinline__ void dgpm_correct_col(const float* __restrict__ eH, const float* __restrict__ rd,
                                                 float* __restrict__ ef, const Geo& gf, const Geo& gc, const ZCol& cc,
                                                 bool lok = false, bool rok = false)
{
    const int I = cc.m, J = cc.j;
    Block9 B;
    B.init(gc, I, J);
    ERaw wm, wk, wp;  // coarse planes K-1, K, K+1
    float o0[4], o1[4];
    e_load<SHFL>(eH, rd, B, wrap_dec(cc.k0, gc.n), lok, rok, wm);
    e_load<SHFL>(eH, rd, B, cc.k0, lok, rok, wk);
    e_load<SHFL>(eH, rd, B, wrap_inc(cc.k0, gc.n), lok, rok, wp);
    dgpm_sons_load<0, NT>(ef, gf, I, J, cc.k0, o0);
    dgpm_sons_load<1, NT>(ef, gf, I, J, cc.k0, o1);
    float em[9], ek[9], ep[9];
    e_form<SHFL>(wm, lok, rok, em);
    e_form<SHFL>(wk, lok, rok, ek);
    for (int K = cc.k0; K < cc.k1; K++) {
        e_form<SHFL>(wp, lok, rok, ep);
        float n0[4], n1[4];
        dgpm_sons_new<0>(em, ek, o0, n0);
        dgpm_sons_new<1>(ep, ek, o1, n1);
        if (K + 1 < cc.k1) {
            dgpm_sons_load<0, NT>(ef, gf, I, J, K + 1, o0);
            dgpm_sons_load<1, NT>(ef, gf, I, J, K + 1, o1);
            e_load<SHFL>(eH, rd, B, wrap_inc(K + 1, gc.n), lok, rok, wp);
        }
        dgpm_sons_store<0, NT>(ef, gf, I, J, K, n0);
        dgpm_sons_store<1, NT>(ef, gf, I, J, K, n1);
#pragma unroll
        for (int q = 0; q < 9; q++) {
            em[q] = ek[q];
            ek[q] = ep[q];
        }
    }
}

}  // namespace mgs
