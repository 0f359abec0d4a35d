// mgs_tail.hip -- the small levels of a V-cycle in one single-workgroup
// launch, for the plain FP64 cycles (f(R) and nDGP) and the mixed nDGP inner
// cycle (the mixed f(R) one is df_tail_vcycle in mgs_fr_dev.h).
//
// A level of 16^3 cells or fewer takes 13 launches (17 for nDGP, whose passes
// were copied back) of 4 to 6 us each per cycle, whatever its size: four such
// levels cost 240 us of a 256^3 f(R) cycle's 970.  Here the levels live in
// the LDS of one CU (all arrays of 16^3 .. 2^3 in FP64: 155 KB of its 160) and
// an operation is one pass of the workgroup between barriers.  Per cell the
// arithmetic is that of the level kernels on the same values, so every array
// is bit-identical to the launch-per-operation cycle's; the FP64 forms write
// all of a level's arrays back (they can be read through the C-ABI).
// From 16^3 down: f(R) FP64 61 us where the launches took 200 (256^3 solve 6.88
// -> 5.83 ms), nDGP FP64 62 us (a 128^3 V-cycle 500 -> 372 us).  The 16^3
// passes are bound by the one CU's FP64 issue rate, the rest by latency.
// Literal reference roots (pow, acos) do not fit the registers of a 1024-thread
// workgroup and keep the launches.

#include <math.h>

#include "mgs_internal.h"
#include "mgs_kernels.h"
#include "mgs_tail_dev.h"

namespace mgs {

template <class MD>
__global__ __launch_bounds__(TAIL_THREADS) void k_plain_tail(PTailDesc<MD> G)
{
    __shared__ typename MD::T lds[PTAIL_LDS<MD>];
    ptail_run<MD>(G, lds);
}

template <class MD, class SET>
static bool launch_ptail(mgs_handle* h, int l, SET set, hipStream_t s)
{
    const int nlev = h->lc - l + 1;
    if (!ptail_fits(h->L[l].n, nlev)) return false;
    PTailDesc<MD> G;
    G.nl = nlev - 1;
    for (int i = 0; i < nlev; i++) {
        G.L[i].g = make_geo(h->L[l + i].n);
        G.L[i].rho = h->L[l + i].rho;
        G.L[i].pb = nullptr;
        set(G.L[i], l + i);
    }
    hipLaunchKernelGGL((k_plain_tail<MD>), dim3(1), dim3(TAIL_THREADS), 0, s, G);
    return true;
}

template <class MD>
static void set_plain(PTailLevel<MD>& t, const LevelD& v, const typename MD::Coef& c)
{
    t.u = v.u;
    t.f = v.f;
    t.res = v.res;
    t.rres = v.rres;
    t.ru = v.ru;
    t.c = c;
}

bool launch_plain_tail(mgs_handle* h, int l)
{
    if (h->p.model == MGS_MODEL_DGP)
        return launch_ptail<TailDgp64>(
            h, l, [h](PTailLevel<TailDgp64>& t, int q) { set_plain(t, h->L[q], dgp_coefs(h->p, q)); }, h->s);
    if (h->p.flags & MGS_FLAG_REFERENCE_ROOTS) return false;
#define FR64(FRN)                                                                                                \
    return launch_ptail<TailFr64<FRN>>(                                                                          \
        h, l, [h](PTailLevel<TailFr64<FRN>>& t, int q) { set_plain(t, h->L[q], fr_coefs(h->p, q)); }, h->s)
    if (h->p.fr_n == 0) FR64(0);
    if (h->p.fr_n == 1) FR64(1);
    FR64(2);
#undef FR64
}

bool launch_dgpm_tail(mgs_handle* h, int l)
{
    return launch_ptail<TailDgpm>(
        h, l,
        [h](PTailLevel<TailDgpm>& t, int q) {
            LevelF& v = h->M[q];
            t.u = v.d;
            t.f = v.f;
            t.res = v.res;
            t.rres = v.rres;
            t.ru = v.rd;
            t.pb = v.xb;
            t.c = dgpf(dgp_coefs(h->p, q));
        },
        h->s);
}

}  // namespace mgs
