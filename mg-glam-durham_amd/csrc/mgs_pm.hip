// mgs_pm.hip -- the particle side of a PM step around the scalar-field solve:
// CIC density deposit (DENSIT) and the particle push with the CIC-gathered
// potential gradient (MOVE), on particles resident in HBM.
//
// Particles are the reference's REAL*4 arrays XPAR..VZ (PMP2mod_tools.f90:46)
// in its convention: positions in grid units in [1, N+1), cell I = INT(X).
// They live on the device in six float arrays owned by the handle.
//
// Deposit into the solver's level-0 density (colour-split FP64, the array
// mgs_set_density fills), so a solve can follow without a host trip.  The
// particles are binned by the 32 x 16 x 8-cell tile of their CIC base cell and
// by the tile faces their +1 nodes cross, in runs of consecutive particles of
// one bin (a counting sort: counts gathered per block in LDS, an exclusive
// scan, a scatter of the particles' indices into bin order); one
// workgroup per tile then accumulates every weight that falls into its cells
// in a fixed-point buffer in LDS and writes each cell's density once.  Integer
// accumulation makes the sum independent of the order of the additions (the
// reference adds into REAL*4 FI).
//
// Move: one thread per particle gathers the 32 potential values of its 2x2x2
// node block and their outer neighbours (PMP2main.f90:496-558), forms the
// doubled central-difference gradients at the 8 nodes, interpolates them
// with the CIC weights, kicks, drifts, wraps, and adds v^2 WPAR to a block
// partial of SVEL.  The potential (mgs_potential, + mgs_potential_add_fifth_force)
// is REAL*4 in x-fastest order, as the reference's FI; the gradients and
// weights are formed in FP64 from it, as there.

#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <cmath>
#include <string>

#include "../../include/mgsolve.h"
#include "mgs_device.h"
#include "mgs_internal.h"
#include "mgs_kernels.h"

namespace mgs {

struct PmState {
    int64_t np = 0;
    int64_t ld = 0;        // floats from one array to the next: np rounded up to 64, so each starts 256-byte aligned
    float* buf = nullptr;  // x, y, z, vx, vy, vz: 6 * ld floats
    float* phi = nullptr;  // N^3 potential, x fastest, REAL*4 like the reference's FI
    double* part = nullptr;
    int* bad = nullptr;    // particles outside [1, N+1) seen by the last kernel
    int npart_blocks = 0;
    // deposit binning (runs of particles, see k_bin_count): the run records
    // and their number per wave, the particles in bin order; per bin its count
    // and first particle
    int64_t nbin = 0;
    unsigned long long* recs = nullptr;
    int* nrec = nullptr;
    unsigned* order = nullptr;  // nbin particle indices
    int nbins = 0;
    int* count = nullptr;
    unsigned* first = nullptr;
    void* scan_tmp = nullptr;
    size_t scan_bytes = 0;
};

static PmState* pm_of(mgs_handle* h) { return (PmState*)h->pm; }

constexpr int PM_BLOCK = 256;
constexpr int PM_GRID_MAX = 8192;  // persistent blocks of the particle kernels

static int pm_grid(int64_t np)
{
    const int64_t b = (np + PM_BLOCK - 1) / PM_BLOCK;
    return (int)(b < PM_GRID_MAX ? (b < 1 ? 1 : b) : PM_GRID_MAX);
}

void pm_release(mgs_handle* h)
{
    PmState* p = pm_of(h);
    if (!p) return;
    if (p->buf) (void)hipFree(p->buf);
    if (p->phi) (void)hipFree(p->phi);
    if (p->part) (void)hipFree(p->part);
    if (p->bad) (void)hipFree(p->bad);
    for (void* q : {(void*)p->recs, (void*)p->nrec, (void*)p->order, (void*)p->count, (void*)p->first, p->scan_tmp})
        if (q) (void)hipFree(q);
    delete p;
    h->pm = nullptr;
}

float* pm_potential(mgs_handle* h)
{
    PmState* p = pm_of(h);
    if (!p) {
        p = new PmState();
        h->pm = p;
    }
    if (!p->phi) {
        const size_t n3 = (size_t)h->p.ngrid * h->p.ngrid * h->p.ngrid;
        if (hipMalloc((void**)&p->phi, n3 * sizeof(float)) != hipSuccess) {
            p->phi = nullptr;
            return nullptr;
        }
    }
    return p->phi;
}

// INT(X) of the reference for X in [1, N+1): the 1-based cell; -1 outside (or
// NaN).  N + 1 <= 1025 is exact in REAL*4.
__device__ __forceinline__ int cell_of(float X, int N)
{
    if (!(X >= 1.0f && X < (float)(N + 1))) return -1;
    return (int)X;
}

// DENSIT's CIC loop, PMP2mod_density.f90:235-281 (0-based cells here), over
// the particles binned by tile.  A tile is 32 x 16 x 8 cells: long in x, so
// that consecutive particles of a lattice-ordered array stay in one tile and
// a tile's rows are whole 128-byte lines of each colour half.
constexpr int PM_TX = 32, PM_TY = 16, PM_TZ = 8;
constexpr int PM_LX = PM_TX + 1;                  // LDS row stride: rows start in different banks
constexpr int PM_TCELLS = PM_LX * PM_TY * PM_TZ;  // 4224 (33 KiB of LDS)

// tiles per side
struct PmTiles {
    int x, y, z;
};

static PmTiles pm_tiles(int N)
{
    return PmTiles{(N + PM_TX - 1) / PM_TX, (N + PM_TY - 1) / PM_TY, (N + PM_TZ - 1) / PM_TZ};
}

// Bin of a particle with 0-based base cell (i0, j0, k0): 8 bins per tile, by
// whether the particle's +1 nodes lie beyond the tile in x (1), y (2), z (4).
__device__ __forceinline__ int bin_of(int i0, int j0, int k0, int N, const PmTiles& T)
{
    const int t = ((k0 / PM_TZ) * T.y + j0 / PM_TY) * T.x + i0 / PM_TX;
    const int fx = (i0 % PM_TX == PM_TX - 1 || i0 == N - 1) ? 1 : 0;
    const int fy = (j0 % PM_TY == PM_TY - 1 || j0 == N - 1) ? 2 : 0;
    const int fz = (k0 % PM_TZ == PM_TZ - 1 || k0 == N - 1) ? 4 : 0;
    return t * 8 + (fx | fy | fz);
}

// The binning passes take PM_RUN consecutive particles per thread (particles
// in array order are usually neighbours in space, so consecutive ones usually
// share a bin) and bin *runs*: maximal sequences of a thread's particles in
// one bin, described by (first particle, length).
constexpr int PM_RUN = 8;
constexpr int PM_WCHUNK = 64 * PM_RUN;  // particles of one wave, whose run records are stored together
constexpr int KEY_OUTSIDE = -1;         // particle outside [1, N+1)

// A run's record between the two binning passes: its rank (the particles of
// the bin before it), the bin (21 bits: 2^21 bins at N = 1024), the first
// particle's place in the wave's 512 and the length - 1.
__device__ __forceinline__ unsigned long long run_record(unsigned rank, int bin, int local, int len)
{
    return (unsigned long long)rank << 33 | (unsigned long long)(unsigned)bin << 12 | (unsigned)local << 3 |
           (unsigned)(len - 1);
}

// per run: its record; per bin: the count of particles.  A block first counts
// its particles per bin in an LDS hash table (a lattice-ordered block of 2048
// meets some tens of bins), then adds each bin's count to the global counter
// once; the global counter's old value plus the run's rank in the block is
// its rank.  Before, one returning global atomic per run bound this pass:
// 2.13 ms for 512^3 particles in lattice order, now 0.49 ms (1.6 GB of
// positions read, 0.4 GB of records written).  A run whose bin finds no slot
// within PM_PROBES (blocks of unordered particles) takes the global atomic
// itself: 2.6 ms for 400^3 shuffled particles, as with one atomic per run (4.0
// without the table, whose bins' atomics are issued together).
constexpr int PM_SLOTS = 1024, PM_PROBES = 8;

__global__ __launch_bounds__(PM_BLOCK) void k_bin_count(const float* __restrict__ xs, const float* __restrict__ ys,
                                                        const float* __restrict__ zs, int64_t np, int N, PmTiles T,
                                                        unsigned long long* __restrict__ recs, int* __restrict__ nrec,
                                                        int* __restrict__ count, int* __restrict__ bad)
{
    __shared__ int keys[PM_SLOTS];
    __shared__ int cnt[PM_SLOTS];
    for (int i = threadIdx.x; i < PM_SLOTS; i += PM_BLOCK) {
        keys[i] = -1;
        cnt[i] = 0;
    }
    const int lane = threadIdx.x & 63;
    const int64_t wave = (int64_t)blockIdx.x * (PM_BLOCK / 64) + (threadIdx.x >> 6);
    const int64_t p0 = wave * PM_WCHUNK + lane * PM_RUN;
    float x[PM_RUN], y[PM_RUN], z[PM_RUN];
    if (p0 + PM_RUN <= np) {  // the arrays start 256-byte aligned: 16-byte loads
#pragma unroll
        for (int v = 0; v < PM_RUN / 4; v++) {
            const float4 a = ((const float4*)(xs + p0))[v], b = ((const float4*)(ys + p0))[v],
                         c = ((const float4*)(zs + p0))[v];
            x[4 * v] = a.x, x[4 * v + 1] = a.y, x[4 * v + 2] = a.z, x[4 * v + 3] = a.w;
            y[4 * v] = b.x, y[4 * v + 1] = b.y, y[4 * v + 2] = b.z, y[4 * v + 3] = b.w;
            z[4 * v] = c.x, z[4 * v + 1] = c.y, z[4 * v + 2] = c.z, z[4 * v + 3] = c.w;
        }
    } else {
#pragma unroll
        for (int r = 0; r < PM_RUN; r++) {
            const int64_t p = p0 + r < np ? p0 + r : np - 1;
            x[r] = xs[p];
            y[r] = ys[p];
            z[r] = zs[p];
        }
    }
    int t[PM_RUN];
    int nbad = 0;
#pragma unroll
    for (int r = 0; r < PM_RUN; r++) {
        t[r] = KEY_OUTSIDE;
        if (p0 + r < np) {
            const int I = cell_of(x[r], N), J = cell_of(y[r], N), K = cell_of(z[r], N);
            if (I < 0 || J < 0 || K < 0)
                nbad++;
            else
                t[r] = bin_of(I - 1, J - 1, K - 1, N, T);
        }
    }
    if (nbad) atomicAdd(bad, nbad);
    __syncthreads();  // the table is clear
    // the run starting at particle r: its length, its slot (-1: none) and its
    // rank in the block's count of the slot, or its global rank without a slot
    int slot[PM_RUN], rk[PM_RUN], len[PM_RUN], ns = 0;
#pragma unroll
    for (int r = 0; r < PM_RUN; r++) {
        slot[r] = -1;
        rk[r] = 0;
        len[r] = 0;
        const bool start = t[r] >= 0 && (r == 0 || t[r] != t[r - 1]);
        if (!start) continue;
        ns++;
        len[r] = 1;
        bool same = true;
#pragma unroll
        for (int q = r + 1; q < PM_RUN; q++) {
            same = same && t[q] == t[r];
            len[r] += same ? 1 : 0;
        }
        unsigned s = ((unsigned)t[r] * 2654435761u) >> 22;
        for (int q = 0; q < PM_PROBES; q++) {
            int k = *(volatile int*)&keys[s];
            if (k == -1) k = atomicCAS(&keys[s], -1, t[r]);
            if (k == -1 || k == t[r]) {
                slot[r] = (int)s;
                break;
            }
            s = (s + 1) & (PM_SLOTS - 1);
        }
        rk[r] = slot[r] >= 0 ? atomicAdd(&cnt[slot[r]], len[r]) : atomicAdd(&count[t[r]], len[r]);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < PM_SLOTS; i += PM_BLOCK)
        if (keys[i] >= 0) cnt[i] = atomicAdd(&count[keys[i]], cnt[i]);
    // the wave's records, one after the other
    int pre = ns;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int v = __shfl_up(pre, off, 64);
        if (lane >= off) pre += v;
    }
    if (lane == 63 && wave * PM_WCHUNK < np) nrec[wave] = pre;
    __syncthreads();
    unsigned long long* out = recs + wave * PM_WCHUNK + (pre - ns);
#pragma unroll
    for (int r = 0; r < PM_RUN; r++) {
        if (!len[r]) continue;
        const unsigned rank = (unsigned)(slot[r] >= 0 ? cnt[slot[r]] + rk[r] : rk[r]);
        *out++ = run_record(rank, t[r], lane * PM_RUN + r, len[r]);
    }
}

// 2 and 4 words stored (loaded) at 4-byte alignment by one instruction
struct __attribute__((packed, aligned(4))) Words2 {
    unsigned v[2];
};
struct __attribute__((packed, aligned(4))) Words4 {
    unsigned v[4];
};

// the particles' indices in bin order (the deposit takes fewer than 2^31
// particles); one wave per PM_WCHUNK particles, its records and their bins'
// starts loaded before the first store.  Bound by the scattered stores: a run's
// words go out in stores of 4, 2 and 1.  A bin's line is filled a word at a time
// by whichever waves meet the bin, so the more waves are under way the more
// partly filled lines there are, and the L2 writes them out and takes them in
// again: PM_SCATTER_LDS of unused LDS holds a CU to three blocks.  Measured with
// eight blocks (and records loaded one by one) -> three, in ms: shuffled
// lattices of 480^3 particles 3.39 -> 1.76, 400^3 1.93 -> 1.06 (four 1.61, two
// 0.82); in order, clustered, 512^3 0.52 -> 0.46 (0.45, 0.52), 250^3 0.046 ->
// 0.045 (0.042, 0.052).
constexpr int PM_SCATTER_LDS = 53000;

__global__ __launch_bounds__(PM_BLOCK) void k_bin_scatter(int64_t nwaves, const unsigned long long* __restrict__ recs,
                                                          const int* __restrict__ nrec,
                                                          const unsigned* __restrict__ first,
                                                          unsigned* __restrict__ order)
{
    const int64_t wave = (int64_t)blockIdx.x * (PM_BLOCK / 64) + (threadIdx.x >> 6);
    if (wave >= nwaves) return;
    const int n = nrec[wave];
    const int lane = threadIdx.x & 63;
    unsigned long long rec[PM_RUN];
    unsigned at[PM_RUN];
#pragma unroll
    for (int q = 0; q < PM_RUN; q++)
        if (lane + 64 * q < n) rec[q] = recs[wave * PM_WCHUNK + lane + 64 * q];
#pragma unroll
    for (int q = 0; q < PM_RUN; q++)
        if (lane + 64 * q < n) at[q] = first[(unsigned)(rec[q] >> 12) & 0x1fffffu] + (unsigned)(rec[q] >> 33);
#pragma unroll
    for (int q = 0; q < PM_RUN; q++) {
        if (lane + 64 * q >= n) continue;
        const unsigned long long r = rec[q];
        unsigned* o = order + at[q];
        const unsigned p = (unsigned)(wave * PM_WCHUNK) + ((unsigned)(r >> 3) & 511u);
        const unsigned len = ((unsigned)r & 7u) + 1u;
        unsigned u = 0;
        for (; u + 4 <= len; u += 4) *(Words4*)(o + u) = Words4{{p + u, p + u + 1, p + u + 2, p + u + 3}};
        if (len & 2) {
            *(Words2*)(o + u) = Words2{{p + u, p + u + 1}};
            u += 2;
        }
        if (len & 1) o[u] = p + u;
    }
}

// The deposit sums in fixed point so that its result does not depend on the
// order in which particles meet a cell: every CIC contribution (DENSIT's
// arithmetic in FP64, a value in [0, WPAR]) is rounded once to an integer
// multiple of 2^-40 and the multiples are added as 64-bit integers, which is
// exact and associative; a cell then holds -1 + (its integer) * 2^-40.  The
// result is bitwise the same run to run, within 2^-41 per contribution of
// the FP64 sum; a cell's integer holds 1 + delta up to 2^24 and converts
// exactly up to 2^13.
constexpr double PM_FIX = 1099511627776.0;          // 2^40
constexpr double PM_UNFIX = 1.0 / 1099511627776.0;  // 2^-40

// SMALL: v < 2^11.  v + 1.5 * 2^12 then lies in [2^12, 2^13), where a double's
// last place is 2^-40: the addition itself rounds v to nearest (ties to even,
// as the conversion does), and the sum's bits less those of 1.5 * 2^12 (whose
// low word is zero) are the integer.  Two instructions instead of the dozen of
// the 64-bit conversion.
template <bool SMALL>
__device__ __forceinline__ unsigned long long pm_fix(double v)
{
    if constexpr (SMALL)
        return (unsigned long long)__double_as_longlong(v + 6144.0) - 0x40B8000000000000ull;
    else
        return __double2ull_rn(v * PM_FIX);
}
constexpr double PM_FIX_SMALL = 2048.0;

// the eight weights of a particle with fractions D1, D2, D3 (DENSIT's products
// in its order) added at LDS cell b and its +1 neighbours, where KEEP says that
// the node is the tile's
template <bool SMALL, typename KEEP>
__device__ __forceinline__ void pm_add8(unsigned long long* acc, int b, double D1, double D2, double D3, double wpar,
                                        KEEP keep)
{
    const double T1 = 1.0 - D1, T2 = 1.0 - D2, T3 = 1.0 - D3;
    const double T2W = T2 * wpar, D2W = D2 * wpar;
    const double TT = T3 * T1, TD = T3 * D1, DT = D3 * T1, DD = D3 * D1;
    constexpr int SY = PM_LX, SZ = PM_TY * PM_LX;
    if (keep(0, 0, 0)) atomicAdd(&acc[b], pm_fix<SMALL>(TT * T2W));
    if (keep(1, 0, 0)) atomicAdd(&acc[b + 1], pm_fix<SMALL>(TD * T2W));
    if (keep(0, 1, 0)) atomicAdd(&acc[b + SY], pm_fix<SMALL>(TT * D2W));
    if (keep(1, 1, 0)) atomicAdd(&acc[b + SY + 1], pm_fix<SMALL>(TD * D2W));
    if (keep(0, 0, 1)) atomicAdd(&acc[b + SZ], pm_fix<SMALL>(DT * T2W));
    if (keep(1, 0, 1)) atomicAdd(&acc[b + SZ + 1], pm_fix<SMALL>(DD * T2W));
    if (keep(0, 1, 1)) atomicAdd(&acc[b + SZ + SY], pm_fix<SMALL>(DT * D2W));
    if (keep(1, 1, 1)) atomicAdd(&acc[b + SZ + SY + 1], pm_fix<SMALL>(DD * D2W));
}

// One workgroup per tile: the CIC weights that fall into the tile's cells
// accumulated in LDS, then written once as delta.  The particles are those of
// the tile's own 8 bins and, for each of the 7 tiles one step back in x, y
// and/or z, those of its bins whose +1 nodes reach this tile; of a particle
// only the nodes inside the tile are added.  Every cell is written by exactly
// one block, so the density needs no clearing, no atomics and no conversion
// pass, at the price of the reach's particles being read twice (1.25 times
// the particles).  One thread per particle: a thread per (run, position) left
// two lanes in three idle, as runs of a clustered lattice are short.
//
// 512^3 cells, 512^3 particles (lattice displaced by 2 cells rms): this kernel
// 1.35 ms (2.75 with a thread per run and position), the whole deposit with
// its reading back 6.5 -> 2.7 ms.  Before, 16^3-cell tiles added into the
// grid in eight launches by parity class (2.65 ms) between a clearing and a
// conversion pass (0.55 ms).  What is left is the gather of
// positions in bin order and the LDS additions; for shuffled particles the
// gather alone (400^3: 4.4 ms, as before).
constexpr int PM_SEGS = 21;  // own inner bin; own bins 1..7; 4 + 4 + 2 + 4 + 2 + 2 + 1 bins of the others
constexpr int PM_DBLOCK = 512;

template <bool SMALL>
__global__ __launch_bounds__(PM_DBLOCK) void k_tile_deposit(const float* __restrict__ xs,
                                                            const float* __restrict__ ys,
                                                            const float* __restrict__ zs,
                                                            const unsigned* __restrict__ order,
                                                            const int* __restrict__ count,
                                                            const unsigned* __restrict__ first, unsigned ntiles,
                                                            PmTiles T, double* __restrict__ rho, Geo g, double wpar)
{
    __shared__ unsigned long long acc[PM_TCELLS];
    __shared__ int64_t seg_off[PM_SEGS];  // item q of segment s is order[seg_off[s] + q]
    __shared__ int64_t seg_end[PM_SEGS];  // running count of particles
    __shared__ int seg_dir[PM_SEGS];
    unsigned t;
    if (!map_block(ntiles, t)) return;
    const int N = g.n;
    const int tx = (int)(t % (unsigned)T.x), ty = (int)((t / (unsigned)T.x) % (unsigned)T.y),
              tz = (int)(t / (unsigned)(T.x * T.y));
    if (threadIdx.x < 64) {
        // segment s > 1: the tile one step back in the directions of d, one of
        // its bins with all of d set
        const int s = (int)threadIdx.x;
        int64_t items = 0, start = 0;
        if (s < PM_SEGS) {
            const int dir[PM_SEGS] = {0, 0, 1, 1, 1, 1, 2, 2, 2, 2, 3, 3, 4, 4, 4, 4, 5, 5, 6, 6, 7};
            const int flag[PM_SEGS] = {0, 1, 1, 3, 5, 7, 2, 3, 6, 7, 3, 7, 4, 5, 6, 7, 5, 7, 6, 7, 7};
            const int d = dir[s];
            const int bx = (d & 1) ? wrap_dec(tx, T.x) : tx, by = (d & 2) ? wrap_dec(ty, T.y) : ty,
                      bz = (d & 4) ? wrap_dec(tz, T.z) : tz;
            const int b = ((bz * T.y + by) * T.x + bx) * 8 + flag[s];
            start = first[b];
            items = s == 1 ? (int64_t)first[b + 6] + count[b + 6] - start : (int64_t)count[b];
            seg_dir[s] = d;
        }
        int64_t end = items;
#pragma unroll
        for (int off = 1; off < 32; off <<= 1) {
            const int64_t v = __shfl_up(end, off, 64);
            if (s >= off) end += v;
        }
        if (s < PM_SEGS) {
            seg_end[s] = end;
            seg_off[s] = start - (end - items);
        }
    }
    for (int i = threadIdx.x; i < PM_TCELLS; i += PM_DBLOCK) acc[i] = 0ull;
    __syncthreads();
    const int i00 = tx * PM_TX, j00 = ty * PM_TY, k00 = tz * PM_TZ;
    const int ex = N - i00 < PM_TX ? N - i00 : PM_TX, ey = N - j00 < PM_TY ? N - j00 : PM_TY,
              ez = N - k00 < PM_TZ ? N - k00 : PM_TZ;
    // INT(X) >= 1 (checked when binned) and the fraction X - INT(X), both exact
    // in REAL*4; the next particle is loaded before this one is added
    const int64_t total = seg_end[PM_SEGS - 1];
    int s = 0, sn = 0;
    float x = 0.0f, y = 0.0f, z = 0.0f;
    auto fetch = [&](int64_t q, int& seg, float& fx, float& fy, float& fz) {
        if (q >= total) return;
        while (q >= seg_end[seg]) seg++;
        const unsigned p = order[seg_off[seg] + q];
        fx = xs[p];
        fy = ys[p];
        fz = zs[p];
    };
    fetch(threadIdx.x, s, x, y, z);
    for (int64_t q = threadIdx.x; q < total; q += PM_DBLOCK) {
        float xn = 0.0f, yn = 0.0f, zn = 0.0f;
        sn = s;
        fetch(q + PM_DBLOCK, sn, xn, yn, zn);
        const float fi = truncf(x), fj = truncf(y), fk = truncf(z);
        const double D1 = (double)(x - fi), D2 = (double)(y - fj), D3 = (double)(z - fk);
        const int I = (int)fi - 1 - i00, J = (int)fj - 1 - j00, K = (int)fk - 1 - k00;
        if (__all(s == 0)) {  // all eight nodes are the tile's
            pm_add8<SMALL>(acc, (K * PM_TY + J) * PM_LX + I, D1, D2, D3, wpar, [](int, int, int) { return true; });
        } else {
            // base cell in the tile's frame: -1 in a direction the particle comes from
            const int d = seg_dir[s];
            const int bi = (d & 1) ? -1 : I, bj = (d & 2) ? -1 : J, bk = (d & 4) ? -1 : K;
            pm_add8<SMALL>(acc, (bk * PM_TY + bj) * PM_LX + bi, D1, D2, D3, wpar, [&](int a, int b, int c) {
                return (a ? bi + 1 < ex : bi >= 0) && (b ? bj + 1 < ey : bj >= 0) && (c ? bk + 1 < ez : bk >= 0);
            });
        }
        s = sn;
        x = xn;
        y = yn;
        z = zn;
    }
    __syncthreads();
    // delta = -1 + sum * 2^-40, 16 values of one colour at a time (the tile's
    // first cell has even coordinates, so local parity is global parity)
    for (int i = threadIdx.x; i < PM_TX * PM_TY * PM_TZ; i += PM_DBLOCK) {
        const int m = i & 15, c = (i >> 4) & 1, j = (i >> 5) & (PM_TY - 1), k = i >> 9;
        if (2 * m >= ex || j >= ey || k >= ez) continue;
        const int xc = 2 * m + ((c + j + k) & 1);
        const unsigned long long v = acc[(k * PM_TY + j) * PM_LX + xc];
        rho[(size_t)c * g.half + row_base(g, j00 + j, k00 + k) + (unsigned)(i00 / 2 + m)] = -1.0 + (double)v * PM_UNFIX;
    }
}

// M adjacent floats from element i of a (4-byte aligned)
template <int M>
__device__ __forceinline__ void row_load(const float* a, unsigned i, float (&v)[M])
{
    const char* p = reinterpret_cast<const char*>(a) + i * (unsigned)sizeof(float);
    if constexpr (M == 4) {
        const Words4 w = *reinterpret_cast<const Words4*>(p);
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = __uint_as_float(w.v[e]);
    } else {
        const Words2 w = *reinterpret_cast<const Words2*>(p);
#pragma unroll
        for (int e = 0; e < 2; e++) v[e] = __uint_as_float(w.v[e]);
    }
}

// Bound by the texture addressers (93 % busy): the lanes of a wave meet
// different rows, so each load costs an address cycle per line it touches.  A
// row's values in one 16- or 8-byte load make 12 loads of the 32; 15.6 M
// particles on 250^3 cells: 633 -> 435 us.  Prefetching the next particle, or
// five waves per SIMD (28 bytes of spills: 527 us), did not help.
//
// MOVE's particle loop for the f(R) and nDGP models (no friction or mass
// terms, PMP2main.f90:488-684): kick with the CIC-interpolated gradient of
// the potential, drift, periodic wrap, SVEL partial per block
__global__ __launch_bounds__(PM_BLOCK) void k_move(float* __restrict__ xs, float* __restrict__ ys,
                                                   float* __restrict__ zs, float* __restrict__ vxs,
                                                   float* __restrict__ vys, float* __restrict__ vzs, int64_t np,
                                                   const float* __restrict__ phi, int N, double pconst,
                                                   double xconst, double wpar, double* __restrict__ part,
                                                   int* __restrict__ bad)
{
    // XN = FLOAT(NGRID)+1.-1.E-8 and YN = FLOAT(NGRID), evaluated as the
    // reference does (default REAL: the 1e-8 is below float resolution)
    const double XN = (double)((float)N + 1.0f - 1.0e-8f);
    const double YN = (double)N;
    const unsigned n = (unsigned)N;
    double svel = 0.0;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < np; p += stride) {
        const float xf0 = xs[p], yf0 = ys[p], zf0 = zs[p];
        double X = xf0, Y = yf0, Z = zf0;
        double VVX = vxs[p], VVY = vys[p], VVZ = vzs[p];
        const int I = cell_of(xf0, N), J = cell_of(yf0, N), K = cell_of(zf0, N);
        if (I < 0 || J < 0 || K < 0) {
            atomicAdd(bad, 1);
            continue;
        }
        const double D1 = X - (double)I, D2 = Y - (double)J, D3 = Z - (double)K;
        const double T1 = 1.0 - D1, T2 = 1.0 - D2, T3 = 1.0 - D3;
        const double T2T1 = T2 * T1, T2D1 = T2 * D1, D2T1 = D2 * T1, D2D1 = D2 * D1;
        // 0-based indices of I-1 .. I+2 (x), J-1 .. J+2 (y), K-1 .. K+2 (z)
        const int x1 = I - 1, x2 = I == N ? 0 : I, x3 = I + 1 >= N ? I + 1 - N : I + 1, x0 = I == 1 ? N - 1 : I - 2;
        const int y1 = J - 1, y2 = J == N ? 0 : J, y3 = J + 1 >= N ? J + 1 - N : J + 1, y0 = J == 1 ? N - 1 : J - 2;
        const int z1 = K - 1, z2 = K == N ? 0 : K, z3 = K + 1 >= N ? K + 1 - N : K + 1, z0 = K == 1 ? N - 1 : K - 2;
        // rows of the 4 x 4 x 4 block: x0 .. x3 in the four centre rows, x1 and x2
        // in the eight rows beside them.  Away from the wrap in x a row's values
        // are adjacent: one 16-byte and one 8-byte load (4-byte aligned) per row
        // instead of 32 loads
        float c11[4], c21[4], c12[4], c22[4];        // (y, z)
        float a01[2], a31[2], a02[2], a32[2];        // y0, y3 at z1, z2
        float b10[2], b13[2], b20[2], b23[2];        // z0, z3 at y1, y2
        // rows as 32-bit element offsets from the uniform base (N^3 <= 2^30)
        const unsigned r11 = n * ((unsigned)y1 + n * (unsigned)z1), r21 = n * ((unsigned)y2 + n * (unsigned)z1);
        const unsigned r12 = n * ((unsigned)y1 + n * (unsigned)z2), r22 = n * ((unsigned)y2 + n * (unsigned)z2);
        const unsigned q01 = n * ((unsigned)y0 + n * (unsigned)z1), q31 = n * ((unsigned)y3 + n * (unsigned)z1);
        const unsigned q02 = n * ((unsigned)y0 + n * (unsigned)z2), q32 = n * ((unsigned)y3 + n * (unsigned)z2);
        const unsigned p10 = n * ((unsigned)y1 + n * (unsigned)z0), p13 = n * ((unsigned)y1 + n * (unsigned)z3);
        const unsigned p20 = n * ((unsigned)y2 + n * (unsigned)z0), p23 = n * ((unsigned)y2 + n * (unsigned)z3);
        if (I > 1 && I < N - 1) {
            const unsigned e0 = (unsigned)x0, e1 = (unsigned)x1;
            row_load(phi, r11 + e0, c11), row_load(phi, r21 + e0, c21), row_load(phi, r12 + e0, c12);
            row_load(phi, r22 + e0, c22), row_load(phi, q01 + e1, a01), row_load(phi, q31 + e1, a31);
            row_load(phi, q02 + e1, a02), row_load(phi, q32 + e1, a32), row_load(phi, p10 + e1, b10);
            row_load(phi, p13 + e1, b13), row_load(phi, p20 + e1, b20), row_load(phi, p23 + e1, b23);
        } else {
            const unsigned xi[4] = {(unsigned)x0, (unsigned)x1, (unsigned)x2, (unsigned)x3};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                c11[e] = elem(phi, r11 + xi[e]), c21[e] = elem(phi, r21 + xi[e]);
                c12[e] = elem(phi, r12 + xi[e]), c22[e] = elem(phi, r22 + xi[e]);
            }
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const unsigned x = xi[e + 1];
                a01[e] = elem(phi, q01 + x), a31[e] = elem(phi, q31 + x), a02[e] = elem(phi, q02 + x);
                a32[e] = elem(phi, q32 + x), b10[e] = elem(phi, p10 + x), b13[e] = elem(phi, p13 + x);
                b20[e] = elem(phi, p20 + x), b23[e] = elem(phi, p23 + x);
            }
        }
        const float F011 = c11[0], F111 = c11[1], F211 = c11[2], F311 = c11[3];
        const float F021 = c21[0], F121 = c21[1], F221 = c21[2], F321 = c21[3];
        const float F012 = c12[0], F112 = c12[1], F212 = c12[2], F312 = c12[3];
        const float F022 = c22[0], F122 = c22[1], F222 = c22[2], F322 = c22[3];
        const float F101 = a01[0], F201 = a01[1], F131 = a31[0], F231 = a31[1];
        const float F102 = a02[0], F202 = a02[1], F132 = a32[0], F232 = a32[1];
        const float F110 = b10[0], F210 = b10[1], F113 = b13[0], F213 = b13[1];
        const float F120 = b20[0], F220 = b20[1], F123 = b23[0], F223 = b23[1];
        // doubled gradients at the 8 nodes (the 1/2 is in pconst); the
        // reference's F's are default REAL, so each difference is a REAL*4
        // subtraction (PMP2main.f90:580-602), widened afterwards
#define G2(a, b) (double)((a) - (b))
        const double GX111 = G2(F211, F011), GX211 = G2(F311, F111), GX121 = G2(F221, F021), GX221 = G2(F321, F121);
        const double GX112 = G2(F212, F012), GX212 = G2(F312, F112), GX122 = G2(F222, F022), GX222 = G2(F322, F122);
        const double GY111 = G2(F121, F101), GY211 = G2(F221, F201), GY121 = G2(F131, F111), GY221 = G2(F231, F211);
        const double GY112 = G2(F122, F102), GY212 = G2(F222, F202), GY122 = G2(F132, F112), GY222 = G2(F232, F212);
        const double GZ111 = G2(F112, F110), GZ211 = G2(F212, F210), GZ121 = G2(F122, F120), GZ221 = G2(F222, F220);
        const double GZ112 = G2(F113, F111), GZ212 = G2(F213, F211), GZ122 = G2(F123, F121), GZ222 = G2(F223, F221);
#undef G2
        const double GX = pconst * (T3 * (T2T1 * GX111 + T2D1 * GX211 + D2T1 * GX121 + D2D1 * GX221) +
                                    D3 * (T2T1 * GX112 + T2D1 * GX212 + D2T1 * GX122 + D2D1 * GX222));
        const double GY = pconst * (T3 * (T2T1 * GY111 + T2D1 * GY211 + D2T1 * GY121 + D2D1 * GY221) +
                                    D3 * (T2T1 * GY112 + T2D1 * GY212 + D2T1 * GY122 + D2D1 * GY222));
        const double GZ = pconst * (T3 * (T2T1 * GZ111 + T2D1 * GZ211 + D2T1 * GZ121 + D2D1 * GZ221) +
                                    D3 * (T2T1 * GZ112 + T2D1 * GZ212 + D2T1 * GZ122 + D2D1 * GZ222));
        VVX = VVX + GX;
        VVY = VVY + GY;
        VVZ = VVZ + GZ;
        X = X + VVX * xconst;
        Y = Y + VVY * xconst;
        Z = Z + VVZ * xconst;
        if (X < 1.0) X = X + YN;
        if (X >= XN) X = X - YN;
        if (Y < 1.0) Y = Y + YN;
        if (Y >= XN) Y = Y - YN;
        if (Z < 1.0) Z = Z + YN;
        if (Z >= XN) Z = Z - YN;
        svel = svel + (VVX * VVX + VVY * VVY + VVZ * VVZ) * wpar;
        float xf = (float)X, yf = (float)Y, zf = (float)Z;
        // a coordinate that rounds to N+1 in REAL*4 is pulled back inside
        if ((int)xf == N + 1) xf = xf - 1.0e-3f;
        if ((int)yf == N + 1) yf = yf - 1.0e-3f;
        if ((int)zf == N + 1) zf = zf - 1.0e-3f;
        xs[p] = xf;
        ys[p] = yf;
        zs[p] = zf;
        vxs[p] = (float)VVX;
        vys[p] = (float)VVY;
        vzs[p] = (float)VVZ;
    }
    const double t = block_sum(svel);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// WPAR = YN**3/FLOAT(Nparticles) (PMP2mod_density.f90:40, PMP2main.f90:470):
// the particle count is converted to default REAL first, as there
// WPAR = YN**3/FLOAT(Nparticles) (PMP2mod_density.f90:40, PMP2main.f90:470):
// the count through default REAL, the quotient in REAL*8, stored in WPAR, an
// implicitly typed default REAL
static double wpar_of(int N, int64_t np)
{
    const double yn = (double)N;
    return (double)(float)(yn * yn * yn / (double)(float)np);
}

static int pm_ensure_particles(mgs_handle* h, int64_t np)
{
    PmState* p = pm_of(h);
    if (!p) {
        p = new PmState();
        h->pm = p;
    }
    if (!p->bad && hipMalloc((void**)&p->bad, sizeof(int)) != hipSuccess) {
        p->bad = nullptr;
        return set_err(h, MGS_E_NOMEM, "particle counters");
    }
    if (!p->part) {
        if (hipMalloc((void**)&p->part, (PM_GRID_MAX + 1024) * sizeof(double)) != hipSuccess) {
            p->part = nullptr;
            return set_err(h, MGS_E_NOMEM, "particle partials");
        }
    }
    if (p->np == np && p->buf) return 0;
    if (p->buf) (void)hipFree(p->buf);
    p->buf = nullptr;
    p->np = 0;
    const int64_t ld = (np + 63) / 64 * 64;
    if (hipMalloc((void**)&p->buf, (size_t)ld * 6 * sizeof(float)) != hipSuccess) {
        p->buf = nullptr;
        return set_err(h, MGS_E_NOMEM, "particle arrays (" + std::to_string(np) + " particles)");
    }
    p->np = np;
    p->ld = ld;
    return 0;
}

// out-of-range particles counted by the last kernel (synchronises)
static int pm_check_bad(mgs_handle* h, const char* what)
{
    int bad = 0;
    if (hipMemcpyAsync(&bad, pm_of(h)->bad, sizeof(int), hipMemcpyDeviceToHost, h->s) != hipSuccess ||
        hipStreamSynchronize(h->s) != hipSuccess)
        return set_err(h, MGS_E_HIP, std::string(what) + ": HIP error");
    if (bad)
        return set_err(h, MGS_E_DOMAIN, std::string(what) + ": " + std::to_string(bad) +
                                            " particle(s) outside [1, N+1) or not finite were skipped");
    return 0;
}

}  // namespace mgs

using namespace mgs;

extern "C" {

int mgs_particles_set(mgs_handle* h, const float* x, const float* y, const float* z, const float* vx, const float* vy,
                      const float* vz, int64_t npart, int32_t where)
{
    if (!h) return MGS_E_ARG;
    if (!x || !y || !z) return set_err(h, MGS_E_ARG, "positions are NULL");
    if (npart < 1) return set_err(h, MGS_E_ARG, "npart < 1");
    if (where != MGS_HOST && where != MGS_DEVICE) return set_err(h, MGS_E_ARG, "where");
    int rc = pm_ensure_particles(h, npart);
    if (rc) return rc;
    PmState* p = pm_of(h);
    const size_t bytes = (size_t)npart * sizeof(float);
    const hipMemcpyKind kind = where == MGS_HOST ? hipMemcpyHostToDevice : hipMemcpyDeviceToDevice;
    const float* src[6] = {x, y, z, vx, vy, vz};
    for (int a = 0; a < 6; a++) {
        float* dst = p->buf + (size_t)a * p->ld;
        const hipError_t e = src[a] ? hipMemcpyAsync(dst, src[a], bytes, kind, h->s) : hipMemsetAsync(dst, 0, bytes, h->s);
        if (e != hipSuccess) return set_err(h, MGS_E_HIP, "particle upload");
    }
    if (hipStreamSynchronize(h->s) != hipSuccess) return set_err(h, MGS_E_HIP, "particle upload");
    return 0;
}

int mgs_particles_get(mgs_handle* h, float* x, float* y, float* z, float* vx, float* vy, float* vz, int32_t where)
{
    if (!h) return MGS_E_ARG;
    PmState* p = pm_of(h);
    if (!p || !p->buf) return set_err(h, MGS_E_STATE, "no particles set");
    if (where != MGS_HOST && where != MGS_DEVICE) return set_err(h, MGS_E_ARG, "where");
    const size_t bytes = (size_t)p->np * sizeof(float);
    const hipMemcpyKind kind = where == MGS_HOST ? hipMemcpyDeviceToHost : hipMemcpyDeviceToDevice;
    float* dst[6] = {x, y, z, vx, vy, vz};
    for (int a = 0; a < 6; a++)
        if (dst[a] && hipMemcpyAsync(dst[a], p->buf + (size_t)a * p->ld, bytes, kind, h->s) != hipSuccess)
            return set_err(h, MGS_E_HIP, "particle download");
    if (hipStreamSynchronize(h->s) != hipSuccess) return set_err(h, MGS_E_HIP, "particle download");
    return 0;
}

// the deposit's binning buffers for the current particle count and nbins
static int pm_ensure_bins(mgs_handle* h, PmState* p, int nbins)
{
    if (p->nbin != p->np) {
        for (void* q : {(void*)p->recs, (void*)p->nrec, (void*)p->order})
            if (q) (void)hipFree(q);
        p->recs = nullptr;
        p->nrec = nullptr;
        p->order = nullptr;
        p->nbin = 0;
        const size_t waves = ((size_t)p->np + PM_WCHUNK - 1) / PM_WCHUNK;
        if (hipMalloc((void**)&p->recs, waves * PM_WCHUNK * sizeof(unsigned long long)) != hipSuccess ||
            hipMalloc((void**)&p->nrec, waves * sizeof(int)) != hipSuccess ||
            hipMalloc((void**)&p->order, (size_t)p->np * sizeof(unsigned)) != hipSuccess)
            return set_err(h, MGS_E_NOMEM, "deposit binning arrays");
        p->nbin = p->np;
    }
    if (p->nbins != nbins) {
        for (void* q : {(void*)p->count, (void*)p->first, p->scan_tmp})
            if (q) (void)hipFree(q);
        p->count = nullptr;
        p->first = nullptr;
        p->scan_tmp = nullptr;
        p->nbins = 0;
        size_t bytes = 0;
        if (hipMalloc((void**)&p->count, (size_t)nbins * sizeof(int)) != hipSuccess ||
            hipMalloc((void**)&p->first, (size_t)nbins * sizeof(unsigned)) != hipSuccess ||
            hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, p->count, p->first, nbins, h->s) != hipSuccess ||
            hipMalloc(&p->scan_tmp, bytes + 256) != hipSuccess)
            return set_err(h, MGS_E_NOMEM, "deposit tile arrays");
        p->scan_bytes = bytes + 256;
        p->nbins = nbins;
    }
    return 0;
}

int mgs_cic_deposit(mgs_handle* h)
{
    if (!h) return MGS_E_ARG;
    PmState* p = pm_of(h);
    if (!p || !p->buf) return set_err(h, MGS_E_STATE, "no particles set");
    if (p->np >= ((int64_t)1 << 31)) return set_err(h, MGS_E_ARG, "the deposit takes fewer than 2^31 particles");
    const int N = h->p.ngrid;
    const Geo g = make_geo(N);
    const PmTiles T = pm_tiles(N);
    const int ntiles = T.x * T.y * T.z;
    int rc = pm_ensure_bins(h, p, 8 * ntiles);
    if (rc) return rc;
    const int64_t np = p->np, ld = p->ld;
    const float* b = p->buf;
    prof_begin(h, MGS_KC_PM, (double)np * 56.0 + 32.0 * (double)N * N * N);
    if (hipMemsetAsync(p->bad, 0, sizeof(int), h->s) != hipSuccess ||
        hipMemsetAsync(p->count, 0, (size_t)p->nbins * sizeof(int), h->s) != hipSuccess)
        return set_err(h, MGS_E_HIP, "deposit");
    const int64_t nwaves = (np + PM_WCHUNK - 1) / PM_WCHUNK;
    const unsigned gbin = (unsigned)((nwaves + PM_BLOCK / 64 - 1) / (PM_BLOCK / 64));
    hipLaunchKernelGGL(k_bin_count, dim3(gbin), dim3(PM_BLOCK), 0, h->s, b, b + ld, b + 2 * ld, np, N, T, p->recs,
                       p->nrec, p->count, p->bad);
    if (hipcub::DeviceScan::ExclusiveSum(p->scan_tmp, p->scan_bytes, p->count, p->first, p->nbins, h->s) !=
        hipSuccess)
        return set_err(h, MGS_E_HIP, "deposit scan");
    hipLaunchKernelGGL(k_bin_scatter, dim3(gbin), dim3(PM_BLOCK), PM_SCATTER_LDS, h->s, nwaves, p->recs, p->nrec, p->first,
                       p->order);
    const double wpar = wpar_of(N, np);
    const unsigned gt = ((unsigned)ntiles + 7) / 8 * 8;  // map_block
    if (wpar < PM_FIX_SMALL)
        hipLaunchKernelGGL(k_tile_deposit<true>, dim3(gt), dim3(PM_DBLOCK), 0, h->s, b, b + ld, b + 2 * ld, p->order,
                           p->count, p->first, (unsigned)ntiles, T, h->L[0].rho, g, wpar);
    else
        hipLaunchKernelGGL(k_tile_deposit<false>, dim3(gt), dim3(PM_DBLOCK), 0, h->s, b, b + ld, b + 2 * ld, p->order,
                           p->count, p->first, (unsigned)ntiles, T, h->L[0].rho, g, wpar);
    prof_end(h);
    rc = pm_check_bad(h, "CIC deposit");
    h->has_density = true;
    h->rho_cached = false;
    return rc;
}

int mgs_move(mgs_handle* h, double pconst, double xconst, double* svel)
{
    if (!h) return MGS_E_ARG;
    PmState* p = pm_of(h);
    if (!p || !p->buf) return set_err(h, MGS_E_STATE, "no particles set");
    if (!p->phi) return set_err(h, MGS_E_STATE, "no potential: call mgs_potential first");
    if (!std::isfinite(pconst) || !std::isfinite(xconst)) return set_err(h, MGS_E_ARG, "pconst/xconst not finite");
    const int N = h->p.ngrid;
    const int grid = pm_grid(p->np);
    prof_begin(h, MGS_KC_PM, (double)p->np * 48.0);
    if (hipMemsetAsync(p->bad, 0, sizeof(int), h->s) != hipSuccess) return set_err(h, MGS_E_HIP, "move");
    const int64_t np = p->np, ld = p->ld;
    float* b = p->buf;
    hipLaunchKernelGGL(k_move, dim3(grid), dim3(PM_BLOCK), 0, h->s, b, b + ld, b + 2 * ld, b + 3 * ld, b + 4 * ld,
                       b + 5 * ld, np, p->phi, N, pconst, xconst, wpar_of(N, np), p->part, p->bad);
    launch_sum_partials(p->part, grid, h->dsum, h->s);
    prof_end(h);
    double s = 0.0;
    if (hipMemcpyAsync(&s, h->dsum, sizeof(double), hipMemcpyDeviceToHost, h->s) != hipSuccess)
        return set_err(h, MGS_E_HIP, "move");
    int rc = pm_check_bad(h, "move");
    if (svel) *svel = s;
    return rc;
}

}  // extern "C"
