// mgs_fft.hip -- grid-level pieces around the solve:
//   * seeded lognormal density (the synthetic input of every benchmark
//     configuration; no reference counterpart): Philox-4x32-10 white noise,
//     hipFFT D2Z, k-space filter, Z2D, normalisation to sigma_g, exp map;
//   * the fifth-force potential psi and its central-difference gradient
//     (POTENT_FOR_MG, PMP2main.f90:884-950, and MOVE's stencil :565-594);
//   * the power spectrum with POWERfft5's options: NGP or linear (CIC)
//     k-space bins, monopole or quadrupole, and its log bins
//     (PMP2mod_power.f90:323-456);
//   * the PM step's potential: POTENTfft5's discrete-Green's-function
//     Poisson solve (PMP2main.f90:705-867) and POTENT_FOR_MG's addition of
//     the scalar field (:869-935), into the handle's REAL*4 potential.

#include <hipfft/hipfft.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "mgs_device.h"
#include "mgs_internal.h"
#include "mgs_kernels.h"
#include "mgs_poisson.h"
#include "mgs_stencil.h"

namespace mgs {

struct FftState {
    int N = 0;
    hipfftHandle fwd = 0, inv = 0;
    bool have_fwd = false, have_inv = false;
    double* real = nullptr;          // N^3 lexicographic
    hipfftDoubleComplex* cplx = nullptr;  // N*N*(N/2+1)
    double* bins = nullptr;          // 6 (N/2 + 1): power, count, sum|m| of the linear and the log bins
    double* binpart = nullptr;       // SPECTRUM_BLOCKS such histograms, one per block
    int* logbin = nullptr;           // log bin of every |m|^2 = 0 .. 3 (N/2)^2
    void* tables = nullptr;          // Poisson solve: (power-of-two grids) twiddles, then Green's function
};

// blocks of the binning kernel: each accumulates a private histogram in LDS
static const int BIN_BLOCKS = 512;

static FftState* fft_of(mgs_handle* h) { return (FftState*)h->fft; }

static FftState* fft_state(mgs_handle* h)
{
    if (!h->fft) h->fft = new FftState();
    FftState* f = fft_of(h);
    f->N = h->p.ngrid;  // a handle's grid does not change
    return f;
}

static int fft_alloc(mgs_handle* h, void** p, size_t bytes, const char* what)
{
    if (*p) return 0;
    if (hipMalloc(p, bytes) == hipSuccess) return 0;
    *p = nullptr;
    return set_err(h, MGS_E_NOMEM, what);
}

static int fft_ensure_cplx(mgs_handle* h)
{
    FftState* f = fft_state(h);
    const size_t nc = (size_t)f->N * f->N * (f->N / 2 + 1);
    return fft_alloc(h, (void**)&f->cplx, nc * sizeof(hipfftDoubleComplex), "FFT buffer");
}

__global__ __launch_bounds__(256) void k_green_table(double* __restrict__ green, int N)
{
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k < N) green[k] = green_g(k, N);
}

static int fft_ensure_bins(mgs_handle* h)
{
    FftState* f = fft_state(h);
    const size_t len = 3 * (size_t)(f->N + 2) * sizeof(double);
    const int rc = fft_alloc(h, (void**)&f->bins, len, "FFT bins");
    return rc ? rc : fft_alloc(h, (void**)&f->binpart, SPECTRUM_BLOCKS * len, "FFT bins");
}

// power-of-two grids: twiddles and Green's function; others: the latter alone
static int fft_ensure_tables(mgs_handle* h)
{
    FftState* f = fft_state(h);
    const int N = f->N;
    if (f->tables) return 0;
    const bool pow2 = poisson_grid(N);
    const int rc = fft_alloc(h, &f->tables, pow2 ? poisson_table_bytes(N) : (size_t)N * sizeof(double), "FFT tables");
    if (rc) return rc;
    if (pow2)
        launch_poisson_tables(f->tables, N, h->s);
    else
        hipLaunchKernelGGL(k_green_table, dim3((N + 255) / 256), dim3(256), 0, h->s, (double*)f->tables, N);
    return 0;
}

// the library's transforms and their buffers
static int fft_ensure(mgs_handle* h)
{
    FftState* f = fft_state(h);
    const int N = f->N;
    int rc;
    if ((rc = fft_ensure_cplx(h))) return rc;
    if ((rc = fft_alloc(h, (void**)&f->real, (size_t)N * N * N * sizeof(double), "FFT buffer"))) return rc;
    if (!f->have_fwd) {
        if (hipfftPlan3d(&f->fwd, N, N, N, HIPFFT_D2Z) != HIPFFT_SUCCESS) return set_err(h, MGS_E_HIP, "hipfftPlan3d D2Z");
        f->have_fwd = true;
        hipfftSetStream(f->fwd, h->s);
    }
    return 0;
}

// the inverse transform's plan (the power spectrum needs none)
static int fft_ensure_inverse(mgs_handle* h)
{
    FftState* f = fft_state(h);
    const int N = f->N;
    if (f->have_inv) return 0;
    if (hipfftPlan3d(&f->inv, N, N, N, HIPFFT_Z2D) != HIPFFT_SUCCESS) return set_err(h, MGS_E_HIP, "hipfftPlan3d Z2D");
    f->have_inv = true;
    hipfftSetStream(f->inv, h->s);
    return 0;
}

void fft_release(mgs_handle* h)
{
    FftState* f = fft_of(h);
    if (!f) return;
    if (f->have_fwd) hipfftDestroy(f->fwd);
    if (f->have_inv) hipfftDestroy(f->inv);
    if (f->real) (void)hipFree(f->real);
    if (f->cplx) (void)hipFree(f->cplx);
    if (f->bins) (void)hipFree(f->bins);
    if (f->binpart) (void)hipFree(f->binpart);
    if (f->logbin) (void)hipFree(f->logbin);
    if (f->tables) (void)hipFree(f->tables);
    delete f;
    h->fft = nullptr;
}

// ---------------------------------------------------------------------------
// Philox-4x32-10 (Salmon, Moraes, Dror, Shaw, "Parallel random numbers: as
// easy as 1, 2, 3", SC'11)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void philox4x32(uint32_t c[4], uint32_t k0, uint32_t k1)
{
    for (int r = 0; r < 10; r++) {
        const uint64_t p0 = (uint64_t)c[0] * 0xD2511F53ull;
        const uint64_t p1 = (uint64_t)c[2] * 0xCD9E8D57ull;
        const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
        const uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
        const uint32_t n0 = hi1 ^ c[1] ^ k0, n1 = lo1, n2 = hi0 ^ c[3] ^ k1, n3 = lo0;
        c[0] = n0;
        c[1] = n1;
        c[2] = n2;
        c[3] = n3;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

// one standard normal per cell: counter (index lo, index hi, 0, 0), key = seed;
// Box-Muller on two 53-bit uniforms, cosine branch
__global__ __launch_bounds__(256) void k_white_noise(double* __restrict__ w, size_t n3, uint32_t k0, uint32_t k1)
{
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n3; i += stride) {
        uint32_t c[4] = {(uint32_t)i, (uint32_t)(i >> 32), 0u, 0u};
        philox4x32(c, k0, k1);
        const double u1 = ((double)(c[0] >> 5) * 67108864.0 + (double)(c[1] >> 6) + 1.0) / 9007199254740992.0;
        const double u2 = ((double)(c[2] >> 5) * 67108864.0 + (double)(c[3] >> 6)) / 9007199254740992.0;
        w[i] = sqrt(-2.0 * log(u1)) * cos(2.0 * 3.14159265358979323846 * u2);
    }
}

// multiply the half spectrum by k^(slope/2) exp(-k^2 / (4 kc^2)), k = 0 -> 0
__global__ __launch_bounds__(256) void k_filter(hipfftDoubleComplex* __restrict__ c, int N, double kf, double kc,
                                                double slope)
{
    const int nh = N / 2 + 1;
    const size_t total = (size_t)N * N * nh;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < total; q += stride) {
        const int i = (int)(q % nh);
        const size_t r = q / nh;
        const int j = (int)(r % N), k = (int)(r / N);
        const double mx = i, my = fold(j, N), mz = fold(k, N);
        const double kk = kf * sqrt(mx * mx + my * my + mz * mz);
        double a = 0.0;
        if (kk > 0.0) a = pow(kk, 0.5 * slope) * exp(-kk * kk / (4.0 * kc * kc));
        c[q].x *= a;
        c[q].y *= a;
    }
}

// block sums of g and of (g - mu)^2
__global__ __launch_bounds__(256) void k_moment(const double* __restrict__ g, size_t n3, double mu, int power,
                                                double* __restrict__ partials)
{
    double acc = 0.0;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n3; i += stride) {
        const double v = g[i] - mu;
        acc += power == 1 ? v : v * v;
    }
    const double t = block_sum(acc);
    if (threadIdx.x == 0) partials[blockIdx.x] = t;
}

// delta = exp((g - mu) * scale - sigma^2/2) - 1, written into the split layout
__global__ __launch_bounds__(256) void k_lognormal(const double* __restrict__ g, double* __restrict__ rho, Geo geo,
                                                   double mu, double scale, double half_var)
{
    const size_t n3 = 2 * geo.half;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n3; q += stride) {
        const int i = (int)(q % geo.n);
        const size_t r = q / geo.n;
        const int j = (int)(r % geo.n), k = (int)(r / geo.n);
        rho[split_index(geo, i, j, k)] = exp((g[q] - mu) * scale - half_var) - 1.0;
    }
}

// psi and its central differences, one thread per pair of cells (2m, 2m+1) of
// a row, marching over a run of planes with psi of the planes k-1, k, k+1 in
// registers: every access is a unit-stride run (the pairs of the rows beside
// it lie at the same m), and the outputs are written once, past the caches.
// A stream of 8 bytes in and 16 out per cell; 256^3, all four outputs in
// REAL*4: 97 us = 4.1 TB/s (one thread per cell with 64-bit divisions 187; when
// the march took 115, pairs without it 139, with cached stores 156).
template <typename T>
__global__ __launch_bounds__(256) void k_fifth_force(const double* __restrict__ u, T* __restrict__ psi,
                                                     T* __restrict__ gx, T* __restrict__ gy, T* __restrict__ gz, Geo g,
                                                     PsiOf psi_of, int TX, int TY, int XB, int JB, int KC, unsigned NB)
{
    ZCol c;
    if (!zcol(g, TX, TY, XB, JB, KC, NB, c)) return;
    const int n = g.n, j = c.j, m = c.m;
    auto at = [&](size_t q) { return psi_of(u[q]); };
    typedef T V2 __attribute__((ext_vector_type(2), aligned(sizeof(T))));  // a caller's array: aligned as its elements
    double pe, po, me = 0.0, mo = 0.0;  // planes k and k-1
    size_t e, o;
    if (gz) {
        pair_split(g, m, j, wrap_dec(c.k0, n), e, o);
        me = at(e), mo = at(o);
    }
    pair_split(g, m, j, c.k0, e, o);
    pe = at(e), po = at(o);
    for (int k = c.k0; k < c.k1; k++) {
        const size_t q = ((size_t)k * n + j) * n + 2 * (unsigned)m;
        auto store = [&](T* out, double a, double b) {
            const V2 v = {(T)a, (T)b};
            __builtin_nontemporal_store(v, reinterpret_cast<V2*>(out + q));
        };
        size_t en, on;
        pair_split(g, m, j, wrap_inc(k, n), en, on);
        double ne = 0.0, no = 0.0;
        if (gz || k + 1 < c.k1) ne = at(en), no = at(on);
        if (psi) store(psi, pe, po);
        if (gx) {
            const int ml = wrap_dec(m, g.h), mr = wrap_inc(m, g.h);
            store(gx, 0.5 * (po - at(o - (unsigned)m + (unsigned)ml)), 0.5 * (at(e - (unsigned)m + (unsigned)mr) - pe));
        }
        if (gy) {
            size_t ep, op, em, om;
            pair_split(g, m, wrap_inc(j, n), k, ep, op);
            pair_split(g, m, wrap_dec(j, n), k, em, om);
            store(gy, 0.5 * (at(ep) - at(em)), 0.5 * (at(op) - at(om)));
        }
        if (gz) store(gz, 0.5 * (ne - me), 0.5 * (no - mo));
        me = pe, mo = po, pe = ne, po = no;
        e = en, o = on;
    }
}

// POWERfft5's binning (bin_mode) of the half spectrum of the library's
// transform (x fastest, N/2+1 of it), one private LDS histogram per block
// written to part[block]
template <int IPOL, int ICIC, bool LOGB>
__global__ __launch_bounds__(256) void k_bin_power(const hipfftDoubleComplex* __restrict__ c, int N, double norm,
                                                   const int* __restrict__ logbin, double* __restrict__ part, int nb)
{
    extern __shared__ double hist[];
    for (int t = threadIdx.x; t < 6 * nb; t += blockDim.x) hist[t] = 0.0;
    __syncthreads();
    const int nh = N / 2 + 1;
    const size_t total = (size_t)N * N * nh;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < total; q += stride) {
        const int i = (int)(q % nh);
        const size_t r = q / nh;
        const int j = (int)(r % N), k = (int)(r / N);
        bin_mode<IPOL, ICIC, LOGB>(hist, nb, N, i, fold(j, N), fold(k, N), (c[q].x * c[q].x + c[q].y * c[q].y) * norm,
                                   logbin);
    }
    __syncthreads();
    double* out = part + (size_t)blockIdx.x * 6 * nb;
    for (int t = threadIdx.x; t < 6 * nb; t += blockDim.x) out[t] = hist[t];
}

// bins[t] = sum over blocks of part[block][t] (some 500 of them): 16 bins of
// 16 threads each per workgroup, a thread adding every 16th block's value, then
// the 16 partial sums in order.  One thread per bin walked 512 dependent
// additions in four workgroups (256^3: 127 us).
__global__ __launch_bounds__(256) void k_bin_reduce(const double* __restrict__ part, int nblk, int len,
                                                    double* __restrict__ bins)
{
    __shared__ double s[16][17];
    const int c = threadIdx.x & 15, q = threadIdx.x >> 4, t = blockIdx.x * 16 + c;
    double v = 0.0;
    if (t < len)
        for (int b = q; b < nblk; b += 16) v += part[(size_t)b * len + t];
    s[q][c] = v;
    __syncthreads();
    if (q == 0 && t < len) {
        double r = s[0][c];
        for (int i = 1; i < 16; i++) r += s[i][c];
        bins[t] = r;
    }
}

// POTENTfft5's Green's function, PMP2main.f90:736-742, 805-816: the discrete
// Laplacian's eigenvalue A = (G(ky) - 6 + G(kx)) + G(kz), A = 1 for the mean
// mode (|A| < 1e-7).  G is the reference's GREENf table over FFTPACK5's
// half-complex wavenumbers i = 0 .. N/2: G(0) = 2, G(N/2) = -2 and
// G(i) = 2cos(P16 i/N) between, with the reference's P16 (PMP2main.f90:711, a
// REAL*8 parameter set from the default REAL literal 6.28318530718, so it
// holds that literal's REAL*4 rounding); a complex wavenumber k > N/2 is the
// half-complex i = N - k.  The half spectrum (x fastest, N/2+1 of it) is
// multiplied by trfi / A and by 1/N^3, hipFFT's transforms being
// unnormalised where FFTPACK5's forward one divides by N per dimension.
// One block row per (ky, kz): G from a table (three cosines and two 64-bit
// divisions per entry took 84 us at 250^3).
__global__ __launch_bounds__(256) void k_green(hipfftDoubleComplex* __restrict__ c, int N, double trfi, double inv_n3,
                                               const double* __restrict__ green)
{
    const unsigned nh = (unsigned)N / 2 + 1, rows = (unsigned)N * (unsigned)N;
    for (unsigned r = blockIdx.x; r < rows; r += gridDim.x) {
        const double gy = green[r % (unsigned)N] - 6.0, gz = green[r / (unsigned)N];
        for (unsigned kx = threadIdx.x; kx < nh; kx += 256) {
            double A = green[kx] + gy;
            A = A + gz;
            if (fabs(A) < 1.0e-7) A = 1.0;
            const size_t q = (size_t)r * nh + kx;
            hipfftDoubleComplex v = c[q];
            v.x = v.x * trfi / A * inv_n3;
            v.y = v.y * trfi / A * inv_n3;
            c[q] = v;
        }
    }
}

__global__ __launch_bounds__(256) void k_to_f32(const double* __restrict__ a, float* __restrict__ b, size_t n)
{
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += stride) b[q] = (float)a[q];
}

__global__ __launch_bounds__(256) void k_to_f64(const float* __restrict__ a, double* __restrict__ b, size_t n)
{
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += stride) b[q] = (double)a[q];
}

// POTENT_FOR_MG, PMP2main.f90:869-935: the REAL*4 potential (x fastest) plus
// the scalar field's contribution at each cell, summed in FP64 and rounded
// once, as FI = FI + sf does there
// (one thread per pair of cells; 512^3: 387 us = 5.5 TB/s, one per cell 505)
__global__ __launch_bounds__(256) void k_add_psi(float* __restrict__ phi, const double* __restrict__ u, Geo g,
                                                 PsiOf psi_of, int TX, int TY, int XB, unsigned NB)
{
    int m;
    unsigned row;
    if (!map_xy(g.h, (long)g.n * g.n, TX, TY, XB, NB, m, row)) return;
    const int j = (int)(row % (unsigned)g.n), k = (int)(row / (unsigned)g.n);
    size_t e, o;
    pair_split(g, m, j, k, e, o);
    Pair<float>* q = reinterpret_cast<Pair<float>*>(phi + ((size_t)row * g.n + 2 * (unsigned)m));
    Pair<float> v = *q;
    v.a = (float)((double)v.a + psi_of(u[e]));
    v.b = (float)((double)v.b + psi_of(u[o]));
    *q = v;
}

static dim3 grid_for(size_t count)
{
    size_t b = (count + 255) / 256;
    if (b > 16384) b = 16384;
    if (b < 1) b = 1;
    return dim3((unsigned)b);
}

// the fifth-force potential of the handle's model
static PsiOf psi_of_handle(const mgs_handle* h)
{
    double ubg = 1.0;
    const double fbg = fr_background(h->p, &ubg);
    const double ctilde = 2.99792458e3 * (double)h->p.ngrid / h->p.box;
    return PsiOf{h->p.model, h->p.fr_n, ctilde * ctilde * 0.5 * fbg, 1.0 / ubg};
}

static int sum_blocks(mgs_handle* h, double* partials, int nblk, double* out)
{
    if (sum_to_host(h, partials, nblk) || hipStreamSynchronize(h->s) != hipSuccess)
        return set_err(h, MGS_E_HIP, "reduction copy");
    *out = h->hsum[0];
    return 0;
}

}  // namespace mgs

using namespace mgs;

extern "C" {

int mgs_make_lognormal_density(mgs_handle* h, uint64_t seed, double sigma_g, double slope, double kcut_frac)
{
    if (!h || !(sigma_g > 0.0) || !(kcut_frac > 0.0)) return set_err(h, MGS_E_ARG, "lognormal parameters");
    int rc = fft_ensure(h);
    if (!rc) rc = fft_ensure_inverse(h);
    if (rc) return rc;
    FftState* f = fft_of(h);
    const int N = h->p.ngrid;
    const size_t n3 = (size_t)N * N * N;
    hipLaunchKernelGGL(k_white_noise, grid_for(n3), dim3(256), 0, h->s, f->real, n3, (uint32_t)(seed & 0xFFFFFFFFu),
                       (uint32_t)(seed >> 32));
    if (hipfftExecD2Z(f->fwd, f->real, f->cplx) != HIPFFT_SUCCESS) return set_err(h, MGS_E_HIP, "hipfftExecD2Z");
    const double kf = 2.0 * M_PI / h->p.box;
    const double kc = kcut_frac * M_PI * N / h->p.box;
    hipLaunchKernelGGL(k_filter, grid_for((size_t)N * N * (N / 2 + 1)), dim3(256), 0, h->s, f->cplx, N, kf, kc, slope);
    if (hipfftExecZ2D(f->inv, f->cplx, f->real) != HIPFFT_SUCCESS) return set_err(h, MGS_E_HIP, "hipfftExecZ2D");
    const dim3 gb = grid_for(n3);
    double s1 = 0.0, s2 = 0.0;
    hipLaunchKernelGGL(k_moment, gb, dim3(256), 0, h->s, f->real, n3, 0.0, 1, h->partials);
    if ((rc = sum_blocks(h, h->partials, (int)gb.x, &s1))) return rc;
    const double mu = s1 / (double)n3;
    hipLaunchKernelGGL(k_moment, gb, dim3(256), 0, h->s, f->real, n3, mu, 2, h->partials);
    if ((rc = sum_blocks(h, h->partials, (int)gb.x, &s2))) return rc;
    const double sd = std::sqrt(s2 / (double)n3);
    if (!(sd > 0.0)) return set_err(h, MGS_E_DOMAIN, "degenerate Gaussian field");
    hipLaunchKernelGGL(k_lognormal, gb, dim3(256), 0, h->s, f->real, h->L[0].rho, make_geo(N), mu, sigma_g / sd,
                       0.5 * sigma_g * sigma_g);
    if (hipStreamSynchronize(h->s) != hipSuccess) return set_err(h, MGS_E_HIP, "lognormal density");
    h->has_density = true;
    h->rho_cached = false;
    return 0;
}

int mgs_get_density(mgs_handle* h, void* dst, int32_t dtype, int32_t where)
{
    if (!h || !dst) return set_err(h, MGS_E_ARG, "NULL argument");
    const int N = h->p.ngrid;
    const size_t bytes = (size_t)N * N * N * (dtype == MGS_F32 ? 4 : 8);
    void* out = dst;
    if (where == MGS_HOST) {
        int rc = ensure_staging(h, bytes);
        if (rc) return rc;
        out = h->staging;
    }
    if (dtype == MGS_F32)
        launch_unpack_f64_to_f32(h->L[0].rho, (float*)out, N, 1.0, h->s);
    else
        launch_unpack_f64_to_f64(h->L[0].rho, (double*)out, N, 1.0, h->s);
    if (where == MGS_HOST && hipMemcpyAsync(dst, out, bytes, hipMemcpyDeviceToHost, h->s) != hipSuccess)
        return set_err(h, MGS_E_HIP, "density copy");
    if (hipStreamSynchronize(h->s) != hipSuccess) return set_err(h, MGS_E_HIP, "density copy");
    return 0;
}

int mgs_fifth_force(mgs_handle* h, void* psi, void* gx, void* gy, void* gz, int32_t dtype, int32_t where)
{
    if (!h) return set_err(h, MGS_E_ARG, "NULL handle");
    if (dtype != MGS_F32 && dtype != MGS_F64) return set_err(h, MGS_E_ARG, "dtype");
    const int N = h->p.ngrid;
    const size_t n3 = (size_t)N * N * N;
    const size_t es = dtype == MGS_F32 ? 4 : 8;
    void* outs[4] = {psi, gx, gy, gz};
    void* dev[4] = {nullptr, nullptr, nullptr, nullptr};
    std::vector<void*> tmp;
    for (int a = 0; a < 4; a++) {
        if (!outs[a]) continue;
        if (where == MGS_DEVICE) {
            dev[a] = outs[a];
        } else {
            void* q = nullptr;
            if (hipMalloc(&q, n3 * es) != hipSuccess) {
                for (void* t : tmp) (void)hipFree(t);
                return set_err(h, MGS_E_NOMEM, "fifth-force staging");
            }
            tmp.push_back(q);
            dev[a] = q;
        }
    }
    const PsiOf psi_of = psi_of_handle(h);
    prof_begin(h, MGS_KC_UPDATE, 0.0);
    const ZLaunch L = make_zlaunch(make_geo(N));
    if (dtype == MGS_F32)
        hipLaunchKernelGGL((k_fifth_force<float>), L.grid, L.block, 0, h->s, h->L[0].u, (float*)dev[0],
                           (float*)dev[1], (float*)dev[2], (float*)dev[3], make_geo(N), psi_of, L.TX, L.TY, L.XB, L.JB, L.KC,
                           L.NB);
    else
        hipLaunchKernelGGL((k_fifth_force<double>), L.grid, L.block, 0, h->s, h->L[0].u, (double*)dev[0],
                           (double*)dev[1], (double*)dev[2], (double*)dev[3], make_geo(N), psi_of, L.TX, L.TY, L.XB, L.JB,
                           L.KC, L.NB);
    prof_end(h);
    int rc = 0;
    if (where == MGS_HOST)
        for (int a = 0; a < 4; a++)
            if (outs[a] && hipMemcpyAsync(outs[a], dev[a], n3 * es, hipMemcpyDeviceToHost, h->s) != hipSuccess)
                rc = set_err(h, MGS_E_HIP, "fifth-force copy");
    if (hipStreamSynchronize(h->s) != hipSuccess) rc = set_err(h, MGS_E_HIP, "fifth force");
    for (void* t : tmp) (void)hipFree(t);
    return rc;
}

// the log bin (PMP2mod_power.f90:396, dLog = 0.02 a REAL*4 parameter, :12)
// of every |m|^2 = 0 .. n2max, in the reference's REAL*4 arithmetic with the C
// library's log10f; entry 0 is never used
static std::vector<int> log_bin_table(int n2max)
{
    std::vector<int> t((size_t)n2max + 1, 1);
    const float dlog = 0.02f;
    for (int n2 = 1; n2 <= n2max; n2++) {
        const float rk = std::sqrt((float)n2);
        const volatile float v = std::log10(rk) / dlog + 1000.0f;  // rounded to REAL*4 as stored
        const int b = (int)v - 1000;
        t[n2] = b < 1 ? 1 : b;
    }
    return t;
}

// which: 0 density delta, 1 field u, 2 fifth-force potential psi
int mgs_power_spectrum_ex(mgs_handle* h, int32_t which, int32_t ipol, int32_t icic, double* k, double* pk,
                          double* count, double* klog, double* pklog, double* countlog)
{
    if (!h || !k || !pk) return set_err(h, MGS_E_ARG, "NULL argument");
    if (which < 0 || which > 2) return set_err(h, MGS_E_ARG, "which must be 0 (delta), 1 (u) or 2 (psi)");
    if (ipol != 0 && ipol != 1) return set_err(h, MGS_E_ARG, "ipol must be 0 (monopole) or 1 (quadrupole)");
    if (icic != 0 && icic != 1) return set_err(h, MGS_E_ARG, "icic must be 0 (NGP bins) or 1 (linear bins)");
    const int N = h->p.ngrid;
    const bool pow2 = poisson_grid(N);  // transforms and binning of mgs_poisson.hip
    int rc = pow2 ? fft_ensure_cplx(h) : fft_ensure(h);
    if (!rc) rc = fft_ensure_bins(h);
    if (!rc && pow2) rc = fft_ensure_tables(h);
    if (rc) return rc;
    FftState* f = fft_of(h);
    const size_t n3 = (size_t)N * N * N;
    const Geo g = make_geo(N);
    const int n2max = 3 * (N / 2) * (N / 2);
    const bool logb = !icic && (klog || pklog || countlog);  // log bins asked for
    if (logb && !f->logbin) {
        const std::vector<int> t = log_bin_table(n2max);
        if (hipMalloc((void**)&f->logbin, t.size() * sizeof(int)) != hipSuccess)
            return set_err(h, MGS_E_NOMEM, "log bin table");
        if (hipMemcpyAsync(f->logbin, t.data(), t.size() * sizeof(int), hipMemcpyHostToDevice, h->s) != hipSuccess ||
            hipStreamSynchronize(h->s) != hipSuccess)
            return set_err(h, MGS_E_HIP, "log bin table copy");
    }
    const int nb = N / 2 + 1;  // bins 1..N/2 are returned
    const double norm = 1.0 / ((double)n3 * (double)n3);
    const PsiOf psi = psi_of_handle(h);
    int nblk = BIN_BLOCKS;
    if (pow2) {
        nblk = launch_spectrum(which == 0 ? h->L[0].rho : h->L[0].u, which == 2 ? &psi : nullptr, f->cplx, f->tables, N,
                               norm, ipol, icic, logb, f->logbin, f->binpart, h->s);
    } else {
        if (which == 0)
            launch_unpack_f64_to_f64(h->L[0].rho, f->real, N, 1.0, h->s);
        else if (which == 1)
            launch_unpack_f64_to_f64(h->L[0].u, f->real, N, 1.0, h->s);
        else {
            const ZLaunch L = make_zlaunch(g);
            hipLaunchKernelGGL((k_fifth_force<double>), L.grid, L.block, 0, h->s, h->L[0].u, f->real, (double*)nullptr,
                               (double*)nullptr, (double*)nullptr, g, psi, L.TX, L.TY, L.XB, L.JB, L.KC, L.NB);
        }
        if (hipfftExecD2Z(f->fwd, f->real, f->cplx) != HIPFFT_SUCCESS) return set_err(h, MGS_E_HIP, "hipfftExecD2Z");
        const size_t lds = 6 * (size_t)nb * sizeof(double);
        const dim3 G(BIN_BLOCKS), B(256);
        if (icic)
            hipLaunchKernelGGL((ipol ? k_bin_power<1, 1, false> : k_bin_power<0, 1, false>), G, B, lds, h->s, f->cplx, N,
                               norm, (const int*)f->logbin, f->binpart, nb);
        else if (logb)
            hipLaunchKernelGGL((ipol ? k_bin_power<1, 0, true> : k_bin_power<0, 0, true>), G, B, lds, h->s, f->cplx, N,
                               norm, (const int*)f->logbin, f->binpart, nb);
        else
            hipLaunchKernelGGL((ipol ? k_bin_power<1, 0, false> : k_bin_power<0, 0, false>), G, B, lds, h->s, f->cplx, N,
                               norm, (const int*)f->logbin, f->binpart, nb);
    }
    hipLaunchKernelGGL(k_bin_reduce, dim3((6 * nb + 15) / 16), dim3(256), 0, h->s, (const double*)f->binpart,
                       nblk, 6 * nb, f->bins);
    std::vector<double> hb(6 * (size_t)nb);
    if (hipMemcpyAsync(hb.data(), f->bins, hb.size() * sizeof(double), hipMemcpyDeviceToHost, h->s) != hipSuccess ||
        hipStreamSynchronize(h->s) != hipSuccess)
        return set_err(h, MGS_E_HIP, "bins copy");
    // PMP2mod_power.f90:420-456: the quadrupole times (2L+1)/2; a bin with no
    // (positive) count keeps zeros
    const double box = h->p.box, scale = 2.0 * M_PI / box, pfac = ipol ? 2.5 : 1.0;
    auto emit = [&](const double* hs, double* kk, double* pp, double* cc) {
        for (int b = 1; b <= N / 2; b++) {
            const double c = hs[nb + b];
            if (kk) kk[b - 1] = c > 0 ? hs[2 * nb + b] / c * scale : 0.0;
            if (pp) pp[b - 1] = c > 0 ? box * box * box * pfac * hs[b] / c : 0.0;
            if (cc) cc[b - 1] = c > 0 ? c : 0.0;
        }
    };
    emit(hb.data(), k, pk, count);
    if (icic) {
        for (int b = 0; b < N / 2; b++) {
            if (klog) klog[b] = 0.0;
            if (pklog) pklog[b] = 0.0;
            if (countlog) countlog[b] = 0.0;
        }
    } else {
        // the log power takes the monopole only (:398-402)
        std::vector<double> lg(hb.begin() + 3 * nb, hb.end());
        emit(lg.data(), klog, pklog, countlog);
        if (ipol && pklog)
            for (int b = 0; b < N / 2; b++) pklog[b] = 0.0;
    }
    return 0;
}

int mgs_power_spectrum(mgs_handle* h, int32_t which, double* k, double* pk, double* count)
{
    return mgs_power_spectrum_ex(h, which, 0, 0, k, pk, count, nullptr, nullptr, nullptr);
}

// the power-of-two form (mgs_poisson.hip)
static int potential_pow2(mgs_handle* h, float* phi, double trfi)
{
    int rc = fft_ensure_cplx(h);
    if (rc) return rc;
    FftState* f = fft_of(h);
    const int N = f->N;
    if ((rc = fft_ensure_tables(h))) return rc;
    launch_poisson(h->L[0].rho, f->cplx, phi, f->tables, N, trfi, h->s);
    return 0;
}

int mgs_potential(mgs_handle* h, double trfi)
{
    if (!h) return MGS_E_ARG;
    if (!std::isfinite(trfi)) return set_err(h, MGS_E_ARG, "trfi not finite");
    if (!h->has_density) return set_err(h, MGS_E_STATE, "no density set");
    float* phi = pm_potential(h);
    if (!phi) return set_err(h, MGS_E_NOMEM, "potential buffer");
    const int N = h->p.ngrid;
    const double n3 = (double)N * N * N;
    int rc;
    if (poisson_grid(N)) {
        prof_begin(h, MGS_KC_PM, 8.0 * n3 * 2.0 + 12.0 * n3);
        rc = potential_pow2(h, phi, trfi);
        prof_end(h);
        if (rc) return rc;
    } else {
        if ((rc = fft_ensure(h)) || (rc = fft_ensure_inverse(h))) return rc;
        FftState* f = fft_of(h);
        if ((rc = fft_ensure_tables(h))) return rc;
        prof_begin(h, MGS_KC_PM, 8.0 * n3 * 2.0 + 12.0 * n3);
        launch_unpack_f64_to_f64(h->L[0].rho, f->real, N, 1.0, h->s);
        if (hipfftExecD2Z(f->fwd, f->real, f->cplx) != HIPFFT_SUCCESS) return set_err(h, MGS_E_HIP, "hipfftExecD2Z");
        hipLaunchKernelGGL(k_green, dim3((unsigned)std::min(N * N, 65536)), dim3(256), 0, h->s, f->cplx, N, trfi, 1.0 / n3,
                           (const double*)f->tables);
        if (hipfftExecZ2D(f->inv, f->cplx, f->real) != HIPFFT_SUCCESS) return set_err(h, MGS_E_HIP, "hipfftExecZ2D");
        // FI is REAL*4 between the reference's transform passes and after them
        hipLaunchKernelGGL(k_to_f32, grid_for((size_t)n3), dim3(256), 0, h->s, f->real, phi, (size_t)n3);
        prof_end(h);
    }
    if (hipStreamSynchronize(h->s) != hipSuccess) return set_err(h, MGS_E_HIP, "potential");
    return 0;
}

int mgs_potential_add_fifth_force(mgs_handle* h)
{
    if (!h) return MGS_E_ARG;
    float* phi = pm_potential(h);
    if (!phi) return set_err(h, MGS_E_NOMEM, "potential buffer");
    const int N = h->p.ngrid;
    const size_t n3 = (size_t)N * N * N;
    prof_begin(h, MGS_KC_PM, 16.0 * (double)n3);
    const Launch L = make_launch(N / 2, (long)N * N);
    hipLaunchKernelGGL(k_add_psi, L.grid, L.block, 0, h->s, phi, h->L[0].u, make_geo(N), psi_of_handle(h), L.TX, L.TY,
                       L.XB, L.NB);
    prof_end(h);
    if (hipStreamSynchronize(h->s) != hipSuccess) return set_err(h, MGS_E_HIP, "fifth-force potential");
    return 0;
}

int mgs_set_potential(mgs_handle* h, const void* src, int32_t dtype, int32_t where)
{
    if (!h || !src) return set_err(h, MGS_E_ARG, "NULL argument");
    if (dtype != MGS_F32 && dtype != MGS_F64) return set_err(h, MGS_E_ARG, "dtype");
    if (where != MGS_HOST && where != MGS_DEVICE) return set_err(h, MGS_E_ARG, "where");
    float* phi = pm_potential(h);
    if (!phi) return set_err(h, MGS_E_NOMEM, "potential buffer");
    const int N = h->p.ngrid;
    const size_t n3 = (size_t)N * N * N;
    const size_t bytes = n3 * (dtype == MGS_F32 ? 4 : 8);
    if (dtype == MGS_F32) {
        if (hipMemcpyAsync(phi, src, bytes, where == MGS_HOST ? hipMemcpyHostToDevice : hipMemcpyDeviceToDevice,
                           h->s) != hipSuccess)
            return set_err(h, MGS_E_HIP, "potential upload");
    } else {
        const void* d = src;
        if (where == MGS_HOST) {
            int rc = ensure_staging(h, bytes);
            if (rc) return rc;
            if (hipMemcpyAsync(h->staging, src, bytes, hipMemcpyHostToDevice, h->s) != hipSuccess)
                return set_err(h, MGS_E_HIP, "potential upload");
            d = h->staging;
        }
        hipLaunchKernelGGL(k_to_f32, grid_for(n3), dim3(256), 0, h->s, (const double*)d, phi, n3);
    }
    if (hipStreamSynchronize(h->s) != hipSuccess) return set_err(h, MGS_E_HIP, "potential upload");
    return 0;
}

int mgs_get_potential(mgs_handle* h, void* dst, int32_t dtype, int32_t where)
{
    if (!h || !dst) return set_err(h, MGS_E_ARG, "NULL argument");
    if (dtype != MGS_F32 && dtype != MGS_F64) return set_err(h, MGS_E_ARG, "dtype");
    if (where != MGS_HOST && where != MGS_DEVICE) return set_err(h, MGS_E_ARG, "where");
    if (!h->pm) return set_err(h, MGS_E_STATE, "no potential: call mgs_potential first");
    float* phi = pm_potential(h);
    const int N = h->p.ngrid;
    const size_t n3 = (size_t)N * N * N;
    const size_t bytes = n3 * (dtype == MGS_F32 ? 4 : 8);
    void* out = dst;
    if (where == MGS_HOST) {
        int rc = ensure_staging(h, bytes);
        if (rc) return rc;
        out = h->staging;
    }
    if (dtype == MGS_F64)
        hipLaunchKernelGGL(k_to_f64, grid_for(n3), dim3(256), 0, h->s, phi, (double*)out, n3);
    else if (hipMemcpyAsync(out, phi, bytes, hipMemcpyDeviceToDevice, h->s) != hipSuccess)
        return set_err(h, MGS_E_HIP, "potential copy");
    if (where == MGS_HOST && hipMemcpyAsync(dst, out, bytes, hipMemcpyDeviceToHost, h->s) != hipSuccess)
        return set_err(h, MGS_E_HIP, "potential copy");
    if (hipStreamSynchronize(h->s) != hipSuccess) return set_err(h, MGS_E_HIP, "potential copy");
    return 0;
}

}  // extern "C"
