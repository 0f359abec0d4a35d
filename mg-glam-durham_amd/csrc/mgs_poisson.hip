// mgs_poisson.hip -- the PM step's Poisson solve on power-of-two grids:
// POTENTfft5's transforms and Green's function (PMP2main.f90:705-867) in five
// passes over the grid, from the solver's colour-split density to the REAL*4
// potential.
//
// Through the FFT library the solve was nine passes: the density to a
// lexicographic array, three transforms, the Green's function, three
// transforms, the rounding to REAL*4; each a stream of 1 to 2 GB at 512^3.
// Here
//   1. x forward: the colour-split row is the packed real row (x = 2m and 2m+1
//      are the real and imaginary part of entry m), so the density is read
//      where it lies; N/2 complex outputs, entry 0 holding the real
//      coefficients of kx = 0 and kx = N/2;
//   2. y forward, in place;
//   3. z forward, Green's function and z inverse in one pass: a column's
//      spectrum stays in registers between the two;
//   4. y inverse, in place;
//   5. x inverse, rounded to REAL*4 as it is stored.
// All transforms are Stockham's autosort form in FP64, 8 values per thread,
// radices 8, 4 and 2, exchanged through LDS; twiddle factors come from a
// table.  A y or z block takes 8 neighbouring kx, so that its accesses are
// 128-byte lines.
//
// 512^3: 395 us (5.4 TB/s), 430, 674, 414 (5.2 TB/s) and 334 us, 2.25 ms in
// all, where the nine passes took 5.2 ms; 10.2 GB pass through HBM instead of
// 26.  The z pass, two transforms and a division per entry between one load
// and one store, is bound by latency at four waves per SIMD, the others by
// HBM.  No library plan is made for these grids (12 ms of a handle's first
// solve).

#include <math.h>

#include "mgs_device.h"
#include "mgs_internal.h"
#include "mgs_poisson.h"

namespace mgs {

struct Cx {
    double x, y;
};

__device__ __forceinline__ Cx operator+(Cx a, Cx b) { return Cx{a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ Cx operator-(Cx a, Cx b) { return Cx{a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ Cx cmul(Cx a, Cx b)
{
    return Cx{__builtin_fma(a.x, b.x, -a.y * b.y), __builtin_fma(a.x, b.y, a.y * b.x)};
}
__device__ __forceinline__ Cx conj(Cx a) { return Cx{a.x, -a.y}; }
// a times -i (DIR = -1, forward) or +i (inverse)
template <int DIR>
__device__ __forceinline__ Cx rot(Cx a)
{
    return DIR < 0 ? Cx{a.y, -a.x} : Cx{-a.y, a.x};
}

template <int DIR>
__device__ __forceinline__ void fft2(Cx& a, Cx& b)
{
    const Cx t = a - b;
    a = a + b;
    b = t;
}

// natural order in and out
template <int DIR>
__device__ __forceinline__ void fft4(Cx& a, Cx& b, Cx& c, Cx& d)
{
    fft2<DIR>(a, c);
    fft2<DIR>(b, d);
    d = rot<DIR>(d);
    fft2<DIR>(a, b);  // outputs 0, 2
    fft2<DIR>(c, d);  // outputs 1, 3
    const Cx t = b;
    b = c;
    c = t;
}

template <int DIR>
__device__ __forceinline__ void fft8(Cx* v)
{
    const double h = 0.70710678118654752440;
    Cx e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6], o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
    fft4<DIR>(e0, e1, e2, e3);
    fft4<DIR>(o0, o1, o2, o3);
    // odd outputs times exp(DIR 2 pi i k / 8)
    o1 = DIR < 0 ? Cx{(o1.x + o1.y) * h, (o1.y - o1.x) * h} : Cx{(o1.x - o1.y) * h, (o1.x + o1.y) * h};
    o2 = rot<DIR>(o2);
    o3 = DIR < 0 ? Cx{(o3.y - o3.x) * h, -(o3.x + o3.y) * h} : Cx{-(o3.x + o3.y) * h, (o3.x - o3.y) * h};
    v[0] = e0 + o0, v[4] = e0 - o0;
    v[1] = e1 + o1, v[5] = e1 - o1;
    v[2] = e2 + o2, v[6] = e2 - o2;
    v[3] = e3 + o3, v[7] = e3 - o3;
}

// radix of the next stage with `rem` of the length left
constexpr int next_radix(int rem) { return rem >= 8 && rem != 16 ? 8 : (rem >= 4 ? 4 : 2); }

// One stage of a length-L transform, Ns the product of the radices before it:
// thread j of the L/8 holds entries j + e L/8 in v[e]; butterfly b of its 8/R
// takes e = b, b + 8/R, ...  tw: exp(-2 pi i k / (TS L)), k < TS L.
template <int L, int TS, int R, int Ns, int DIR>
__device__ __forceinline__ void fft_stage(Cx* v, int j, const Cx* __restrict__ tw)
{
    constexpr int NB = 8 / R, T = L / 8;
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int jj = j + b * T;
        Cx w[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            w[r] = v[b + r * NB];
            if (Ns > 1 && r > 0) {
                const Cx t = tw[TS * (L / (Ns * R)) * ((jj % Ns) * r)];
                w[r] = cmul(w[r], DIR < 0 ? t : conj(t));
            }
        }
        if constexpr (R == 8)
            fft8<DIR>(w);
        else if constexpr (R == 4)
            fft4<DIR>(w[0], w[1], w[2], w[3]);
        else
            fft2<DIR>(w[0], w[1]);
#pragma unroll
        for (int r = 0; r < R; r++) v[b + r * NB] = w[r];
    }
}

// The transform of length L on the 8 values of each of its L/8 threads:
// entries j + e L/8 in v[e] before and after.  X(pos): LDS place of entry pos;
// every thread of the block takes part.
template <int L, int TS, int DIR, int Ns, class X>
__device__ __forceinline__ void fft_from(Cx* v, int j, const Cx* __restrict__ tw, Cx* lds, X at)
{
    constexpr int R = next_radix(L / Ns), NB = 8 / R, T = L / 8;
    fft_stage<L, TS, R, Ns, DIR>(v, j, tw);
    if constexpr (Ns * R < L) {
        __syncthreads();  // the exchange before this one has been read
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int jj = j + b * T, o = (jj / Ns) * Ns * R + jj % Ns;
#pragma unroll
            for (int r = 0; r < R; r++) lds[at(o + r * Ns)] = v[b + r * NB];
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = lds[at(j + e * T)];
        fft_from<L, TS, DIR, Ns * R>(v, j, tw, lds, at);
    }
}

// Green's function of the discrete Laplacian: see k_green in mgs_fft.hip
__device__ __forceinline__ double green_scale(double gx, double gy, double gz, double trfi, double inv_n3)
{
    double A = gy - 6.0;
    A = gx + A;
    A = A + gz;
    if (fabs(A) < 1.0e-7) A = 1.0;
    return trfi / A * inv_n3;
}

// ---- x: rows of N reals <-> N/2 complex -----------------------------------
// ROWS rows per block; LDS rows padded by one entry in 8 (the exchange writes
// entries 8 apart)
template <int N>
struct RowPlan {
    static constexpr int M = N / 2, T = M / 8, ROWS = 256 / T < 1 ? 1 : 256 / T, THREADS = T * ROWS;
    static constexpr int LD = M + M / 8 + 1;
};

// VAL: what is transformed, of a cell's value
struct Identity {
    __device__ __forceinline__ double operator()(double v) const { return v; }
};

template <int N, class VAL>
__global__ __launch_bounds__(RowPlan<N>::THREADS) void k_x_forward(const double* __restrict__ rho, Cx* __restrict__ out,
                                                                   const Cx* __restrict__ tw, VAL val)
{
    using P = RowPlan<N>;
    __shared__ Cx lds[P::ROWS * P::LD];
    const int j = threadIdx.x % P::T, rl = threadIdx.x / P::T;
    const unsigned row = blockIdx.x * P::ROWS + rl;  // y + N z; a multiple of ROWS rows
    const Geo g = make_geo(N);
    const bool odd = ((row % N) + (row / N)) & 1;
    const double* even = rho + (odd ? g.half : 0) + (size_t)row * P::M;
    const double* other = rho + (odd ? 0 : g.half) + (size_t)row * P::M;
    Cx* const l = lds + rl * P::LD;
    auto at = [](int p) { return p + (p >> 3); };
    Cx v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = Cx{even[j + e * P::T], other[j + e * P::T]};
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = Cx{val(v[e].x), val(v[e].y)};  // (branches: after every load is issued)
    fft_from<P::M, 2, -1, 1>(v, j, tw, l, at);
    // X[k] = (Z[k] + Z*[M-k]) / 2 - i/2 exp(-2 pi i k / N) (Z[k] - Z*[M-k])
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 8; e++) l[at(j + e * P::T)] = v[e];
    __syncthreads();
    Cx* o = out + (size_t)row * P::M;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const int k = j + e * P::T;
        if (k == 0) {
            o[0] = Cx{v[0].x + v[0].y, v[0].x - v[0].y};  // kx = 0 and N/2, both real
            continue;
        }
        const Cx z = v[e], y = conj(l[at(P::M - k)]);
        const Cx s = z + y, d = cmul(z - y, tw[k]);
        o[k] = Cx{0.5 * (s.x + d.y), 0.5 * (s.y - d.x)};
    }
}

template <int N>
__global__ __launch_bounds__(RowPlan<N>::THREADS) void k_x_inverse(const Cx* __restrict__ in, float* __restrict__ phi,
                                                                   const Cx* __restrict__ tw)
{
    using P = RowPlan<N>;
    __shared__ Cx lds[P::ROWS * P::LD];
    const int j = threadIdx.x % P::T, rl = threadIdx.x / P::T;
    const unsigned row = blockIdx.x * P::ROWS + rl;
    Cx* const l = lds + rl * P::LD;
    auto at = [](int p) { return p + (p >> 3); };
    const Cx* x = in + (size_t)row * P::M;
    Cx v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = x[j + e * P::T];
#pragma unroll
    for (int e = 0; e < 8; e++) l[at(j + e * P::T)] = v[e];
    __syncthreads();
    // Z[k] = X[k] + X*[M-k] + i exp(2 pi i k / N) (X[k] - X*[M-k])
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const int k = j + e * P::T;
        if (k == 0) {
            v[e] = Cx{v[e].x + v[e].y, v[e].x - v[e].y};
            continue;
        }
        const Cx y = conj(l[at(P::M - k)]);
        const Cx d = cmul(v[e] - y, conj(tw[k]));
        v[e] = Cx{v[e].x + y.x - d.y, v[e].y + y.y + d.x};
    }
    fft_from<P::M, 2, 1, 1>(v, j, tw, l, at);
    float* o = phi + (size_t)row * N;
#pragma unroll
    for (int e = 0; e < 8; e++) *reinterpret_cast<float2*>(o + 2 * (j + e * P::T)) = make_float2((float)v[e].x, (float)v[e].y);
}

// ---- y and z: columns of the half spectrum --------------------------------
// C neighbouring kx per block (C = 8: 128-byte lines), N/8 threads per column.
// The half spectrum is [z][y][kx], kx < M = N/2.
template <int N>
struct ColPlan {
    static constexpr int M = N / 2, C = 8192 / N < 8 ? 8192 / N : (M < 8 ? M : 8), T = N / 8;
    static constexpr int THREADS = T * C;  // N = 1024: 128 KiB of LDS
};

template <int N, int DIR>
__global__ __launch_bounds__(ColPlan<N>::THREADS) void k_y_pass(Cx* __restrict__ a, const Cx* __restrict__ tw)
{
    using P = ColPlan<N>;
    __shared__ Cx lds[N * P::C];
    const int c = threadIdx.x % P::C, j = threadIdx.x / P::C;
    const unsigned tile = blockIdx.x % (P::M / P::C), z = blockIdx.x / (P::M / P::C);
    Cx* p = a + (size_t)z * N * P::M + tile * P::C + c;
    Cx v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = p[(size_t)(j + e * P::T) * P::M];
    fft_from<N, 1, DIR, 1>(v, j, tw, lds, [c](int q) { return q * P::C + c; });
#pragma unroll
    for (int e = 0; e < 8; e++) p[(size_t)(j + e * P::T) * P::M] = v[e];
}

// z forward, Green's function, z inverse; kx = 0, whose entries hold two
// coefficients each, is k_z_pair's
template <int N>
__global__ __launch_bounds__(ColPlan<N>::THREADS) void k_z_pass(Cx* __restrict__ a, const Cx* __restrict__ tw,
                                                                const double* __restrict__ green, double trfi,
                                                                double inv_n3)
{
    using P = ColPlan<N>;
    __shared__ Cx lds[N * P::C];
    const int c = threadIdx.x % P::C, j = threadIdx.x / P::C;
    const unsigned tile = blockIdx.x % (P::M / P::C), ky = blockIdx.x / (P::M / P::C);
    const int kx = (int)(tile * P::C) + c;
    Cx* p = a + (size_t)ky * P::M + kx;
    constexpr size_t plane = (size_t)N * P::M;
    auto at = [c](int q) { return q * P::C + c; };
    Cx v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = p[(size_t)(j + e * P::T) * plane];
    fft_from<N, 1, -1, 1>(v, j, tw, lds, at);
    const double gx = green[kx], gy = green[ky];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const double s = green_scale(gx, gy, green[j + e * P::T], trfi, inv_n3);
        v[e] = Cx{v[e].x * s, v[e].y * s};
    }
    fft_from<N, 1, 1, 1>(v, j, tw, lds, at);
    if (kx == 0) return;
#pragma unroll
    for (int e = 0; e < 8; e++) p[(size_t)(j + e * P::T) * plane] = v[e];
}

// kx = 0: with F0, F1 the spectra of the real fields packed as P = X0 + i X1
// (kx = 0 and N/2), P(k) = F0 + i F1 and P*(-k) = F0 - i F1, so scaling F0 by g0
// and F1 by g1 gives (g0 + g1)/2 P(k) + (g0 - g1)/2 P*(-k).  A block takes the
// columns ky and -ky.
template <int N>
__global__ __launch_bounds__(N / 4) void k_z_pair(Cx* __restrict__ a, const Cx* __restrict__ tw,
                                                  const double* __restrict__ green, double trfi, double inv_n3)
{
    constexpr int M = N / 2, T = N / 8;
    __shared__ Cx lds[2 * N];
    const int c = threadIdx.x & 1, j = threadIdx.x >> 1;
    const int ky0 = blockIdx.x, ky1 = ky0 == 0 ? 0 : N - ky0;  // ky0 <= N/2
    const int ky = c ? ky1 : ky0;
    Cx* p = a + (size_t)ky * M;
    constexpr size_t plane = (size_t)N * M;
    auto at = [c](int q) { return 2 * q + c; };
    Cx v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = p[(size_t)(j + e * T) * plane];
    fft_from<N, 1, -1, 1>(v, j, tw, lds, at);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 8; e++) lds[at(j + e * T)] = v[e];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const int kz = j + e * T, mz = kz == 0 ? 0 : N - kz;
        const Cx q = conj(lds[2 * mz + (1 - c)]);
        const double g0 = green_scale(green[0], green[ky], green[kz], trfi, inv_n3);
        const double g1 = green_scale(green[M], green[ky], green[kz], trfi, inv_n3);
        const double s = 0.5 * (g0 + g1), d = 0.5 * (g0 - g1);
        v[e] = Cx{s * v[e].x + d * q.x, s * v[e].y + d * q.y};
    }
    fft_from<N, 1, 1, 1>(v, j, tw, lds, at);
    if (c && ky1 == ky0) return;  // ky = 0 or N/2: one column, held twice
#pragma unroll
    for (int e = 0; e < 8; e++) p[(size_t)(j + e * T) * plane] = v[e];
}

// ---- power spectrum: the z transform and the binning in one pass -----------
// The x and y passes as above; the spectrum is binned from registers and never
// stored.  Blocks walk the column tiles with a histogram in LDS each.  Bound by
// the histogram's LDS atomics (24 per thread and tile): 73 us at 256^3, where
// the read alone takes 25.  With psi formed in the x pass once every load is
// issued (44 us; 60 as each value arrives) and the y pass (42 us) a spectrum of
// psi takes 0.17 ms; a pass for psi, the library's
// transform and a binning pass took 0.31.
template <int IPOL, int ICIC, bool LOGB, int N>
__global__ __launch_bounds__(ColPlan<N>::THREADS) void k_z_bin(const Cx* __restrict__ a, const Cx* __restrict__ tw,
                                                               double norm, const int* __restrict__ logbin,
                                                               double* __restrict__ part)
{
    using P = ColPlan<N>;
    constexpr int NB = N / 2 + 1, TILES = N * (P::M / P::C);
    __shared__ Cx lds[N * P::C];
    __shared__ double hist[6 * NB];
    for (int t = threadIdx.x; t < 6 * NB; t += P::THREADS) hist[t] = 0.0;
    const int c = threadIdx.x % P::C, j = threadIdx.x / P::C;
    constexpr size_t plane = (size_t)N * P::M;
    for (unsigned b = blockIdx.x; b < TILES; b += gridDim.x) {
        const int kx = (int)(b % (P::M / P::C)) * P::C + c, ky = (int)(b / (P::M / P::C));
        const Cx* p = a + (size_t)ky * P::M + kx;
        Cx v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = p[(size_t)(j + e * P::T) * plane];
        // (its first barrier also completes the histogram's clearing)
        fft_from<N, 1, -1, 1>(v, j, tw, lds, [c](int q) { return q * P::C + c; });
        if (kx != 0)  // (kx = 0 carries N/2 too: k_z_pair_bin)
#pragma unroll
            for (int e = 0; e < 8; e++)
                bin_mode<IPOL, ICIC, LOGB>(hist, NB, N, kx, fold(ky, N), fold(j + e * P::T, N),
                                           (v[e].x * v[e].x + v[e].y * v[e].y) * norm, logbin);
    }
    __syncthreads();
    for (int t = threadIdx.x; t < 6 * NB; t += P::THREADS) part[(size_t)blockIdx.x * 6 * NB + t] = hist[t];
}

// kx = 0 and N/2 (see k_z_pair): F0 = (P(k) + P*(-k)) / 2, F1 = (P(k) - P*(-k)) / 2i
template <int IPOL, int ICIC, bool LOGB, int N>
__global__ __launch_bounds__(N / 4) void k_z_pair_bin(const Cx* __restrict__ a, const Cx* __restrict__ tw, double norm,
                                                      const int* __restrict__ logbin, double* __restrict__ part)
{
    constexpr int M = N / 2, T = N / 8, NB = N / 2 + 1;
    __shared__ Cx lds[2 * N];
    __shared__ double hist[6 * NB];
    for (int t = threadIdx.x; t < 6 * NB; t += N / 4) hist[t] = 0.0;
    const int c = threadIdx.x & 1, j = threadIdx.x >> 1;
    constexpr size_t plane = (size_t)N * M;
    for (int ky0 = blockIdx.x; ky0 <= N / 2; ky0 += gridDim.x) {
        const int ky1 = ky0 == 0 ? 0 : N - ky0, ky = c ? ky1 : ky0;
        const Cx* p = a + (size_t)ky * M;
        Cx v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = p[(size_t)(j + e * T) * plane];
        auto at = [c](int q) { return 2 * q + c; };
        fft_from<N, 1, -1, 1>(v, j, tw, lds, at);
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 8; e++) lds[at(j + e * T)] = v[e];
        __syncthreads();
        if (!(c && ky1 == ky0))  // ky = 0 or N/2: one column, held twice
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int kz = j + e * T, mz = kz == 0 ? 0 : N - kz;
                const Cx q = conj(lds[2 * mz + (1 - c)]);
                const Cx f0 = v[e] + q, f1 = v[e] - q;
                bin_mode<IPOL, ICIC, LOGB>(hist, NB, N, 0, fold(ky, N), fold(kz, N),
                                           0.25 * (f0.x * f0.x + f0.y * f0.y) * norm, logbin);
                bin_mode<IPOL, ICIC, LOGB>(hist, NB, N, M, fold(ky, N), fold(kz, N),
                                           0.25 * (f1.x * f1.x + f1.y * f1.y) * norm, logbin);
            }
    }
    __syncthreads();
    for (int t = threadIdx.x; t < 6 * NB; t += N / 4) part[(size_t)blockIdx.x * 6 * NB + t] = hist[t];
}

// tw[k] = exp(-2 pi i k / N); green[k]: the reference's GREENf table (green_g)
__global__ __launch_bounds__(256) void k_poisson_tables(Cx* __restrict__ tw, double* __restrict__ green, int N)
{
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= N) return;
    double s, c;
    sincospi(2.0 * k / N, &s, &c);
    tw[k] = Cx{c, -s};
    green[k] = green_g(k, N);
}

bool poisson_grid(int N) { return N >= 32 && N <= 1024 && (N & (N - 1)) == 0; }

size_t poisson_table_bytes(int N) { return (size_t)N * (sizeof(Cx) + sizeof(double)); }

void launch_poisson_tables(void* tables, int N, hipStream_t s)
{
    Cx* tw = (Cx*)tables;
    hipLaunchKernelGGL(k_poisson_tables, dim3((N + 255) / 256), dim3(256), 0, s, tw, (double*)(tw + N), N);
}

template <int N>
static void poisson_n(const double* rho, Cx* a, float* phi, const Cx* tw, double trfi, hipStream_t s)
{
    using R = RowPlan<N>;
    using C = ColPlan<N>;
    const double* green = (const double*)(tw + N);
    const double inv_n3 = 1.0 / ((double)N * N * N);
    const dim3 rows((unsigned)N * N / R::ROWS), cols((unsigned)N * (C::M / C::C));
    hipLaunchKernelGGL((k_x_forward<N, Identity>), rows, dim3(R::THREADS), 0, s, rho, a, tw, Identity());
    hipLaunchKernelGGL((k_y_pass<N, -1>), cols, dim3(C::THREADS), 0, s, a, tw);
    hipLaunchKernelGGL((k_z_pass<N>), cols, dim3(C::THREADS), 0, s, a, tw, green, trfi, inv_n3);
    hipLaunchKernelGGL((k_z_pair<N>), dim3(N / 2 + 1), dim3(N / 4), 0, s, a, tw, green, trfi, inv_n3);
    hipLaunchKernelGGL((k_y_pass<N, 1>), cols, dim3(C::THREADS), 0, s, a, tw);
    hipLaunchKernelGGL((k_x_inverse<N>), rows, dim3(R::THREADS), 0, s, a, phi, tw);
}

void launch_poisson(const double* rho, void* work, float* phi, const void* tables, int N, double trfi, hipStream_t s)
{
    Cx* a = (Cx*)work;
    const Cx* tw = (const Cx*)tables;
    switch (N) {
    case 32: return poisson_n<32>(rho, a, phi, tw, trfi, s);
    case 64: return poisson_n<64>(rho, a, phi, tw, trfi, s);
    case 128: return poisson_n<128>(rho, a, phi, tw, trfi, s);
    case 256: return poisson_n<256>(rho, a, phi, tw, trfi, s);
    case 512: return poisson_n<512>(rho, a, phi, tw, trfi, s);
    case 1024: return poisson_n<1024>(rho, a, phi, tw, trfi, s);
    }
}

template <int IPOL, int ICIC, bool LOGB, int N>
static int spectrum_opt(const Cx* a, const Cx* tw, double norm, const int* logbin, double* part, hipStream_t s)
{
    using C = ColPlan<N>;
    constexpr int tiles = N * (C::M / C::C), blocks = tiles < 512 ? tiles : 512;
    constexpr int pairs = N / 2 + 1 < 64 ? N / 2 + 1 : 64;
    hipLaunchKernelGGL((k_z_bin<IPOL, ICIC, LOGB, N>), dim3(blocks), dim3(C::THREADS), 0, s, a, tw, norm, logbin, part);
    hipLaunchKernelGGL((k_z_pair_bin<IPOL, ICIC, LOGB, N>), dim3(pairs), dim3(N / 4), 0, s, a, tw, norm, logbin,
                       part + (size_t)blocks * 6 * (N / 2 + 1));
    return blocks + pairs;
}

template <int N>
static int spectrum_n(const double* field, const PsiOf* psi, Cx* a, const Cx* tw, double norm, int ipol, int icic,
                      bool logb, const int* logbin, double* part, hipStream_t s)
{
    using R = RowPlan<N>;
    using C = ColPlan<N>;
    const dim3 rows((unsigned)N * N / R::ROWS), cols((unsigned)N * (C::M / C::C));
    if (psi)
        hipLaunchKernelGGL((k_x_forward<N, PsiOf>), rows, dim3(R::THREADS), 0, s, field, a, tw, *psi);
    else
        hipLaunchKernelGGL((k_x_forward<N, Identity>), rows, dim3(R::THREADS), 0, s, field, a, tw, Identity());
    hipLaunchKernelGGL((k_y_pass<N, -1>), cols, dim3(C::THREADS), 0, s, a, tw);
    if (icic) return ipol ? spectrum_opt<1, 1, false, N>(a, tw, norm, logbin, part, s)
                          : spectrum_opt<0, 1, false, N>(a, tw, norm, logbin, part, s);
    if (logb) return ipol ? spectrum_opt<1, 0, true, N>(a, tw, norm, logbin, part, s)
                          : spectrum_opt<0, 0, true, N>(a, tw, norm, logbin, part, s);
    return ipol ? spectrum_opt<1, 0, false, N>(a, tw, norm, logbin, part, s)
                : spectrum_opt<0, 0, false, N>(a, tw, norm, logbin, part, s);
}

int launch_spectrum(const double* field, const PsiOf* psi, void* work, const void* tables, int N, double norm, int ipol,
                    int icic, bool logb, const int* logbin, double* part, hipStream_t s)
{
    Cx* a = (Cx*)work;
    const Cx* tw = (const Cx*)tables;
    switch (N) {
    case 32: return spectrum_n<32>(field, psi, a, tw, norm, ipol, icic, logb, logbin, part, s);
    case 64: return spectrum_n<64>(field, psi, a, tw, norm, ipol, icic, logb, logbin, part, s);
    case 128: return spectrum_n<128>(field, psi, a, tw, norm, ipol, icic, logb, logbin, part, s);
    case 256: return spectrum_n<256>(field, psi, a, tw, norm, ipol, icic, logb, logbin, part, s);
    case 512: return spectrum_n<512>(field, psi, a, tw, norm, ipol, icic, logb, logbin, part, s);
    default: return spectrum_n<1024>(field, psi, a, tw, norm, ipol, icic, logb, logbin, part, s);
    }
}

}  // namespace mgs
