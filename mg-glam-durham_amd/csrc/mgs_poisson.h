// mgs_poisson.h -- the power-of-two Poisson solve (mgs_poisson.hip) and the
// Green's function table it shares with the general one (mgs_fft.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/mgsolve.h"

namespace mgs {

// the reference's GREENf table over the complex wavenumber k: see k_green
__device__ __forceinline__ double green_g(int k, int N)
{
    const double P16 = (double)6.28318530718f;
    const int i = k <= N / 2 ? k : N - k;
    if (2 * i == N) return -2.0;
    return 2.0 * cos(P16 * i / N);
}

// fifth-force potential of a cell with field value v
struct PsiOf {
    int model, frn;
    double fct, inv_ubg;
    __device__ __forceinline__ double operator()(double v) const
    {
        if (model == MGS_MODEL_DGP) return 0.5 * v;
        const double x = v * inv_ubg;
        const double w = frn == 0 ? x : (frn == 1 ? x * x : x * x * x);
        return -fct * w;
    }
};

__device__ __forceinline__ int fold(int a, int N) { return a <= N / 2 ? a : a - N; }

// POWERfft5's binning of one entry of the half spectrum (PMP2mod_power.f90:
// 359-410): wavenumbers i = 0 .. N/2, my, mz, squared amplitude amp, into hist
// (power, mode count and sum of |m| of the linear bins, then of the log bins,
// nb each).  An entry stands for itself and, but at i = 0 and N/2, for its
// conjugate mirror.  |m|, the bin boundaries and the weights are the
// reference's REAL*4 values (RK = sqrt(REAL(|m|^2)) correctly rounded, as the
// compiled reference's is); the log bin of each |m|^2 comes from a table the
// host fills with the C library's log10f, the function the compiled reference
// calls.  The quadrupole's line of sight is z: the reference fills its bins
// after the I <-> K transposition (:307-316), so its MI is the z wavenumber.
// LOGB: also fill the log bins (NGP only)
template <int IPOL, int ICIC, bool LOGB>
__device__ __forceinline__ void bin_mode(double* hist, int nb, int N, int i, int my, int mz, double amp,
                                         const int* __restrict__ logbin)
{
    const int n2 = i * i + my * my + mz * mz;
    if (n2 == 0) return;  // RK < 0.5: the mean
    const float rk = sqrtf((float)n2);
    const double w = (i == 0 || 2 * i == N) ? 1.0 : 2.0;  // conjugate half
    if (IPOL) {
        const float cosmu2 = (float)(mz * mz) / (rk * rk);
        amp *= (double)(1.5f * cosmu2 - 0.5f);
    }
    if (ICIC) {
        int mp = (int)(rk + 0.0001f);
        if (mp < 1) mp = 1;
        const int mp2 = mp + 1 < N ? mp + 1 : N;
        const float w1 = (float)mp - rk + 1.0f;
        const float w2 = 1.0f - w1;
        const float d1 = (float)mp, d2 = d1 + 1.0f;
        if (mp < nb) {
            atomicAdd(&hist[mp], w * amp * (double)w1);
            atomicAdd(&hist[nb + mp], w * (double)w1);
            atomicAdd(&hist[2 * nb + mp], w * (double)(d1 * w1));
        }
        if (mp2 < nb) {
            atomicAdd(&hist[mp2], w * amp * (double)w2);
            atomicAdd(&hist[nb + mp2], w * (double)w2);
            atomicAdd(&hist[2 * nb + mp2], w * (double)(d2 * w2));
        }
    } else {
        int mp = (int)(rk + 0.5f);
        if (mp < 1) mp = 1;
        if (mp < nb) {
            atomicAdd(&hist[mp], w * amp);
            atomicAdd(&hist[nb + mp], w);
            atomicAdd(&hist[2 * nb + mp], w * (double)rk);
        }
        const int ml = LOGB ? logbin[n2] : nb;
        if (LOGB && ml < nb) {
            if (!IPOL) atomicAdd(&hist[3 * nb + ml], w * amp);
            atomicAdd(&hist[4 * nb + ml], w);
            atomicAdd(&hist[5 * nb + ml], w * (double)rk);
        }
    }
}

bool poisson_grid(int N);  // power of two, 32 .. 1024
size_t poisson_table_bytes(int N);
void launch_poisson_tables(void* tables, int N, hipStream_t s);
// phi (REAL*4, x fastest) from the colour-split density; work: N^3 doubles
void launch_poisson(const double* rho, void* work, float* phi, const void* tables, int N, double trfi, hipStream_t s);

// The binned power of a colour-split field (psi: of its fifth-force potential)
// on such a grid: histograms of 6 (N/2 + 1) doubles into part, one per block;
// returns their number (at most SPECTRUM_BLOCKS).  ipol, icic, logb as in
// bin_mode's template arguments.
constexpr int SPECTRUM_BLOCKS = 512 + 64;
int launch_spectrum(const double* field, const PsiOf* psi, void* work, const void* tables, int N, double norm, int ipol,
                    int icic, bool logb, const int* logbin, double* part, hipStream_t s);

}  // namespace mgs
