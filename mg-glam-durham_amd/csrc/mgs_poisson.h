// mgs_poisson.h -- the power-of-two Poisson solve (mgs_poisson.hip) and the
// Green's function table it shares with the general one (mgs_fft.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace mgs {

// the reference's GREENf table over the complex wavenumber k: see k_green
__device__ __forceinline__ double green_g(int k, int N)
{
    const double P16 = (double)6.28318530718f;
    const int i = k <= N / 2 ? k : N - k;
    if (2 * i == N) return -2.0;
    return 2.0 * cos(P16 * i / N);
}

bool poisson_grid(int N);  // power of two, 32 .. 1024
size_t poisson_table_bytes(int N);
void launch_poisson_tables(void* tables, int N, hipStream_t s);
// phi (REAL*4, x fastest) from the colour-split density; work: N^3 doubles
void launch_poisson(const double* rho, void* work, float* phi, const void* tables, int N, double trfi, hipStream_t s);

}  // namespace mgs
