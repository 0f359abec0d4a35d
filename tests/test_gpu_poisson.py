"""The power-of-two Poisson solve (mgs_poisson.hip) over its whole range, 32 to
1024, against FP64 transforms by torch, and beside it the grids that take the
FFT library."""
import ctypes

import numpy as np
import pytest

import mgsolve as M


def _potential(delta, trfi):
    """POTENTfft5 in FP64 (see mgs_fft.hip's k_green for the eigenvalue's table)"""
    import torch

    N = delta.shape[0]
    twopi = float(np.float32(6.28318530718))
    i = torch.arange(N, device="cuda")
    i = torch.minimum(i, N - i)
    g = torch.where(2 * i == N, -2.0, 2.0 * torch.cos(twopi * i.double() / N))
    c = torch.fft.rfftn(delta)
    for z in range(N):  # plane by plane: no second array of the spectrum's size
        a = (g[:, None] - 6.0 + g[None, :N // 2 + 1]) + g[z]
        c[z] *= trfi / torch.where(a.abs() < 1e-7, torch.ones_like(a), a)
    return torch.fft.irfftn(c, s=(N, N, N))


@pytest.mark.gpu
@pytest.mark.parametrize("N", [32, 64, 128, 256, 512, 1024, 16, 48])
def test_potential_matches_fp64_transforms(N):
    import torch

    gen = torch.Generator(device="cuda")
    gen.manual_seed(N)
    delta = torch.randn((N, N, N), generator=gen, device="cuda", dtype=torch.float64)
    delta += 0.3  # a mean, which the mean mode multiplies by trfi
    torch.cuda.synchronize()
    print(f"[poisson] N={N}", flush=True)
    out = torch.empty((N, N, N), device="cuda", dtype=torch.float32)
    with M.Solver(M.Config(N=N, box=2.0 * N, precision=M.PREC_FP64)) as S:
        S._chk(S.L.mgs_set_density(S.h, ctypes.c_void_p(delta.data_ptr()), M.F64, M.DEVICE), "density")
        for _ in range(2):  # the second solve reuses the work array and the tables
            S.potential(0.45)
        S._chk(S.L.mgs_get_potential(S.h, ctypes.c_void_p(out.data_ptr()), M.F32, M.DEVICE), "potential")
    ref = _potential(delta, 0.45)
    big = float(ref.abs().max())
    # rounded once to REAL*4: half an ulp of the largest value, and the
    # transforms' FP64 rounding (1e-15 of the norm)
    assert float((out.double() - ref).abs().max()) <= 2.0 ** -24 * big * 1.001
    assert float((out == ref.float()).double().mean()) > 0.999
