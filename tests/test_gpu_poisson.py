"""The power-of-two Poisson solve and power spectrum (mgs_poisson.hip) over
their whole range, 32 to 1024, against FP64 transforms by torch and the oracle,
and beside them the grids that take the FFT library."""
import ctypes

import numpy as np
import pytest

import mgsolve as M
import oracle as O


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


def _binned(delta):
    """POWERfft5's linear NGP bins 1..N/2 (oracle.power_spectrum_ex) in FP64:
    (count, sum of |c_m|^2), plane by plane"""
    import torch

    N = delta.shape[0]
    nb = N // 2 + 1
    m = torch.arange(N, device="cuda")
    m = torch.where(m <= N // 2, m, m - N)
    c = torch.fft.rfftn(delta)
    w = torch.full((N, nb), 2.0, device="cuda", dtype=torch.float64)
    w[:, 0] = w[:, N // 2] = 1.0
    cnt = torch.zeros(N, device="cuda", dtype=torch.float64)
    pw = torch.zeros(N, device="cuda", dtype=torch.float64)
    for z in range(N):
        n2 = m[:, None] ** 2 + m[None, :nb] ** 2 + m[z] ** 2
        rk = n2.double().sqrt().float()  # correctly rounded
        b = (rk + np.float32(0.5)).long().clamp(min=1)
        ok = (n2 > 0) & (b < nb)
        cnt.index_add_(0, b[ok], w[ok])
        pw.index_add_(0, b[ok], (w * (c[z].abs() / N ** 3) ** 2)[ok])
    return cnt[1:nb].cpu().numpy(), pw[1:nb].cpu().numpy()


@pytest.mark.gpu
@pytest.mark.parametrize("N", [256, 512, 1024])
def test_spectrum_matches_fp64_transforms(N):
    import torch

    gen = torch.Generator(device="cuda")
    gen.manual_seed(N)
    delta = torch.randn((N, N, N), generator=gen, device="cuda", dtype=torch.float64)
    torch.cuda.synchronize()
    print(f"[spectrum] N={N}", flush=True)
    with M.Solver(M.Config(N=N, box=2.0 * N, precision=M.PREC_FP64)) as S:
        S._chk(S.L.mgs_set_density(S.h, ctypes.c_void_p(delta.data_ptr()), M.F64, M.DEVICE), "density")
        k, Pk, cnt = S.power_spectrum(0)
        ex = S.power_spectrum_ex(0, 0, 0)  # with the log bins
    cr, pr = _binned(delta)
    assert np.array_equal(cnt, cr) and np.array_equal(ex[2], cr)
    ref = (2.0 * N) ** 3 * pr / cr
    assert np.allclose(Pk, ref, rtol=1e-9) and np.allclose(ex[1], ref, rtol=1e-9)


@pytest.mark.gpu
@pytest.mark.parametrize("N", [32, 128])
@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("ipol,icic", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_spectrum_options_match_the_oracle(N, which, ipol, icic):
    rng = np.random.default_rng(7 * N + which)
    print(f"[spectrum] N={N} which={which} ipol={ipol} icic={icic}", flush=True)
    with M.Solver(M.Config(N=N, box=2.0 * N, precision=M.PREC_FP64)) as S:
        S.set_density(rng.standard_normal((N, N, N)))
        if which:
            S.set_field(rng.uniform(0.5, 1.5, (N, N, N)))
        got = S.power_spectrum_ex(which, ipol, icic)
        field = S.get_density() if which == 0 else S.get_field() if which == 1 else S.fifth_force()[0]
    ref = O.power_spectrum_ex(field, 2.0 * N, ipol, icic)
    # counts as in the oracle (linear weights summed in another order), the
    # powers to the rounding of an FP64 transform, of the largest bin
    for g, r, rtol in zip(got[:3], ref[:3], (1e-12, 1e-9, 1e-12)):
        assert np.allclose(g, r, rtol=rtol, atol=rtol * np.abs(r).max())
    if not icic:
        assert np.array_equal(got[2], ref[2])
        for g, r in zip(got[3:], ref[3:]):
            assert np.allclose(g, r, rtol=1e-9, atol=1e-9 * np.abs(r).max())
