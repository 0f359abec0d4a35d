"""Layout conversions and the fifth force at the edges of their launches:
the smallest grid, rows that do not fill a wave, a plane run that does not
divide the grid, wide rows, and caller arrays aligned only as their elements."""
import ctypes

import numpy as np
import pytest

import mgsolve as M
import oracle as O


@pytest.mark.gpu
@pytest.mark.parametrize("N", [2, 6, 34, 130])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("model", [M.MODEL_FR, M.MODEL_DGP])
def test_field_round_trip_and_fifth_force(N, dtype, model):
    import torch

    rng = np.random.default_rng(N)
    u = rng.uniform(0.1, 1.0, (N, N, N)) * 3e-3
    cfg = M.Config(N=N, model=model, fr_n=1, box=2.0 * N, fr0=-1e-5)
    td = torch.float32 if dtype == np.float32 else torch.float64
    dt = M.F32 if dtype == np.float32 else M.F64
    src = u.astype(dtype)
    with M.Solver(cfg) as S:
        # device arrays that start one element into their storage
        buf = torch.empty(N ** 3 + 1, dtype=td, device="cuda")
        buf[1:] = torch.from_numpy(src.reshape(-1)).to("cuda")
        out = torch.empty(N ** 3 + 1, dtype=td, device="cuda")
        ff = [torch.empty(N ** 3 + 1, dtype=td, device="cuda") for _ in range(4)]
        torch.cuda.synchronize()
        ptr = lambda t: ctypes.c_void_p(t[1:].data_ptr())  # noqa: E731
        S._chk(S.L.mgs_set_field(S.h, ptr(buf), dt, M.DEVICE), "set")
        S._chk(S.L.mgs_get_field(S.h, ptr(out), dt, M.DEVICE, 1.0), "get")
        S._chk(S.L.mgs_fifth_force(S.h, *[ptr(t) for t in ff], dt, M.DEVICE), "ff")
        half = S.get_field(dtype, 0.5)
        ubg = S.background()[1]
    assert np.array_equal(out[1:].cpu().numpy().reshape(N, N, N), src)
    assert np.array_equal(half, (src.astype(np.float64) * 0.5).astype(dtype))
    p = O.Params(N=N, model=model, fr_n=1, branch=1, box=2.0 * N, om=0.3, oml=0.7, a=1.0, fr0=-1e-5, h0rc=1.0)
    u64 = src.astype(np.float64)
    psi = O.fifth_force_potential(p, u64 / ubg if model == M.MODEL_FR else u64)
    # one FP64 product and difference apart, then rounded to dtype
    tol = 8 * np.finfo(dtype).eps * np.max(np.abs(psi))
    for got, ref in zip(ff, (psi, *O.central_gradient(psi))):
        assert np.max(np.abs(got[1:].cpu().numpy().reshape(N, N, N) - ref)) <= tol
