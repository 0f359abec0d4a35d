"""Device memory that calls take beside their inputs."""
import numpy as np
import pytest

import mgsolve as M

MIB = 1 << 20


# per particle a record of 8 bytes and an index of 4, and a word per 512
# particles; allocations are rounded up, to 2 MiB at most
@pytest.mark.gpu
def test_deposit_takes_twelve_bytes_a_particle():
    import torch

    N, n = 32, 1 << 24
    rng = np.random.default_rng(5)
    pos = [rng.uniform(1.0, N + 0.99, n).astype(np.float32) for _ in range(3)]
    with M.Solver(M.Config(N=N, model=M.MODEL_FR, fr_n=1, box=2.0 * N, fr0=-1e-5, precision=M.PREC_FP64)) as S:
        S.set_particles(*[a[:1000] for a in pos])
        S.cic_deposit()  # loads the kernels and makes the per-tile arrays
        S.set_particles(*pos)
        print(f"[memory] deposit of {n} particles", flush=True)
        before = torch.cuda.mem_get_info()[0]
        S.cic_deposit()
        taken = before - torch.cuda.mem_get_info()[0]
        mean = S.get_density(np.float64).mean()
    assert taken <= 12 * n + 4 * n // 512 + 3 * 2 * MIB, taken / MIB
    # eight weights a particle, each rounded to a multiple of 2^-40
    assert abs(mean) <= 8 * n / N ** 3 * 2.0 ** -41 + 1e-12


# FP64 nDGP on a grid whose passes do not z-march (h = 450): its levels, the
# passes' scratch and the norm's partials take 19.1 GB, and the field's second
# array, which it can do without, 5.8
@pytest.mark.gpu
def test_ndgp_handle_fits_without_its_second_array():
    import torch

    room, held = 22 * 10 ** 9, []
    try:
        while True:
            free = torch.cuda.mem_get_info()[0] - room
            if free < 64 * MIB:
                break
            held.append(torch.empty(min(free, 1 << 36), dtype=torch.uint8, device="cuda"))
        print(f"[memory] nDGP 900^3 in {torch.cuda.mem_get_info()[0] / 1e9:.1f} GB", flush=True)
        with M.Solver(M.Config(N=900, model=M.MODEL_DGP, branch=1, box=900.0, h0rc=1.0, precision=M.PREC_FP64)) as S:
            S.initialise()
    finally:
        held.clear()
        torch.cuda.empty_cache()
