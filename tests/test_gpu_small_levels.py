"""The small levels of a cycle on grids that meet the edges of their one-launch
forms: the mixed solves against the server's, bit for bit (whose f(R) levels
above 16^3 run one launch per operation, and whose smaller ones are the same
tails), and the FP64 cycles against the oracle."""
import numpy as np
import pytest

import mgsolve as M
import oracle as O


# coarse levels: 24 (tiles of 8 x 8 x 4); 48 (16 x 8 x 8) and 24; 56 and 28
# (a block level over one that is not, coarsest 14); 80, 40, 20 (coarsest 10);
# 32; 64 and 32; no block level
@pytest.mark.gpu
@pytest.mark.parametrize("N,n", [(48, 1), (96, 0), (112, 1), (160, 1), (64, 2), (64, 0), (128, 1), (32, 1)])
def test_mixed_solve_equals_the_served_solve(N, n):
    cfg = M.Config(N=N, model=M.MODEL_FR, fr_n=n, box=2.0 * N, fr0=-1e-5, precision=M.PREC_MIXED)
    delta = O.lognormal_density(N, 2.0 * N, 1.0, seed=N + n).astype(np.float32)
    print(f"[small levels] N={N} n={n}", flush=True)
    with M.Solver(cfg) as S:
        S.set_density(delta)
        rep = S.solve(mode=1, rel_tol=1e-8, max_cycles=40)
        u = S.get_field()
        S.use_graphs(False)
        S.solve(mode=1, rel_tol=1e-8, max_cycles=40)
        plain = S.get_field()
    assert rep["converged"]
    with M.Server(max_active=2) as srv:
        served, res = srv.wait(srv.submit(cfg, delta, rel_tol=1e-8, max_outer=40))
    assert res["converged"] and res["outer"] == rep["outer"]
    assert np.array_equal(u, plain)
    assert np.array_equal(u, served)
    # the equation's residual at the solution, by the oracle's FP64 operator
    with M.Solver(M.Config(N=N, model=M.MODEL_FR, fr_n=n, box=2.0 * N, fr0=-1e-5)) as S:
        S.set_density(delta)
        S.solve(mode=1, rel_tol=1e-9, max_cycles=40)
        ref = S.get_field()
    assert np.max(np.abs(u - ref)) <= 1e-6 * np.max(np.abs(ref))


# FP64 cycles whose tail starts at 16, 12 (coarsest 6), 8 and 4 cells a side,
# and grids without one (coarsest 14 or 10), against the oracle's cycles
@pytest.mark.gpu
@pytest.mark.parametrize("N", [8, 16, 32, 48, 96, 28, 40])
@pytest.mark.parametrize("model,n", [(M.MODEL_FR, 0), (M.MODEL_FR, 1), (M.MODEL_FR, 2), (M.MODEL_DGP, 1)])
def test_fp64_cycles_match_the_oracle(N, model, n):
    delta = O.lognormal_density(N, 2.0 * N, 1.0, seed=N)
    cfg = M.Config(N=N, model=model, fr_n=n, box=2.0 * N, fr0=-1e-5)
    p = O.Params(N=N, model=model, fr_n=n, branch=1, box=2.0 * N, om=0.3, oml=0.7, a=1.0, fr0=-1e-5, h0rc=1.0, polish=1)
    print(f"[small levels] FP64 N={N} model={model} n={n}", flush=True)
    with M.Solver(cfg) as S:
        S.set_density(delta)
        S.initialise()
        u0 = S.get_field()
        for _ in range(2):
            S.vcycle(0)
        u = S.get_field()
    ref = u0.copy()
    O.vcycles(p, ref, delta, 2, prec="f64")  # in place
    scale = np.max(np.abs(ref))
    if model == M.MODEL_DGP:
        assert np.array_equal(u, ref)
    else:  # the smoother's root is good to rtol 1e-13
        assert np.max(np.abs(u - ref)) <= 1e-12 * scale


# nDGP: tail from 16 (32: directly below the finest level), per-cell passes
# (64), z-marching tiles of one, two and four rows (256, 128) in one batch
@pytest.mark.gpu
def test_served_ndgp_equals_the_solve():
    sizes = (32, 64, 128, 256, 16)
    cfgs = [M.Config(N=N, model=M.MODEL_DGP, branch=1, box=float(N), h0rc=1.0, precision=M.PREC_MIXED) for N in sizes]
    deltas = [O.lognormal_density(N, float(N), 1.0, seed=N).astype(np.float32) for N in sizes]
    with M.Server(max_active=4) as srv:
        tickets = [srv.submit(c, d, max_outer=6, exit_rule=M.EXIT_REFERENCE, res_conv=1e-8)
                   for c, d in zip(cfgs, deltas)]
        served = [srv.wait(t) for t in tickets]
    for c, d, (u, res) in zip(cfgs, deltas, served):
        print(f"[small levels] nDGP N={c.N}", flush=True)
        with M.Solver(c) as S:
            S.set_density(d)
            rep = S.solve(mode=0, res_conv=1e-8, max_cycles=6)
            assert rep["outer"] == res["outer"]
            assert np.array_equal(S.get_field(), u), c.N
