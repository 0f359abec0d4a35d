"""The one-launch forms of the small inner levels (the tail, the half-cycle
blocks) against the server's operation-by-operation launches of the same
cycle, bit for bit, on grids whose coarse levels meet their edges."""
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
