"""The one-launch forms of the small levels (tails, half-cycle blocks) against
one launch per operation, bit for bit.  A mistake in them would otherwise only
slow a mixed solve down, whose FP64 outer iteration corrects what the inner
cycle gets wrong."""
import numpy as np
import pytest

import mgsolve as M
import oracle as O


def _both(cfg, run):
    delta = O.lognormal_density(cfg.N, 2.0 * cfg.N, 1.0, seed=cfg.N).astype(np.float32)
    print(f"[fused levels] N={cfg.N} model={cfg.model} n={cfg.fr_n} precision={cfg.precision}", flush=True)
    out = []
    with M.Solver(cfg) as S:
        S.set_density(delta)
        for fused in (True, False, True):
            S.use_fused_levels(fused)
            rep = run(S)
            out.append((rep, S.get_field()))
    for rep, u in out[1:]:
        assert rep == out[0][0]
        assert np.array_equal(u, out[0][1])


def _solve(**opts):
    def run(S):
        rep = S.solve(**opts)
        return [rep[k] for k in ("converged", "outer", "cycles", "res0", "res_final")]
    return run


# tails from 16 (4 levels), 12 (to 6), 14's none; blocks 24 | 32, 48, 64, over a
# tail or over a level (28) that is neither
@pytest.mark.gpu
@pytest.mark.parametrize("N", [32, 48, 96, 112, 128])
@pytest.mark.parametrize("n", [0, 1, 2])
def test_mixed_fr(N, n):
    _both(M.Config(N=N, model=M.MODEL_FR, fr_n=n, box=2.0 * N, fr0=-1e-5, precision=M.PREC_MIXED),
          _solve(mode=1, rel_tol=1e-8, max_cycles=40))


@pytest.mark.gpu
@pytest.mark.parametrize("N", [8, 16, 32, 48, 96, 128])
@pytest.mark.parametrize("branch", [1, -1])
def test_mixed_ndgp(N, branch):
    _both(M.Config(N=N, model=M.MODEL_DGP, branch=branch, box=float(N), h0rc=1.0, precision=M.PREC_MIXED),
          _solve(mode=0, res_conv=1e-8, max_cycles=6))


# F and W cycles reach the tails from another caller; FP64 cycles
@pytest.mark.gpu
@pytest.mark.parametrize("model", [M.MODEL_FR, M.MODEL_DGP])
@pytest.mark.parametrize("cycle", [1, 2])
def test_other_cycles(model, cycle):
    _both(M.Config(N=96, model=model, fr_n=1, branch=1, box=192.0, fr0=-1e-5, precision=M.PREC_MIXED),
          _solve(mode=1, rel_tol=1e-6, max_cycles=3, cycle=cycle))


# (the levels' arrays too, which a caller can read)
@pytest.mark.gpu
@pytest.mark.parametrize("model,n", [(M.MODEL_FR, 0), (M.MODEL_FR, 1), (M.MODEL_FR, 2), (M.MODEL_DGP, 1)])
@pytest.mark.parametrize("N", [32, 48])
def test_fp64(N, model, n):
    def run(S):
        S.initialise()
        S.vcycle(0)
        levels = [S.get_level(l, a).tobytes() for l in range(1, S.levels()[2] + 1)
                  for a in (M.ARR_U, M.ARR_F, M.ARR_RES, M.ARR_RRES, M.ARR_RU, M.ARR_RHO)]
        S.fcycle(0)
        return levels, S.residual(0)
    _both(M.Config(N=N, model=model, fr_n=n, branch=1, box=2.0 * N, fr0=-1e-5), run)
