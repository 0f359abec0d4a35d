"""The deposit's tiles (32 x 16 x 8 cells) and run binning at their edges,
against the numpy restatement in oracle/pm.py."""
import numpy as np
import pytest

import mgsolve as M
import pm as P


def _cfg(N):
    return M.Config(N=N, model=M.MODEL_FR, fr_n=1, box=2.0 * N, fr0=-1e-5, precision=M.PREC_FP64)


# one partial tile; a last tile two cells wide in x and y; whole tiles; a
# weight of 2^11 and more (the 64-bit conversion); more bins in a block of
# unordered particles than its table has slots; a single particle
@pytest.mark.gpu
@pytest.mark.parametrize("N,n,edge", [(8, 4001, True), (34, 30007, True), (64, 50000, False), (64, 100, True),
                                      (192, 40000, False), (16, 1, False)])
def test_deposit_at_tile_edges(N, n, edge):
    rng = np.random.default_rng(N + n)
    pos = [rng.uniform(1.0, N + 1.0, n).astype(np.float32) for _ in range(3)]
    last = np.nextafter(np.float32(N + 1), np.float32(0))
    if edge:  # a third of the coordinates on or beside tile faces and the wrap
        for a, t in zip(pos, (32, 16, 8)):
            faces = np.arange(0, N + 1, t)
            v = rng.choice(faces, n // 3) + rng.choice([0.5, 1.0, 1.5, 0.99999994], n // 3)
            a[:n // 3] = np.clip(v, 1.0, last)
    pos = [np.clip(a, np.float32(1.0), last) for a in pos]
    print(f"[pm tiles] N={N} np={n}", flush=True)
    with M.Solver(_cfg(N)) as S:
        S.set_particles(*pos)
        S.cic_deposit()
        d = S.get_density(np.float64)
        perm = rng.permutation(n)
        S.set_particles(*[a[perm] for a in pos])
        S.cic_deposit()
        d2 = S.get_density(np.float64)
    ref = P.cic_deposit(*pos, N)
    # contributions per cell: each is rounded to a multiple of 2^-40, and the
    # oracle's FP64 sum rounds once per addition
    cnt = np.zeros((N, N, N))
    idx = [a.astype(np.int64) - 1 for a in pos]
    for o in range(8):
        i, j, k = ((v + ((o >> b) & 1)) % N for b, v in enumerate(idx))
        np.add.at(cnt, (k, j, i), 1.0)
    tol = cnt.max() * (2.0 ** -41 + 2.0 ** -52 * (ref.max() + 2.0)) + 2.0 ** -52 * (ref.max() + 2.0)
    assert np.max(np.abs(d - ref)) <= tol, (np.max(np.abs(d - ref)), tol)
    assert np.array_equal(d, d2)


# every row of the potential's block wraps (N = 4); an odd particle count;
# cells 1, N-1 and N in x, whose rows are gathered value by value
@pytest.mark.gpu
@pytest.mark.parametrize("N,n", [(4, 777), (6, 64), (34, 20001)])
def test_move_rows_at_the_wrap(N, n):
    rng = np.random.default_rng(N)
    pos = [rng.uniform(1.0, N + 1.0, n).astype(np.float32) for _ in range(3)]
    last = np.nextafter(np.float32(N + 1), np.float32(0))
    pos = [np.clip(a, np.float32(1.0), last) for a in pos]
    vel = [rng.normal(0.0, 0.3, n).astype(np.float32) for _ in range(3)]
    phi = rng.standard_normal((N, N, N)).astype(np.float32)
    print(f"[pm move] N={N} np={n}", flush=True)
    with M.Solver(_cfg(N)) as S:
        S.set_potential(phi)
        S.set_particles(*pos, *vel)
        S.move(-0.07, 0.9)
        got = S.get_particles()
    ref = P.move(phi.astype(np.float64), *pos, *vel, -0.07, 0.9)
    for a, b, name in zip(got, ref[:6], ("x", "y", "z", "vx", "vy", "vz")):
        assert np.array_equal(a, b), (name, int(np.sum(a != b)))
