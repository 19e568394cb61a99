"""The force law within a few grid units of its edges, in every kernel that
evaluates it: a pair just past rmax adds nothing, and a pair within the
rounding of 1/dist of beta or rmax gets the same bits whichever kernel steps
the world."""
from __future__ import annotations

import numpy as np
import pytest

from parity_util import check_one_step

pytestmark = pytest.mark.gpu

# rmax on the 2^-32 grid (0.0155) and beta for which an FP32 1/|D| at rmax and at
# beta is far off, 7e-8 and 6e-8 of itself, and one Newton step 8e-15 and 5e-15 low
R = 66620907
BETA = 0.2821598
LATTICE = 16                                   # isolated pairs, 4 rmax apart


def _differences(edge):
    """Grid differences (dx, dy) whose squared length is so near an edge of the
    law that 1/|D| cannot tell the side: past rmax, up to it, around beta."""
    target = R * R if edge != "beta" else int((BETA * R) ** 2)
    dx = np.arange(1, 18_000_000, dtype=np.int64)
    dy = np.sqrt((target - dx * dx).astype(np.float64)).astype(np.int64)
    lo, hi = {"past rmax": (1, 64), "up to rmax": (-64, 0), "beta": (-3, 3)}[edge]
    got = []
    for c in (0, 1):
        k = dx * dx + (dy + c) ** 2 - target
        near = (k >= lo) & (k <= hi)
        got.append(np.stack([dx[near], dy[near] + c], 1))
    return np.concatenate(got)


def _world(edge, dim, wrap):
    from particle_life.worlds import World

    d = _differences(edge)
    assert len(d) >= 4
    rng = np.random.default_rng(900 + dim)
    m = LATTICE * LATTICE
    d = d[rng.integers(0, len(d), m)] * rng.choice([-1, 1], (m, 2))
    swap = rng.random(m) < 0.5
    d[swap] = d[swap][:, ::-1]
    at = np.stack(np.meshgrid(np.arange(LATTICE), np.arange(LATTICE)), -1).reshape(-1, 2)
    p = np.full((m, 3), 1 << 31, np.int64)
    p[:, :2] = (at * 4 + 2) * R + rng.integers(0, R // 4, (m, 2))
    if dim == 2:
        p[:, 2] = 0
    q = p.copy()
    q[:, :2] += d
    pos = np.concatenate([p, q]).astype(np.float64) * 2.0 ** -32
    n = 2 * m
    return World(pos=pos, vel=np.zeros((n, 3)), types=rng.integers(0, 3, n).astype(np.int32),
                 matrix=np.array([[1.0, -0.7, 40.0], [0.3, 1.0, -1.0], [-1e6, 0.5, 1.0]]), rmax=R * 2.0 ** -32,
                 friction=0.8, dt=0.01, beta=BETA, dim=dim, wrap=wrap)


@pytest.mark.parametrize("edge", ["past rmax", "up to rmax", "beta"])
@pytest.mark.parametrize("dim, wrap", [(2, True), (2, False), (3, True)])
def test_edges_of_the_law(edge, dim, wrap):
    from particle_life import Engine

    print(f"\n[law edges] {edge} dim={dim} wrap={wrap}", flush=True)
    w = _world(edge, dim, wrap)
    states = []
    # staged, windowed, one thread per home, one launch (2D: its grid fits)
    modes = [dict(sparse_worlds=1, small_step=1), dict(sparse_worlds=1, windowed_only=True, small_step=1),
             dict(sparse_worlds=2, small_step=1)] + ([dict(small_step=2)] if dim == 2 else [])
    for mode in modes:
        with Engine(0) as e:
            e.set_tuning(**mode)
            e.load_world(w)
            e.step(1)
            plain = e.state()
            e.load_world(w)
            check_one_step(e, w)
            states.append((plain, e.state(), e.pair_count(), e.accelerations()))
    want = 0 if edge == "past rmax" else w.n
    for plain, debug, pairs, acc in states:
        assert pairs == want
        if edge == "past rmax":
            assert not plain["vel"].any() and not acc.any()
        for k in ("pos", "vel", "ids"):
            np.testing.assert_array_equal(plain[k], states[0][0][k])
            np.testing.assert_array_equal(debug[k], states[0][0][k])
        np.testing.assert_array_equal(acc, states[0][3])
