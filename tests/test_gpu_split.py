"""The split kernel (four lanes a home) at the sizes where it can go wrong:
clustered worlds that the planner sends to it, in 2D and 3D, periodic and
clamped, with a matrix in LDS and not, against the staged kernel bit for bit
and against the oracle; a batch of which only some worlds take it."""
from __future__ import annotations

import numpy as np
import pytest

from parity_util import check_one_step

pytestmark = pytest.mark.gpu


def _cluster(seed, n, dim, types, wrap, spread):
    from particle_life.worlds import World

    rng = np.random.default_rng(seed)
    pos = np.zeros((n, 3))
    k = n - n // 8                           # one tight cluster across the seam, the rest anywhere
    pos[:k, :dim] = (0.02 if wrap else 0.1) + spread * rng.normal(size=(k, dim))
    pos[k:, :dim] = rng.uniform(size=(n - k, dim))
    pos = pos - np.floor(pos) if wrap else np.clip(pos, 0.0, 1.0 - 2.0 ** -32)
    pos = np.floor(pos * 2.0 ** 32) * 2.0 ** -32
    return World(pos=pos, vel=np.zeros((n, 3)), types=rng.integers(0, types, n).astype(np.int32),
                 matrix=rng.uniform(-1, 1, (types, types)), rmax=0.06, friction=0.8, dt=1e-4, dim=dim, wrap=wrap)


CASES = [(2, True, 5, 3001), (2, False, 40, 3001), (3, True, 6, 5003), (3, False, 5, 5003), (2, True, 3, 2049)]


@pytest.mark.parametrize("dim,wrap,types,n", CASES)
def test_split_kernel(dim, wrap, types, n):
    from particle_life import Engine

    print(f"\n[split] case=dim {dim} wrap {wrap} types {types} n {n}", flush=True)
    w = _cluster(500 + n + types, n, dim, types, wrap, 0.012)
    got = []
    with Engine(0) as e:
        for windowed in (False, True):        # the planner's choice; k_force
            e.set_tuning(small_step=1, windowed_only=windowed)
            e.load_world(w)
            for _ in range(3):                # the second step on: planned from measured work
                e.step(1)
                e.sync()
            check_one_step(e, w)
            e.set_debug(False)
            e.step(2)
            got.append((e.state(), e.pair_count()))
    for k in ("pos", "vel", "types", "ids"):
        np.testing.assert_array_equal(got[0][0][k], got[1][0][k])
    assert got[0][1] == got[1][1]


def test_batch_of_split_and_staged_worlds():
    from particle_life import Batch, Engine, worlds

    print("\n[split] case=batch", flush=True)
    ws = [_cluster(601, 3000, 2, 4, True, 0.012), worlds.uniform_world(602, 9000, 4, rmax=0.02, dt=0.01),
          _cluster(603, 2500, 2, 6, False, 0.01), worlds.uniform_world(604, 4000, 4, rmax=0.01, dt=0.01)]
    with Batch(0) as b:
        b.set_tuning(small_step=1)
        ids = [b.add_world(w) for w in ws]
        for _ in range(4):
            b.step(1)
            b.sync()
        b.step(6)                             # graph replays of forked launches
        b.step(6)
        got = [b.state(i) for i in ids]
    for w, g in zip(ws, got):
        with Engine(0) as e:
            e.set_tuning(small_step=1, windowed_only=True)
            e.load_world(w)
            e.step(16)
            ref = e.state()
        for k in ("pos", "vel", "types", "ids"):
            np.testing.assert_array_equal(g[k], ref[k])
