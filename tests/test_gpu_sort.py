"""The counting sort of the multi-launch path (k_bin, k_place, k_rank) at the
sizes where it can go wrong: cells that hold one less, exactly and one more
than a multiple of the sixteen indices k_rank reads at a time, arrivals that
cross waves, in random and in sorted input order."""
from __future__ import annotations

import numpy as np
import pytest

from parity_util import check_one_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
def test_cell_occupancies(dim):
    from particle_life import Engine
    from particle_life.worlds import World

    print(f"\n[sort] case=occupancies dim={dim}", flush=True)
    rng = np.random.default_rng(40 + dim)
    nx = 10
    counts = [1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 129, 300]
    cells = rng.permutation(nx ** dim)[: len(counts)]
    pos = []
    for c, k in zip(cells, counts):
        corner = np.array([c % nx, c // nx % nx, c // (nx * nx)])
        p = np.zeros((k, 3))
        p[:, :dim] = (corner[:dim] + rng.uniform(0.05, 0.95, (k, dim))) / nx
        pos.append(p)
    pos = np.floor(np.concatenate(pos) * 2.0 ** 32) * 2.0 ** -32
    n = len(pos)
    pos = pos[rng.permutation(n)]
    w = World(pos=pos, vel=np.zeros((n, 3)), types=rng.integers(0, 5, n).astype(np.int32),
              matrix=rng.uniform(-1, 1, (5, 5)), rmax=0.1, friction=0.8, dt=0.001, dim=dim)
    with Engine(0) as e:
        e.set_tuning(small_step=1)
        e.load_world(w)
        for _ in range(3):                    # random input order, then the last step's
            check_one_step(e, w)
