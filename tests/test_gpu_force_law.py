"""The staged kernels' form of the force law: squared distances by FMA where
they are exact (rmax up to 2^-6) and not above, against the oracle on both
sides of that line; matrices with entries that are not finite step like the
literal stencil's."""
from __future__ import annotations

import numpy as np
import pytest

from parity_util import check_one_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("rmax", [2.0 ** -6, 2.0 ** -6 * (1 + 2.0 ** -20)])
def test_exact_squares_boundary(dim, rmax):
    from particle_life import Engine, worlds

    print(f"\n[law] case=exact_squares dim={dim} rmax={rmax!r}", flush=True)
    w = worlds.uniform_world(300 + dim, 40_000, 5, rmax=rmax, dt=0.01, dim=dim)
    with Engine(0) as e:
        e.set_tuning(sparse_worlds=1, small_step=1)
        e.load_world(w)
        for _ in range(2):
            check_one_step(e, w)


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan, 1e305])
def test_matrix_entries_that_are_not_finite(bad):
    from particle_life import Engine, worlds

    print(f"\n[law] case=not_finite {bad}", flush=True)
    w = worlds.uniform_world(310, 20_000, 5, rmax=0.02, dt=0.01)
    w.matrix[1, 3] = bad
    got = []
    with Engine(0) as e:
        for mode in (1, 2):                   # staged kernel, one thread per home over the literal stencil
            e.set_tuning(sparse_worlds=mode, small_step=1)
            e.load_world(w)
            e.step(1)
            got.append((e.state(), e.pair_count()))
    for k in ("pos", "vel", "ids"):
        np.testing.assert_array_equal(got[0][0][k], got[1][0][k])
    assert got[0][1] == got[1][1]
    fine = ~(w.types == 1)                    # only homes of type 1 meet the entry
    by_id = np.empty_like(got[0][0]["vel"])
    by_id[got[0][0]["ids"]] = got[0][0]["vel"]
    assert np.isfinite(by_id[fine]).all()
