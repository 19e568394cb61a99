"""The staged force kernel's mask words (20 candidates each) and the planner's
choices around them, against the oracle and against one thread per home over
the literal stencil, bit for bit: stencil row runs around one and two words,
dense worlds that stream several windows, a layout above 64 KB of LDS, clamped
worlds whose saturating differences meet both walls."""
from __future__ import annotations

import numpy as np
import pytest

from parity_util import check_one_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim, wrap, n, rmax", [
    (2, True, 2_600, 0.05),       # 6.5 a cell: runs of about one word
    (2, False, 5_300, 0.05),      # 13 a cell: two words, and the walls
    (2, True, 40_000, 0.05),      # 100 a cell: several windows
    (2, False, 257, 0.3),         # three cells an axis, one home past a workgroup
    (3, True, 130_000, 0.04),     # 8.3 a cell: more than 64 KB of LDS
    (3, False, 20_011, 0.12),     # 39 a cell: several windows, and the walls
])
def test_words_and_windows(dim, wrap, n, rmax):
    from particle_life import Engine, worlds

    print(f"\n[words] dim={dim} wrap={wrap} n={n} rmax={rmax}", flush=True)
    w = worlds.uniform_world(400 + dim, n, 6, rmax=rmax, dt=0.01, dim=dim)
    w.wrap = wrap
    states = []
    for mode in (1, 2):                   # staged; one thread per home
        with Engine(0) as e:
            e.set_tuning(sparse_worlds=mode, small_step=1)
            e.load_world(w)
            if mode == 1:
                check_one_step(e, w)
                e.set_debug(False)
            else:
                e.step(1)
            e.step(3)
            states.append((e.state(), e.pair_count()))
    for k in ("pos", "vel", "ids"):
        np.testing.assert_array_equal(states[0][0][k], states[1][0][k])
    assert states[0][1] == states[1][1]
