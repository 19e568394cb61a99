"""The force kernels run where tests and planner mean them to: the split kernel
on the worlds of test_gpu_split.py, its global path and, beside the staged
kernel, its forked launches; a staged launch above 64 KB of LDS; windows that
halve until their mask words fit; the no-alloc step's literal path."""
from __future__ import annotations

import numpy as np
import pytest

from parity_util import check_one_step
from test_gpu_split import CASES, _cluster
from test_zz_no_alloc import _hip, _noalloc_step

pytestmark = pytest.mark.gpu


def _measured(e):
    """Two steps apart, so that the next is planned from measured work."""
    for _ in range(3):
        e.step(1)
        e.sync()


@pytest.mark.parametrize("dim,wrap,types,n", CASES)
def test_clustered_worlds_take_the_split_kernel(dim, wrap, types, n):
    from particle_life import Engine

    print(f"\n[kernels] split: dim {dim} wrap {wrap} types {types} n {n}", flush=True)
    w = _cluster(500 + n + types, n, dim, types, wrap, 0.012)
    with Engine(0) as e:
        for windowed, want in ((False, "split"), (True, "staged")):
            e.set_tuning(small_step=1, windowed_only=windowed)
            e.load_world(w)
            _measured(e)
            e.step(2)
            got = e.force_kernels()
            assert got[want] > 0 and sum(got.values()) == got[want]


def _rows_of_workgroups(w, homes):
    """Most grid rows that `homes` consecutive particles of the cell order lie in."""
    nx = int(1.0 / w.rmax)
    c = np.minimum((w.pos[:, :w.dim] / w.rmax).astype(np.int64), nx - 1)
    row = np.sort(c[:, 1] * nx + c[:, 0]) // nx
    return max(len(np.unique(row[k:k + homes])) for k in range(0, len(row), homes))


def test_split_kernel_global_path():
    """A cluster with so thin a rest that a workgroup of 64 homes spans more
    rows than are staged: bit for bit one thread per home's, and the oracle's."""
    from particle_life import Engine

    print("\n[kernels] split: global path", flush=True)
    w = _cluster(700, 3073, 2, 5, True, 0.012)
    rng = np.random.default_rng(701)
    k = w.n - w.n // 8
    keep = np.concatenate([np.arange(k), k + rng.choice(w.n - k, 60, replace=False)])
    w.pos, w.vel, w.types = w.pos[keep], w.vel[keep], w.types[keep]
    assert _rows_of_workgroups(w, 64) > 4
    states = []
    for mode, want in ((0, "split"), (2, "sparse")):
        with Engine(0) as e:
            e.set_tuning(small_step=1, sparse_worlds=mode)
            e.load_world(w)
            _measured(e)
            check_one_step(e, w)
            got = e.force_kernels()
            assert got[want] > 0 and sum(got.values()) == got[want]
            e.set_debug(False)
            e.step(2)
            states.append((e.state(), e.pair_count()))
    for key in ("pos", "vel", "types", "ids"):
        np.testing.assert_array_equal(states[0][0][key], states[1][0][key])
    assert states[0][1] == states[1][1]


def test_batch_takes_split_and_staged_kernels():
    from particle_life import Batch, worlds

    print("\n[kernels] batch", flush=True)
    ws = [_cluster(601, 3000, 2, 4, True, 0.012), worlds.uniform_world(602, 9000, 4, rmax=0.02, dt=0.01),
          _cluster(603, 2500, 2, 6, False, 0.01), worlds.uniform_world(604, 4000, 4, rmax=0.01, dt=0.01)]
    with Batch(0) as b:
        b.set_tuning(small_step=1)
        for w in ws:
            b.add_world(w)
        _measured(b)
        b.step(6)
        b.step(6)
        got = b.force_kernels()
    assert got["split"] > 0 and got["staged"] > 0


def test_staged_launch_above_64_kb():
    from particle_life import Engine, worlds

    print("\n[kernels] LDS", flush=True)
    w = worlds.uniform_world(403, 130_000, 6, rmax=0.04, dt=0.01, dim=3)
    with Engine(0) as e:
        e.set_tuning(sparse_worlds=1, small_step=1)
        e.load_world(w)
        e.step(1)
        assert e.tuning()["lds_bytes"] > 65536 and e.force_kernels()["staged"] > 0


def _full_cells_with_thin_neighbours():
    """Cells of 600 particles, each with one particle in every other row of its
    27 cells: a home's first 64 staged candidates are four runs of one and 60 of
    its own cell, 4 + 3 mask words."""
    from particle_life.worlds import World

    rng = np.random.default_rng(710)
    nx, rmax = 11, 1.0 / 11.2
    pos = []
    for at in [(2, 2, 2), (6, 2, 2), (2, 6, 6), (6, 6, 9), (9, 9, 5)]:
        pos.append((np.array(at) + rng.uniform(0.02, 0.98, (600, 3))) * rmax)
        rows = [(0, y, z) for y in (-1, 0, 1) for z in (-1, 0, 1) if (y, z) != (0, 0)]
        pos.append((np.array(at) + np.array(rows) + rng.uniform(0.2, 0.8, (8, 3))) * rmax)
    pos = np.floor(np.concatenate(pos) * 2.0 ** 32) * 2.0 ** -32
    n = len(pos)
    assert pos.max() < nx * rmax
    return World(pos=pos, vel=np.zeros((n, 3)), types=rng.integers(0, 5, n).astype(np.int32),
                 matrix=rng.uniform(-1, 1, (5, 5)), rmax=rmax, friction=0.8, dt=1e-3, dim=3)


@pytest.mark.parametrize("homes", [64, 128, 256])
def test_windows_that_halve(homes):
    """Four mask words a home where its first window needs seven: the window
    halves until its words fit."""
    from particle_life import Engine

    print(f"\n[kernels] halving windows: {homes} homes", flush=True)
    w = _full_cells_with_thin_neighbours()
    states = []
    for tuning in (dict(windowed_only=True, sparse_worlds=1, list_cap=1, block_homes=homes, small_step=1),
                   dict(sparse_worlds=2, small_step=1)):
        with Engine(0) as e:
            e.set_tuning(**tuning)
            e.load_world(w)
            check_one_step(e, w)
            e.set_debug(False)
            e.step(2)
            states.append((e.state(), e.pair_count()))
    for key in ("pos", "vel", "types", "ids"):
        np.testing.assert_array_equal(states[0][0][key], states[1][0][key])
    assert states[0][1] == states[1][1]


@pytest.mark.parametrize("bad", [np.inf, np.nan, -1e305])
def test_noalloc_step_with_a_matrix_that_is_not_finite(bad):
    from particle_life import Engine, worlds

    print(f"\n[kernels] no-alloc, entry {bad}", flush=True)
    w = worlds.uniform_world(720, 20_000, 5, rmax=0.02, dt=0.01)
    w.matrix[4, 0] = bad
    got = _noalloc_step(_hip(), w)
    with Engine(0) as e:
        e.set_tuning(sparse_worlds=2, small_step=1)
        e.load_world(w)
        e.step(1)
        ref, pairs = e.state(), e.pair_count()
    for key in ("pos", "vel", "types", "ids"):
        np.testing.assert_array_equal(got[key], ref[key])
    assert got["pairs"] == pairs > 0
    assert np.isfinite(got["vel"][got["types"] != 4]).all()
