"""The force kernel's phase-A screen (screen_hi, WorldDev::sbias) restated in
numpy: it must keep every pair with |D| <= rmax, whatever the low halves of the
coordinates and however close to rmax, and drop most of the rest."""
from __future__ import annotations

import numpy as np
import pytest


def _kept(p, q, rmax, dim):
    bias = -int(min((rmax * 65536.0 * (1.0 + 2.0 ** -20) + np.sqrt(dim + 3.0)) ** 2 + 2.0, 2147483646.0))
    hi = lambda a: ((a[:, 0] >> np.uint32(16)) | (a[:, 1] & np.uint32(0xFFFF0000)))      # noqa: E731
    d = hi(q) - hi(p)                                                                    # one 32-bit subtract
    dx = (d & np.uint32(0xFFFF)).astype(np.uint16).view(np.int16).astype(np.int64)
    dy = (d >> np.uint32(16)).astype(np.uint16).view(np.int16).astype(np.int64)
    s = dx * dx + dy * dy + bias
    if dim == 3:
        dz = ((q[:, 2] - p[:, 2]) >> np.uint32(16)).astype(np.uint16).view(np.int16).astype(np.int64)
        s += dz * dz
    return np.clip(s, -2 ** 31, 2 ** 31 - 1) < 0


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("rmax", [0.0005, 0.005, 0.01, 0.0416, 1.0 / 3.0])
def test_screen_keeps_every_pair_in_range(rmax, dim):
    rng = np.random.default_rng(int(1e6 * rmax) + dim)
    n = 200_000
    p = rng.integers(0, 2 ** 32, (n, 3), dtype=np.uint32)
    u = rng.normal(size=(n, 3))
    u[:, dim:] = 0.0
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    u[: n // 4] = np.round(u[: n // 4])                   # along the axes too
    for scale, keep in ((1.0, True), (rng.uniform(0.0, 1.0, (n, 1)), True), (2.0, False)):
        d = np.trunc(u * rmax * scale * 2.0 ** 32 * (1.0 - 2.0 ** -30)).astype(np.int64)
        q = ((p.astype(np.int64) + d) % (1 << 32)).astype(np.uint32)
        inside = (d.astype(np.float64) ** 2).sum(axis=1) <= (rmax * 2.0 ** 32) ** 2
        kept = _kept(p, q, rmax, dim)
        assert kept[inside].all()
        if not keep and 0.005 <= rmax < 0.25:             # twice rmax stays within half the box
            assert kept[~inside].mean() < 0.01
