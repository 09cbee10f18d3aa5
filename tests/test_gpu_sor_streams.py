"""The one-per-tile pressure solve beside other streams' kernels: several tanks on their
own streams, stepped without waiting, each with more fluid tiles than are resident
whatever else runs (and one with fewer), and a batch of as many tiles with a tank beside
it, give the bits each gives alone, and no wait times out (sync would say so)."""
import numpy as np
import pytest

from splashtank_amd import capi
from splashtank_amd.capi import FlipBatchC, FlipSimC

pytestmark = pytest.mark.gpu


def _layer(tx, tz, seed):
    """A box one tile high, wet all over: tx x tz fluid tiles."""
    h = 0.02
    cells = (8 * tx - 2, 6, 8 * tz - 2)
    size = [c * h for c in cells]
    rng = np.random.default_rng(seed)
    x, y, z = np.meshgrid(np.arange(cells[0]), np.arange(2), np.arange(cells[2]), indexing="ij")
    pos = np.zeros((x.size, 4), np.float32)
    pos[:, :3] = np.stack([x.ravel() + 0.5, y.ravel() + 0.5, z.ravel() + 0.5], 1) * h - np.array([size[0] / 2, 0, size[2] / 2])
    pos[:, :3] += rng.uniform(-0.4, 0.4, (len(pos), 3)) * h
    vel = np.zeros_like(pos)
    vel[:, :3] = rng.uniform(-1, 1, (len(pos), 3))
    s = FlipSimC(capi.make_opts(h / 2, size, max_n=len(pos)))
    s.upload(pos, vel)
    return s


SHAPES = [(36, 36), (40, 40), (30, 30), (42, 36)]
PRM = dict(dt=1.0 / 240, iters=12, omega=1.7)


def _state(s):
    s.sync()
    return [s.dump(f).view(np.uint32).copy() for f in ("pres", "pos", "vel")]


@pytest.mark.parametrize("batched", [False, True])
def test_tanks_on_streams_of_their_own(batched):
    prm = capi.make_params(**PRM)
    alone = []
    for k, (tx, tz) in enumerate(SHAPES):
        s = _layer(tx, tz, k)
        for _ in range(6):
            s.step(prm)
            s.sync()
        alone.append(_state(s))
        s.close()
    tanks = [_layer(tx, tz, k) for k, (tx, tz) in enumerate(SHAPES)]
    batch = FlipBatchC([tanks[2]]) if batched else None
    for _ in range(6):
        for k, s in enumerate(tanks):
            if batch and k == 2:
                batch.step(prm)
            else:
                s.step(prm)
    if batch:
        batch.sync()
        batch.close()
    for s, want in zip(tanks, alone):
        for a, b in zip(_state(s), want):
            assert np.array_equal(a, b)
        s.close()
