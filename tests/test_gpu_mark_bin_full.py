"""Binning through the workgroups' tables where they are full: 2048 particles a
workgroup (its groups of 256 taken four apart, a last set of fewer workgroups), in the
order of rows, and at random over more tiles than a table has places, so that runs are
counted and marked in memory. The state after two substeps against the oracle."""
import numpy as np
import pytest

from splashtank_amd import capi
from splashtank_amd.capi import FlipSimC
from oracle.oracle import Oracle
from tests.helpers import assert_f32_close, assert_int_equal

pytestmark = pytest.mark.gpu

PLACES = 512  # of a table
N = 1_200_001  # 586 workgroups of 8 groups of 256


@pytest.mark.parametrize("order", ["rows", "random"])
def test_full_tables_match_oracle(order):
    d, h = 0.02, 0.04
    size = (7.6, 0.28, 27.0)  # 24 x 1 x 85 tiles of 8 cells
    rng = np.random.default_rng(5)
    lo = np.array([-3.79, 0.01, -13.49])
    pos = np.zeros((N, 4), np.float32)
    pos[:, :3] = rng.uniform(lo, (3.79, 0.27, 13.49), (N, 3))
    if order == "rows":
        pos = pos[np.lexsort((pos[:, 0], np.floor(pos[:, 1] / h), np.floor(pos[:, 2] / h)))]
    pos[rng.random(N) < 0.1, 1] = -1.0e6
    vel = np.zeros_like(pos)
    vel[:, :3] = rng.uniform(-1, 1, (N, 3)) * (pos[:, 1:2] > -1)
    # the tiles of one workgroup's particles
    first = pos[(np.arange(8)[:, None] * 1024 + np.arange(256)).ravel()]
    first = first[first[:, 1] > -1]
    cell = np.floor((first[:, [0, 2]] + (size[0] / 2, size[2] / 2)) / h).astype(int)
    tiles = len(np.unique(cell[:, 0] // 8 + 24 * (cell[:, 1] // 8)))
    assert tiles > PLACES if order == "random" else tiles < PLACES // 2, tiles
    opts = capi.make_opts(d, size, max_n=N)
    prm = capi.make_params(dt=1.0 / 240, iters=3, omega=1.5)
    g, o = FlipSimC(opts), Oracle(opts)
    for s in (g, o):
        s.upload(pos, vel)
        for _ in range(2):
            s.step(prm)
    assert_int_equal(g.dump("cnt"), o.dump("cnt"), "cnt")
    for f in ("pos", "vel"):
        assert_f32_close(g.dump(f), o.dump(f), f)
    g.close()
