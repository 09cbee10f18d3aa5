"""Binning through the workgroups' tables: particle counts around a workgroup and a
full table, bins in the order of a fill and at random over more tiles than a table
holds (runs that find no place in it), with dead particles among them.  The bins are
checked by what follows from them: the state after two substeps, in id order, against
the oracle."""
import numpy as np
import pytest

from splashtank_amd import capi
from splashtank_amd.capi import FlipSimC
from oracle.oracle import Oracle
from tests.helpers import assert_f32_close, assert_int_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["rows", "random"])
@pytest.mark.parametrize("n", [1, 63, 257, 2047, 2049, 150001])
def test_bins_match_oracle(n, order):
    d = 0.02
    size = (3.8, 0.6, 3.8)  # 12 x 2 x 12 tiles of 8 cells of 0.04
    rng = np.random.default_rng(n)
    pos = np.zeros((n, 4), np.float32)
    pos[:, :3] = rng.uniform((-1.89, 0.01, -1.89), (1.89, 0.59, 1.89), (n, 3))
    if order == "rows":
        pos = pos[np.lexsort((pos[:, 0], np.floor(pos[:, 1] / 0.04), np.floor(pos[:, 2] / 0.04)))]
    pos[rng.random(n) < 0.1, 1] = -1.0e6
    vel = np.zeros_like(pos)
    vel[:, :3] = rng.uniform(-1, 1, (n, 3)) * (pos[:, 1:2] > -1)
    opts = capi.make_opts(d, size, max_n=n)
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


def test_more_bins_than_a_table_holds():
    """2048 particles in a row, each in a tile of its own, next to a full tile."""
    d = 0.02
    size = (7.6, 0.28, 27.0)  # 24 x 1 x 85 tiles: 2040 of them
    x, z = np.meshgrid(np.arange(24) * 0.32 - 3.65, np.arange(84) * 0.32 - 13.35)
    lone = np.zeros((x.size, 4), np.float32)
    lone[:, 0], lone[:, 1], lone[:, 2] = x.ravel(), 0.1, z.ravel()
    rng = np.random.default_rng(1)
    many = np.zeros((3000, 4), np.float32)
    many[:, :3] = rng.uniform((-0.3, 0.0, -0.3), (0.3, 0.27, 0.3), (3000, 3))
    pos = np.concatenate([lone, many])
    vel = np.zeros_like(pos)
    opts = capi.make_opts(d, size, max_n=len(pos))
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
