"""Snapshots are copied piece by piece in one launch: particle counts whose arrays
end inside, at and just past a 16-byte access and a 32 KB piece come back whole,
and the substeps after a restore repeat bit for bit."""
import numpy as np
import pytest

from splashtank_amd import capi
from splashtank_amd.capi import FlipSimC, SnapshotC

pytestmark = pytest.mark.gpu

FIELDS = ["pos", "vel", "tmap", "ctype", "pres"]


@pytest.mark.parametrize("n", [1, 2, 3, 5, 2047, 2048, 2049, 8191, 8192, 8193, 20001])
def test_restore_gives_back_every_word(n):
    h = 1.0 / 24
    rng = np.random.default_rng(n)
    pos = np.zeros((n, 4), np.float32)
    pos[:, :3] = rng.uniform((-0.45, 0.05, -0.3), (0.45, 0.6, 0.3), (n, 3))
    vel = np.zeros((n, 4), np.float32)
    vel[:, :3] = rng.uniform(-2, 2, (n, 3))
    g = FlipSimC(capi.make_opts(h / 2, (1.0, 0.8, 0.7), max_n=n))
    g.upload(pos, vel)
    prm = capi.make_params(dt=1.0 / 120, iters=5, omega=1.7)
    g.step(prm)
    was = {f: g.dump(f) for f in FIELDS}
    snap = SnapshotC(g)
    g.step_n(prm, 3)
    after = {f: g.dump(f) for f in FIELDS}
    snap.restore()
    for f in FIELDS:
        assert np.array_equal(g.dump(f).view(np.uint32), was[f].view(np.uint32)), f"{f} after the restore"
    g.step_n(prm, 3)
    for f in FIELDS:
        assert np.array_equal(g.dump(f).view(np.uint32), after[f].view(np.uint32)), f"{f} of the substeps run again"
    snap.close()
    g.close()
