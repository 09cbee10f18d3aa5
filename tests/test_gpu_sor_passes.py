"""The pressure solve as stream launches of two iterations each (few tiles) or one
each (many): iteration counts around the pairs match the oracle, eager and replayed
from a graph, alone and in a batch with unequal counts, and tanks on both sides of
the line give the bits of the one-launch solve."""
import numpy as np
import pytest

from splashtank_amd import capi, scenes
from splashtank_amd.capi import FlipBatchC, FlipSimC
from oracle.oracle import Oracle
from tests.helpers import assert_f32_close

pytestmark = pytest.mark.gpu


def _tank(seed):
    d = 1.0 / 60
    size = (1.0, 0.7, 0.6)
    rng = np.random.default_rng(seed)
    p1, _ = scenes.fill_box(d, -0.5, 0.5, 0.0, 0.15, -0.3, 0.3, rng)
    p2, _ = scenes.fill_sphere(d, 0.2, 0.45, -0.1, 0.1, rng)
    pos = np.concatenate([p1, p2])
    vel = np.zeros_like(pos)
    vel[:, :3] = rng.uniform(-1, 1, (len(pos), 3))
    return capi.make_opts(d, size, max_n=len(pos)), pos, vel


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("iters", [1, 2, 3, 4, 5, 6, 7, 8])
def test_iteration_counts_match_oracle(iters, graph):
    opts, pos, vel = _tank(iters)
    prm = capi.make_params(dt=1.0 / 240, iters=iters, omega=1.7, sor_mode=0 if graph else 1)
    g, o = FlipSimC(opts), Oracle(opts)
    for s in (g, o):
        s.upload(pos, vel)
    for _ in range(3):
        o.step(prm)
        if not graph:
            g.step(prm)
    if graph:
        g.step_n(prm, 3, graph=True)
    assert g.sor_path() == 0
    for f in ("pres", "pos", "vel"):
        assert_f32_close(g.dump(f), o.dump(f), f)
    g.close()


@pytest.mark.parametrize("counts", [(3, 4), (6, 1), (2, 7)])
def test_batch_of_unequal_counts(counts):
    prm = [capi.make_params(dt=1.0 / 240, iters=k, omega=1.7, sor_mode=1) for k in counts]
    tanks, alone = [], []
    for t, k in enumerate(counts):
        opts, pos, vel = _tank(20 + t)
        for to in (tanks, alone):
            s = FlipSimC(opts)
            s.upload(pos, vel)
            to.append(s)
    b = FlipBatchC(tanks)
    b.step_n(prm, 3, graph=True)
    for s, p in zip(alone, prm):
        for _ in range(3):
            s.step(p)
    for s, a in zip(tanks, alone):
        for f in ("pres", "pos", "vel"):
            assert np.array_equal(s.dump(f).view(np.uint32), a.dump(f).view(np.uint32)), f
    b.close()
    for s in tanks + alone:
        s.close()


# particles of 690 and 720 full tiles, on either side of the line
@pytest.mark.parametrize("tiles", [690, 720])
def test_both_sides_of_the_line(tiles):
    h = 0.01
    d = h / 2
    nx, ny, nz = 96, 48, 80
    size = (nx * h, ny * h, nz * h)
    rng = np.random.default_rng(tiles)
    n = tiles * 512 * 8
    pos = np.zeros((n, 4), np.float32)
    vel = np.zeros_like(pos)
    top = n / 8.0 / (nx * nz) * h
    pos[:, :3] = rng.uniform((-size[0] / 2, 0, -size[2] / 2), (size[0] / 2, top, size[2] / 2), (n, 3))
    vel[:, :3] = rng.uniform(-1, 1, (n, 3))
    out = []
    for mode in (0, 1):
        g = FlipSimC(capi.make_opts(d, size, max_n=n))
        g.upload(pos, vel)
        g.step(capi.make_params(dt=1.0 / 400, iters=7, omega=1.7, sor_mode=mode))
        assert g.sor_path() == (1 if mode == 0 else 0)
        out.append((g.dump("pres"), g.dump("vel")))
        g.close()
    for a, b, f in zip(out[0], out[1], ("pres", "vel")):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), f
    assert np.any(out[0][0] != 0)
