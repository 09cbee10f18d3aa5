"""The pressure solve with a workgroup per tile (two iterations per exchange).
Iteration counts around an exchange, on a tank with a pool, a collider, lone
drops and a box that is no multiple of the tile, match the oracle; layers of
tiles on each side of its limits (workgroups at once, tiles in use it can
number) give the bits of one launch per iteration."""
import numpy as np
import pytest

from splashtank_amd import capi, scenes
from splashtank_amd.capi import FlipSimC
from oracle.oracle import Oracle
from tests.helpers import assert_f32_close, assert_int_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("iters", [1, 2, 3, 4, 5, 9])
def test_iteration_counts_match_oracle(iters):
    d = 1.0 / 70
    size = (1.0, 0.7, 0.8)
    rng = np.random.default_rng(iters)
    p1, v1 = scenes.fill_box(d, -0.5, 0.5, 0.0, 0.2, -0.4, 0.4, rng)
    p2, v2 = scenes.fill_sphere(d, 0.2, 0.45, -0.1, 0.1, rng)
    p3 = np.zeros((40, 4), np.float32)
    p3[:, :3] = rng.uniform((-0.49, 0.3, -0.39), (0.49, 0.69, 0.39), (40, 3))
    pos = np.concatenate([p1, p2, p3])
    vel = np.zeros_like(pos)
    vel[:, :3] = rng.uniform(-1, 1, (len(pos), 3))
    h = 2 * d
    dims, lo, data = scenes.box_sdf((0.1, 0.08, 0.12), h, 4 * h)
    rec = scenes.collider_record(0, dims, lo, h, (-0.2, 0.15, 0.05), vel=(0.3, 0.0, 0.0))
    opts = capi.make_opts(d, size, max_n=len(pos))
    prm = capi.make_params(dt=1.0 / 240, iters=iters, omega=1.7)
    g, o = FlipSimC(opts), Oracle(opts)
    for s in (g, o):
        s.upload(pos, vel)
        s.set_colliders(rec, data, 1)
        for _ in range(3):
            s.step(prm)
    assert g.sor_path() == 1
    assert_int_equal(g.dump("ctype"), o.dump("ctype"), "ctype")
    for f in ("pres", "pos", "vel"):
        assert_f32_close(g.dump(f), o.dump(f), f)
    g.close()


# tiles along x, y and z, all of the lowest layer wet: below the workgroups resident at
# once (7 per CU), above them, above the tiles in use that can be numbered (2048), and
# more tiles than workgroups in the box but few of them wet
@pytest.mark.parametrize("tiles", [(32, 1, 40), (42, 1, 43), (46, 1, 46), (30, 2, 40)])
def test_limits_give_the_bits_of_single_iterations(tiles):
    h = 0.02
    d = h / 2
    cells = [8 * t - 2 for t in tiles]
    size = [c * h for c in cells]
    rng = np.random.default_rng(tiles[0])
    x, y, z = np.meshgrid(np.arange(cells[0]), np.arange(2), np.arange(cells[2]), indexing="ij")
    pos = np.zeros((x.size, 4), np.float32)
    pos[:, :3] = np.stack([x.ravel() + 0.5, y.ravel() + 0.5, z.ravel() + 0.5], 1) * h - np.array([size[0] / 2, 0, size[2] / 2])
    pos[:, :3] += rng.uniform(-0.4, 0.4, (len(pos), 3)) * h
    vel = np.zeros_like(pos)
    vel[:, :3] = rng.uniform(-1, 1, (len(pos), 3))
    out = []
    for mode in (0, 1):
        g = FlipSimC(capi.make_opts(d, size, max_n=len(pos)))
        assert g.dims.ntiles == tiles[0] * tiles[1] * tiles[2]
        g.upload(pos, vel)
        prm = capi.make_params(dt=1.0 / 240, iters=7, omega=1.7, sor_mode=mode)
        for _ in range(2):
            g.step(prm)
        g.sync()
        assert g.sor_path() == (1 if mode == 0 else 0)
        out.append((g.dump("pres"), g.dump("pos"), g.dump("vel")))
        print(f"[tile sor] {tiles} mode {mode}: {int(g.ctl()[4])} tiles in use", flush=True)
        g.close()
    for a, b, f in zip(out[0], out[1], ("pres", "pos", "vel")):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), f
    assert np.any(out[0][0] != 0)
