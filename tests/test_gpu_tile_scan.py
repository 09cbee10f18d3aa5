"""The tile bookkeeping scans blocks of 1024 tiles (and 1025 bins for 1024 tiles):
tile counts around one and two blocks, with tiles freed and allocated in several
blocks and, for one, a pool too small for them.  Tile map, tiles, control words
and particles match the oracle after every substep."""
import numpy as np
import pytest

from splashtank_amd import capi
from splashtank_amd.capi import FlipSimC
from oracle.oracle import Oracle
from tests.helpers import assert_f32_close, assert_int_equal

pytestmark = pytest.mark.gpu


# tiles per axis (cells = 8 t - 1 or less per axis), slots of the pool (0: every tile)
@pytest.mark.parametrize("tiles,slots", [((3, 11, 31), 0), ((4, 8, 32), 0), ((5, 5, 41), 0), ((2, 31, 33), 0), ((2, 23, 45), 40), ((1, 1, 3), 0)])
def test_tile_scan_blocks_match_oracle(tiles, slots):
    h = 0.05
    d = h / 2
    cells = [8 * t - 2 for t in tiles]
    size = [c * h for c in cells]
    assert [(c + 8) // 8 for c in cells] == list(tiles)
    rng = np.random.default_rng(sum(tiles))
    n = 4000
    lo, hi = np.array([-size[0] / 2, 0.0, -size[2] / 2]), np.array([size[0] / 2, size[1], size[2] / 2])
    # clumps spread over the whole tile range, moving fast enough to leave their tiles
    c = lo + rng.random((25, 3)) * (hi - lo)
    pos = np.zeros((n, 4), np.float32)
    pos[:, :3] = np.clip(c[rng.integers(0, 25, n)] + rng.normal(0, 0.08, (n, 3)), lo + 0.3 * d, hi - 0.3 * d)
    vel = np.zeros((n, 4), np.float32)
    vel[:, :3] = rng.uniform(-9, 9, (25, 3))[rng.integers(0, 25, n)]
    opts = capi.make_opts(d, size, max_n=n, slots=slots)
    prm = capi.make_params(dt=0.04, iters=4, omega=1.7)
    g, o = FlipSimC(opts), Oracle(opts)
    assert g.dims.ntiles == tiles[0] * tiles[1] * tiles[2]
    for s in (g, o):
        s.upload(pos, vel)
    for step in range(4):
        g.step(prm)
        o.step(prm)
        cg, co = g.ctl(), o.ctl()
        print(f"[tile scan] {tiles} slots {slots} step {step}: ctl {list(cg[:7])}", flush=True)
        assert_int_equal(cg[:6], co[:6], f"step {step}: ctl")
        for f in ("tmap", "tiles", "cnt", "ctype"):
            assert_int_equal(g.dump(f), o.dump(f), f"step {step}: {f}")
        for f in ("pos", "vel"):
            assert_f32_close(g.dump(f), o.dump(f), f"step {step}: {f}")
    assert not slots or cg[5] > 0, "the small pool ran out"
    g.close()
