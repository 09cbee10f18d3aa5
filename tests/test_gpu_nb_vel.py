"""The narrow band's kept velocity carried further than the two cells a tile's window
reaches, at the box's edges and in tiles whose neighbours have no storage: faces
within the window and out of it match the oracle."""
import numpy as np
import pytest

from splashtank_amd import capi, scenes
from splashtank_amd.capi import FlipSimC
from oracle.oracle import Oracle
from tests.helpers import assert_f32_close, assert_int_equal, opts_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("speed", [0.0, 3.0, 40.0])
def test_carried_velocity_matches_oracle(speed):
    sc = scenes.nb_pool(d=1.0 / 42, depth=0.55, drop=(0.1, 0.8, 0.0, 0.08))
    live = sc.pos[:, 1] > -1e5
    rng = np.random.default_rng(int(speed))
    sc.vel[live, :3] = rng.uniform(-speed, speed, (int(live.sum()), 3))
    opts = opts_for(sc)
    g, o = FlipSimC(opts), Oracle(opts)
    for s in (g, o):
        s.upload(sc.pos, sc.vel)
    for step in range(3):
        kw = dict(sc.params, dt=1.0 / 60, vmax=100.0, iters=8)
        if step == 0:
            kw.update(nb_init=1, nfill=len(sc.nb_fills) // 8, fills=list(sc.nb_fills))
        prm = capi.make_params(**kw)
        for s in (g, o):
            s.begin_step(prm)
        for st in range(capi.ST_STAGE_COUNT):
            for s in (g, o):
                s.stage(st)
            if st == capi.ST_STAGE_CLASSIFY:
                for f in ("accv", "accw"):
                    assert_int_equal(g.dump(f), o.dump(f), f"step {step}: {f}")
        for f in ("velg", "pos", "vel"):
            assert_f32_close(g.dump(f), o.dump(f), f"step {step}: {f}")
    if speed == 40.0:  # carried by more than the window's two cells
        assert np.abs(g.dump("velg")).max() * (1.0 / 60) * 21 > 3.0
    g.close()
