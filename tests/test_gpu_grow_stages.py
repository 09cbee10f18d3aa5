"""The pool grown between two stages of a substep: the rest of that substep and the
next one give the bits of a tank whose pool did not grow."""
import numpy as np
import pytest

from splashtank_amd import capi, scenes
from splashtank_amd.capi import FlipSimC
from tests.helpers import assert_int_equal, opts_for, set_colliders_at, upload_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("extra", [dict(), dict(sor_mode=1), dict(extrap_layers=2), dict(nb_on=1, nb_band=2.0)])
@pytest.mark.parametrize("after", [capi.ST_STAGE_BLOCKS, capi.ST_STAGE_P2G, capi.ST_STAGE_CLASSIFY, capi.ST_STAGE_DIVERGENCE, capi.ST_STAGE_PRESSURE,
                                   capi.ST_STAGE_G2P])
def test_grown_between_stages(after, extra):
    sc = scenes.sparse_splash(d=1.0 / 64, iters=6)
    tanks = [FlipSimC(opts_for(sc, slots=110)) for _ in range(2)]  # of 125 tiles and the spare slot
    prm = capi.make_params(**dict(sc.params, **extra))
    print(f"[grow] after stage {after}, {extra}", flush=True)
    for k, g in enumerate(tanks):
        upload_scene(g, sc)
        g.step(prm)
        set_colliders_at(g, sc, sc.params["dt"])
        g.begin_step(prm)
        for s in range(capi.ST_STAGE_COUNT):
            g.stage(s)
            if k and s == after:
                assert int(g.ctl()[5]) == 0
                g.grow(126)
        g.step(prm)
        g.sync()
    a, b = tanks
    assert b.dims.scap == 126 and a.dims.scap == 110
    for f in ("pos", "vel", "pres"):
        assert_int_equal(b.dump(f).view(np.uint32), a.dump(f).view(np.uint32), f)
    for g in tanks:
        g.close()
