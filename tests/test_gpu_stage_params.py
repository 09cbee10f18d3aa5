"""Stages of a substep taken one by one, its parameters given anew between them
(st_begin_step twice): g2p goes by those in force when it runs, as the oracle does."""
import numpy as np
import pytest

from splashtank_amd import capi, scenes
from splashtank_amd.capi import FlipSimC
from oracle.oracle import Oracle
from tests.helpers import assert_f32_close, opts_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", [dict(foam_tau=0.05, drag=0.0), dict(only_tiles=1)])
def test_g2p_takes_the_parameters_in_force(first):
    sc = scenes.dam_break(d=1.0 / 32, iters=6)
    base = dict(sc.params, foam_tau=0.8, drag=0.6, wind=(2.0, 0.0, 1.0))
    prm, other = capi.make_params(**base), capi.make_params(**dict(base, **first))
    rng = np.random.default_rng(3)
    vel = sc.vel.copy()
    vel[:, :3] = rng.uniform(-2, 2, (sc.n, 3))
    vel[:, 3] = rng.uniform(0, 1, sc.n)  # foam
    opts = opts_for(sc)
    g, o = FlipSimC(opts), Oracle(opts)
    for s in (g, o):
        s.upload(sc.pos, vel)
        for _ in range(2):
            s.begin_step(other)
            s.stages(capi.ST_STAGE_BLOCKS)
            s.begin_step(prm)
            for k in range(capi.ST_STAGE_CLEAR, capi.ST_STAGE_COUNT):
                s.stage(k)
    for f in ("pos", "vel"):
        assert_f32_close(g.dump(f), o.dump(f), f)
    g.close()
