"""A batch whose one-launch solve is capped (st_batch_sor_grid) at fewer workgroups
than its fluid tiles, though its particles at rest would fill fewer tiles than the
cap: every tank keeps the bits of a step alone.  (`full` below is what the launch
rule estimates: tiles filled at rest density, rounded down per tank.)"""
import numpy as np
import pytest

from splashtank_amd import capi, scenes
from splashtank_amd.capi import FlipBatchC, FlipSimC
from tests.helpers import assert_int_equal, opts_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap,count", [(2, 2), (4, 3), (8, 6)])
def test_capped_solve_matches_single_tanks(cap, count):
    # 16^3 tanks, 5,408 particles each: 1.3 full tiles, over two tiles and more
    tanks = [scenes.dam_break(d=1.0 / 32, seed=3 + k, frac=(0.4, 0.4, 1.0), iters=9 + k) for k in range(count)]
    prms = [capi.make_params(**sc.params) for sc in tanks]
    solo, bt = ([FlipSimC(opts_for(sc)) for sc in tanks] for _ in range(2))
    full = sum(sc.n // 4096 for sc in tanks)
    assert full + full // 5 <= cap
    for sims in (solo, bt):
        for s, sc in zip(sims, tanks):
            s.upload(sc.pos, sc.vel)
    batch = FlipBatchC(bt)
    batch.sor_grid(cap)
    try:
        for step in range(3):
            for a, p in zip(solo, prms):
                a.step(p)
                a.sync()
            batch.step(prms)
            batch.sync()
            tiles = sum(int(a.ctl()[4]) for a in solo)
            assert tiles > cap
            print(f"[batch cap] cap {cap}, {tiles} tiles in use, step {step}", flush=True)
            for a, b in zip(solo, bt):
                for f in ("pres", "pos", "vel"):
                    assert_int_equal(b.dump(f).view(np.uint32), a.dump(f).view(np.uint32), f"step {step} {f}")
            assert any(np.any(a.dump("pres") != 0) for a in solo)
    finally:
        batch.close()
    for s in solo + bt:
        s.close()
