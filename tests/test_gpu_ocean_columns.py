"""The ocean's waves worked out per column of a half tile (face velocities, the
starting fill) and particles handed out one by one when the band is refilled: with
no wave, one, a few and the most the parameter block holds, in a box whose sides
are no multiple of the tile, the substeps match the oracle."""
import numpy as np
import pytest

from splashtank_amd import capi, scenes
from splashtank_amd.capi import FlipSimC
from oracle.oracle import Oracle
from tests.helpers import assert_f32_close, assert_int_equal, opts_for, set_colliders_at, upload_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nwave", [0, 1, 7, 32])
def test_wave_counts_match_oracle(nwave):
    sc = scenes.stress(d=1.0 / 54, iters=10, dt=1.0 / 120)  # 27^3 cells
    w = np.concatenate([sc.params["waves"], 0.5 * sc.params["waves"][:8]]).astype(np.float32)[:nwave]
    sc.params["waves"] = w
    opts = opts_for(sc)
    g, o = FlipSimC(opts), Oracle(opts)
    for s in (g, o):
        upload_scene(s, sc)
        s.set_spray_cap(sc.spray_cap)
    t = 0.0
    for step in range(4):
        t += sc.params["dt"]
        kw = sc.params_at(t)
        if step == 0:
            kw.update(nb_init=1, nfill=len(sc.nb_fills) // 8, fills=list(sc.nb_fills))
        prm = capi.make_params(**kw)
        assert prm.nwave == nwave
        for s in (g, o):
            set_colliders_at(s, sc, t)
            s.step(prm)
        assert_int_equal(g.dump("ctype"), o.dump("ctype"), f"{nwave} waves, step {step}: ctype")
        assert list(g.ctl()[7:11]) == list(o.ctl()[7:11])
        for f in ("facev", "velg", "pos", "vel"):
            assert_f32_close(g.dump(f), o.dump(f), f"{nwave} waves, step {step}: {f}")
    print(f"[ocean columns] {nwave} waves: {sc.n} particle slots, reseed ctl {list(o.ctl()[7:11])}", flush=True)
    g.close()
