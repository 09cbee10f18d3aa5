"""The narrow band's reseed around the edges of its blocks: particle counts of whole
blocks of 1024, one more, and more than 2048 blocks of 1024 (each block then takes
several), dead particles listed from all of them; the counts of dead, short cells and
filled slots and the state after each substep match the oracle."""
import numpy as np
import pytest

from splashtank_amd import capi, scenes
from splashtank_amd.capi import FlipSimC
from oracle.oracle import Oracle
from tests.helpers import assert_f32_close, opts_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("total", [0, 1, 1023, 2048 * 1024 + 5000])
def test_reseed_matches_oracle(total):
    sc = scenes.nb_pool(d=1.0 / 40, depth=0.45, drop=(0.1, 0.7, 0.0, 0.08))
    live = np.flatnonzero(sc.pos[:, 1] > -1e5)
    sc.pos[live[::2], :] = [0.0, -1e6, 0.0, 0.0]  # the reseed refills their cells
    n = total if total > 1024 else (len(sc.pos) + 1023) // 1024 * 1024 + total
    rng = np.random.default_rng(total)
    at = np.sort(rng.permutation(n)[: len(sc.pos)])  # the pool's particles spread over all ids
    pos = np.zeros((n, 4), np.float32)
    pos[:, 1] = -1.0e6
    vel = np.zeros_like(pos)
    pos[at], vel[at] = sc.pos, sc.vel
    sc.pos, sc.vel = pos, vel
    opts = opts_for(sc, max_n=n)
    g, o = FlipSimC(opts), Oracle(opts)
    for s in (g, o):
        s.upload(pos, vel)
    for step in range(2):
        kw = dict(sc.params)
        if step == 0:
            kw.update(nb_init=1, nfill=len(sc.nb_fills) // 8, fills=list(sc.nb_fills))
        prm = capi.make_params(**kw)
        for s in (g, o):
            s.step(prm)
        a, b = g.ctl(), o.ctl()
        assert list(a[7:11]) == list(b[7:11]), (a[7:11], b[7:11])
        assert a[8] > 0 and (a[9] > 0 or step)
        for f in ("pos", "vel"):
            assert_f32_close(g.dump(f), o.dump(f), f"step {step}: {f}")
    g.close()
