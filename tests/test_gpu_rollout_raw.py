"""Rollout's passes over arrays: several forward passes of different sizes may be
outstanding, and each backward pass reverses its own."""
import numpy as np
import pytest

from splashtank_amd import adjoint, capi, scenes
from tests.helpers import opts_for

pytestmark = pytest.mark.gpu

RTOL = 1e-5  # two runs of one gradient differ by the order of f32 atomics alone


def _inputs(sc, seed):
    rng = np.random.default_rng(seed)
    n = sc.n // (1 + seed)
    return sc.pos[:n, :3], rng.uniform(-0.5, 0.5, (n, 3)).astype(np.float32), rng.standard_normal((n, 3)).astype(np.float32)


def test_backward_takes_the_count_of_its_own_pass():
    sc = scenes.dam_break(d=1.0 / 32, iters=20)
    prm = capi.make_params(**sc.params)
    cases = [_inputs(sc, k) for k in range(2)]
    alone = []
    for pos, vel, w in cases:
        ro = adjoint.Rollout(opts_for(sc), prm, 4, every=3)
        _, _, snaps = ro.forward_raw(pos, vel, keep_snaps=True)
        alone.append(ro.backward_raw(snaps, w, 0.5 * w)[:2])
        ro.close()
    ro = adjoint.Rollout(opts_for(sc), prm, 4, every=3)
    outstanding = [ro.forward_raw(pos, vel, keep_snaps=True)[2] for pos, vel, _ in cases]
    for k in (0, 1):
        w = cases[k][2]
        for a, b in zip(ro.backward_raw(outstanding[k], w, 0.5 * w)[:2], alone[k]):
            assert a.shape == w.shape
            assert np.linalg.norm(a - b) <= RTOL * np.linalg.norm(b)
    ro.close()
