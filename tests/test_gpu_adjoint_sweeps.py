"""The transposed pressure solve with both colours of an iteration per launch: odd and
even iteration counts (the result ends in either buffer), a box that is no multiple of
the tile, lone drops and a collider give the gradients of the one-launch solve, which
makes the sweeps one by one.  The reversed g2p and p2g add with f32 atomics in any
order, hence 1e-5 in norm."""
import numpy as np
import pytest

from splashtank_amd import capi, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("iters", [1, 2, 5, 8])
def test_gradients_match_single_sweeps(iters):
    d = 1.0 / 52
    size = (1.0, 0.7, 0.6)
    rng = np.random.default_rng(iters)
    p1, _ = scenes.fill_box(d, -0.5, 0.5, 0.0, 0.2, -0.3, 0.3, rng)
    p3 = np.zeros((40, 4), np.float32)
    p3[:, :3] = rng.uniform((-0.49, 0.3, -0.29), (0.49, 0.69, 0.29), (40, 3))
    pos = np.concatenate([p1, p3])
    vel = np.zeros_like(pos)
    vel[:, :3] = rng.uniform(-1, 1, (len(pos), 3))
    h = 2 * d
    dims, lo, data = scenes.box_sdf((0.1, 0.08, 0.12), h, 4 * h)
    rec = scenes.collider_record(0, dims, lo, h, (-0.2, 0.15, 0.05), vel=(0.3, 0.0, 0.0))
    prm = capi.make_params(dt=1.0 / 240, iters=iters, omega=1.7)
    seed = rng.standard_normal((2, len(pos), 3))
    out = []
    for one in (True, False):
        g = capi.FlipSimC(capi.make_opts(d, size, max_n=len(pos)))
        g.upload(pos, vel)
        g.set_colliders(rec, data, 1)
        a = capi.AdjointC(g, 2)
        a.set_sor_path(one)
        for _ in range(2):
            a.record(prm)
        a.seed(seed[0], seed[1])
        for _ in range(2):
            a.backward()
            assert bool(a.sor_path()) == one
        out.append([x.copy() for x in a.grad()])
        a.close()
        g.close()
    for x, y in zip(*out):
        assert np.linalg.norm(x) > 0
        assert np.linalg.norm(x - y) <= 1e-5 * np.linalg.norm(x)
