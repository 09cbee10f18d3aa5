"""A rollout keeps its host rows and adjoint context between calls: results do not
depend on what it ran before (other states, other counts, two forward passes
before their backward passes, a failed backward pass), on the device or on the
type of its inputs.  And the id-order dump made on the device: the same particles
as the id-order readback, and still refused when an id is past the live count."""
import numpy as np
import pytest
import torch

from splashtank_amd import adjoint, capi, scenes
from tests.helpers import opts_for

pytestmark = pytest.mark.gpu

# two runs of one gradient differ by the order of f32 atomics alone
RTOL = 1e-5


def _case(seed, sc):
    rng = np.random.default_rng(seed)
    n = sc.n - 100 * seed
    pos = torch.from_numpy(sc.pos[:n, :3].copy())
    vel = torch.from_numpy(rng.uniform(-0.5, 0.5, (n, 3)).astype(np.float32))
    return pos, vel, torch.from_numpy(rng.standard_normal((n, 3)).astype(np.float32))


def _grad(ro, pos, vel, w, device="cpu", dtype=torch.float32):
    p, v = pos.to(device, dtype).requires_grad_(), vel.to(device, dtype).requires_grad_()
    x, u = ro(p, v)
    assert x.dtype == dtype and x.device.type == device and x.shape == pos.shape
    return (p, v, x, u, w.to(device, dtype))


def _back(p, v, x, u, w):
    gp, gv = torch.autograd.grad([x, u], [p, v], [w, 0.5 * w])
    return [q.detach().to("cpu", torch.float64).numpy() for q in (x, u, gp, gv)]


def _same(a, b):
    for x, y in zip(a, b):
        assert np.linalg.norm(x - y) <= RTOL * max(np.linalg.norm(y), 1e-30)


@pytest.mark.parametrize("device,dtype", [("cpu", torch.float32), ("cuda", torch.float32), ("cuda", torch.float64)])
def test_rollout_results_do_not_depend_on_earlier_calls(device, dtype):
    sc = scenes.dam_break(d=1.0 / 32, iters=20)
    prm = capi.make_params(**sc.params)
    cases = [_case(k, sc) for k in range(3)]
    alone = []
    for c in cases:
        ro = adjoint.Rollout(opts_for(sc), prm, 4, every=3)
        alone.append(_back(*_grad(ro, *c)))
        ro.close()
    ro = adjoint.Rollout(opts_for(sc), prm, 4, every=3)
    for k in (1, 0, 2):
        _same(_back(*_grad(ro, *cases[k], device=device, dtype=dtype)), alone[k])
    first, second = _grad(ro, *cases[0], device=device, dtype=dtype), _grad(ro, *cases[1], device=device, dtype=dtype)
    _same(_back(*first), alone[0])
    _same(_back(*second), alone[1])
    bad = _grad(ro, *cases[2], device=device, dtype=dtype)
    ro.prm.drag = 0.1  # recording refuses this
    with pytest.raises(capi.StError):
        _back(*bad)
    ro.prm.drag = 0.0
    _same(_back(*_grad(ro, *cases[2], device=device, dtype=dtype)), alone[2])
    ro.close()


def test_dump_in_id_order():
    sc = scenes.dam_break(d=1.0 / 32, iters=10)
    g = capi.FlipSimC(opts_for(sc))
    g.upload(sc.pos, sc.vel)
    prm = capi.make_params(**sc.params)
    for _ in range(3):
        g.step(prm)
    assert np.array_equal(g.dump("pos"), g.read_particles())
    assert g.dump("vel").shape == (sc.n, 4)
    assert capi.load().st_set_count(g.h, sc.n // 2) == 0
    with pytest.raises(capi.StError, match="id out of range"):
        g.dump("pos")
    g.close()
