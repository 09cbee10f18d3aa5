"""Rollouts hold no tapes between their passes: what several of them keep of the
device memory their backward passes took stays within the one block that the
library keeps, and a rollout may be closed after its tank."""
import pytest
import torch

from splashtank_amd import adjoint, capi, scenes
from tests.helpers import opts_for

pytestmark = pytest.mark.gpu

KEPT = 2**28  # the block, at most
RUNTIME = 2**26  # what the HIP runtime keeps of freed memory


def test_backward_gives_its_memory_back():
    sc = scenes.dam_break(d=1.0 / 128, iters=6)  # 64^3 cells: eight tapes and the gradients, over 300 MB
    pos, vel = (torch.from_numpy(q[:, :3].copy()).requires_grad_() for q in (sc.pos, sc.vel))
    rollouts, taken = [], 0
    for _ in range(4):
        ro = adjoint.Rollout(opts_for(sc), capi.make_params(**sc.params), 8, every=8)
        rollouts.append(ro)
        x, u = ro(pos, vel)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        (x.sum() + u.sum()).backward()
        torch.cuda.synchronize()
        assert not list(capi._LIVE["adjoint"])
        taken += free - torch.cuda.mem_get_info()[0]
        print(f"[rollout memory] {taken} bytes kept after {len(rollouts)} backward passes", flush=True)
    first = capi.AdjointC(rollouts[0].sim, 8)  # has the block
    free = torch.cuda.mem_get_info()[0]
    second = capi.AdjointC(rollouts[0].sim, 8)
    assert free - torch.cuda.mem_get_info()[0] > KEPT // 2  # each held more, with all of its tapes
    first.close()
    second.close()
    assert taken <= KEPT + RUNTIME
    for ro in rollouts:
        ro.sim.close()
        ro.close()
