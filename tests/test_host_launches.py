"""What the library's host code launches, on a HIP runtime of host memory (no
kernel runs, tests/host_hip.py): the routes of the pressure solve where a launch
cannot do all of it, is refused, or has done it already."""
import json

import pytest

from tests.host_hip import run

SOR = ("k_sor_tiles", "k_sor_resident", "k_sor_pass", "k_sor_pipe", "kb_sor_counts", "kb_sor_tiles", "kb_sor_plan", "kb_sor_resident", "kb_sor_pass",
       "kb_sor_pipe")


@pytest.mark.parametrize("cap", [0, 2, 4, 8, 54, 255, 256])
def test_capped_batch_always_has_a_solve_that_covers_it(cap):
    """Two 16^3 tanks can use 54 tiles; the one-per-tile launch alone is enough only
    with a workgroup for each of them."""
    names = json.loads(run(f"""
        import json
        tanks = [scenes.dam_break(d=1.0 / 32, iters=6) for _ in range(2)]
        sims = [capi.FlipSimC(opts_for(sc)) for sc in tanks]
        for s, sc in zip(sims, tanks):
            s.upload(sc.pos, sc.vel)
        b = capi.FlipBatchC(sims)
        b.sor_grid({cap})
        log()
        b.step([capi.make_params(**sc.params) for sc in tanks])
        print(json.dumps([(n, g) for _, n, g, _ in launches() if "sor" in n]))
        """))
    assert all(n in SOR for n, _ in names)
    if cap == 0:
        assert {n for n, _ in names} <= {"kb_sor_pass", "kb_sor_pipe"}
        return
    covered = any(n == "kb_sor_tiles" and g >= 54 for n, g in names)
    assert covered or ("kb_sor_plan" in dict(names) and "kb_sor_resident" in dict(names)), names


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("solved", [1, 0])
def test_refused_second_launch_does_not_repeat_a_solve(batch, solved):
    """Where more tiles can be in use than are sure to fit at once, a second
    cooperative launch follows the one-per-tile one. If it is refused, launches per
    iteration follow where the first did not do the solve, and only there."""
    names = json.loads(run(f"""
        import json
        sc = scenes.dam_break(d=1.0 / 176, frac=(0.2, 0.2, 0.2), iters=6)
        assert 12 ** 3 > 4 * 256
        sims = [capi.FlipSimC(opts_for(sc)) for _ in range(2 if {batch} else 1)]
        for s in sims:
            s.upload(sc.pos, sc.vel)
        b = capi.FlipBatchC(sims) if {batch} else sims[0]
        prm = capi.make_params(**sc.params)
        hip.host_hip_set(b"refuse", 1024)
        hip.host_hip_set(b"solves", {solved})
        log()
        b.step(prm)
        print(json.dumps([(w, n) for w, n, _, _ in launches() if "sor" in n]))
        """))
    per_iteration = [n for _, n in names if n.endswith(("pass", "pipe"))]
    assert [w for w, n in names if n.endswith("sor_tiles")] == ["coop"]
    assert [w for w, n in names if n.endswith("resident")] == ["refused"]
    assert bool(per_iteration) == (not solved), names
