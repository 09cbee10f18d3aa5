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


@pytest.mark.parametrize("steps", [0, 1, 2])
def test_failed_capture_leaves_the_tank_as_it_was(steps):
    """A substep whose capture fails has run no kernel: the particles are those
    before it, and the next substep marks and bins what a tank without it would."""
    out = json.loads(run(f"""
        import json
        sc = scenes.sparse_splash(d=1.0 / 64, iters=6)
        cf, sdf, sig = sc.collider_state(0.0, sc.params["dt"])
        prm = capi.make_params(**sc.params)
        out = []
        for fails in (0, 1):
            g = capi.FlipSimC(opts_for(sc))
            g.upload(sc.pos, sc.vel)
            for _ in range({steps}):
                g.step(prm)
            before = g.read_particles()
            g.set_colliders(cf, sdf, sig)
            if fails:
                hip.host_hip_set(b"failCapture", 1)
                try:
                    g.step_n(prm, 1, graph=True)
                    raise SystemExit("the capture did not fail")
                except capi.StError:
                    pass
                assert np.array_equal(g.read_particles(), before)
            log()
            g.step(prm)
            out.append(launches())
            g.step_n(prm, 2, graph=True)
            out.append(log())
        print(json.dumps(out))
        """))
    assert out[:2] == out[2:]


def test_failed_launch_clears_the_marks_again():
    """A blocks stage that failed may not have cleared the tile marks and bin counts:
    the next substep does before it marks."""
    out = json.loads(run("""
        import json
        sc = scenes.dam_break(d=1.0 / 32, iters=6)
        prm = capi.make_params(**sc.params)
        g = capi.FlipSimC(opts_for(sc))
        g.upload(sc.pos, sc.vel)
        g.begin_step(prm)
        g.stage(capi.ST_STAGE_SORT)
        log()
        hip.host_hip_set(b"failLaunch", 1)
        try:
            g.stage(capi.ST_STAGE_BLOCKS)
            raise SystemExit("the stage did not fail")
        except capi.StError:
            out = [[n for _, n, _, _ in launches()][:4]]
        g.step(prm)
        out.append([n for _, n, _, _ in launches()][:4])
        print(json.dumps(out))
        """))
    assert out[0] == out[1] == ["k_fill_u32", "k_fill_u32", "k_mark_bin", "k_tiles_scan"]


def test_failed_batch_launch_clears_the_marks_again():
    out = json.loads(run("""
        import json
        sc = scenes.dam_break(d=1.0 / 32, iters=6)
        prm = capi.make_params(**sc.params)
        g = capi.FlipSimC(opts_for(sc))
        g.upload(sc.pos, sc.vel)
        g.begin_step(prm)
        g.stages(capi.ST_STAGE_BLOCKS)  # leaves the marks and counts cleared
        b = capi.FlipBatchC([g])
        hip.host_hip_set(b"failLaunch", 1)
        try:
            b.step(prm)
            raise SystemExit("the step did not fail")
        except capi.StError:
            log()
        b.step(prm)
        print(json.dumps([n for _, n, _, _ in launches()][:3]))
        """))
    assert out == ["kb_fill_bins", "kb_mark_bin", "kb_tiles_scan"]


def test_grown_pool_is_cleared_before_it_is_filled():
    """st_grow clears new arrays on the tank's stream and copies the old ones in
    without a stream: a wait lies between."""
    out = json.loads(run("""
        import json
        sc = scenes.dam_break(d=1.0 / 32, iters=6)
        g = capi.FlipSimC(opts_for(sc, slots=20))
        g.upload(sc.pos, sc.vel)
        log()
        g.grow(25)
        print(json.dumps(log()))
        """))
    assert out.index("memset stream") < out.index("copy null")
    pending = False
    for line in out[:len(out) - out[::-1].index("copy null")]:
        if line == "memset stream":
            pending = True
        if line == "sync":
            pending = False
        if line == "copy null":
            assert not pending
            break


def test_adjoint_context_gives_its_memory_back():
    """A context's memory is free again after it but for one block, which the next
    context takes, and which goes with the last tank or when memory runs out. A tape
    that could not be allocated is allocated again by the next record."""
    out = json.loads(run("""
        import json
        sc = scenes.dam_break(d=1.0 / 32, iters=6)
        prm = capi.make_params(**sc.params)
        g = capi.FlipSimC(opts_for(sc))
        g.upload(sc.pos, sc.vel)
        g.step(prm)
        live = dict(before=hip.host_hip_live())
        a = capi.AdjointC(g, 2000)
        for k in ("failed", "again"):
            hip.host_hip_set(b"failMalloc", 1)
            try:  # until the tapes of one allocation are used up
                for _ in range(2000):
                    a.record(prm)
                raise SystemExit("no record failed")
            except capi.StError:
                live[k] = hip.host_hip_live()
        a.record(prm)
        live["more"] = hip.host_hip_live()
        a.close()
        live["closed"] = hip.host_hip_live()
        for k in ("second", "third"):
            a = capi.AdjointC(g, 2000)
            a.record(prm)
            live[k] = hip.host_hip_live()
            a.close()
        hip.host_hip_set(b"failMalloc", 1)
        q = capi.SnapshotC(g)
        q.close()
        live["dropped"] = hip.host_hip_live()
        capi.AdjointC(g, 1).close()
        live["kept"] = hip.host_hip_live()
        g.close()
        live["end"] = hip.host_hip_live()
        print(json.dumps(live))
        """))
    assert out["failed"] == out["again"] < out["more"]
    assert out["before"] < out["closed"] <= out["before"] + 2**28 + 4096
    assert out["second"] == out["third"] == out["closed"]
    assert out["dropped"] == out["before"] < out["kept"]
    assert out["end"] == 0


@pytest.mark.parametrize("sor_mode,cells,expect", [(1, 80, "k_sor_pipe"), (1, 64, "k_sor_pipe"), (0, 80, "k_sor_tiles"), (0, 112, "k_sor_tiles"),
                                                   (0, 150, "k_sor_resident")])
def test_band_routes_go_by_its_water_not_its_particles(sor_mode, cells, expect):
    """A narrow band has particles under the surface only: few of them say nothing of
    how many tiles hold water. Its launches per iteration are those of many tiles
    unless the pool itself is small, and the one-per-tile solve is tried only where
    the pool is at most three times what it holds."""
    names = json.loads(run(f"""
        import json
        d = 1.0 / {2 * cells}
        sc = scenes.dam_break(d=d, frac=(0.2, 0.05, 0.2), iters=6)
        g = capi.FlipSimC(opts_for(sc))
        g.upload(sc.pos, sc.vel)
        log()
        g.step(capi.make_params(**dict(sc.params, nb_on=1, nb_band=3.0, sor_mode={sor_mode})))
        print(json.dumps([n for _, n, _, _ in launches() if "sor" in n]))
        """))
    assert names[0] == expect, names


def test_small_band_takes_two_iterations_a_launch():
    names = json.loads(run("""
        import json
        sc = scenes.dam_break(d=1.0 / 96, frac=(0.2, 0.05, 0.2), iters=6)
        g = capi.FlipSimC(opts_for(sc))
        g.upload(sc.pos, sc.vel)
        log()
        g.step(capi.make_params(**dict(sc.params, nb_on=1, nb_band=3.0, sor_mode=1)))
        print(json.dumps([n for _, n, _, _ in launches() if "sor" in n]))
        """))
    assert set(names) == {"k_sor_pass"}


def test_clear_stage_on_its_own_clears():
    """A whole step clears the spare slot in the blocks stage; a caller that runs p2g
    twice with the clear stage between gets it cleared there."""
    out = json.loads(run("""
        import json
        sc = scenes.dam_break(d=1.0 / 32, iters=6)
        prm = capi.make_params(**sc.params)
        g = capi.FlipSimC(opts_for(sc))
        g.upload(sc.pos, sc.vel)
        log()
        g.step(prm)
        out = [[n for _, n, _, _ in launches()]]
        g.begin_step(prm)
        g.stages(capi.ST_STAGE_P2G)
        log()
        g.stage(capi.ST_STAGE_CLEAR)
        out.append([n for _, n, _, _ in launches()])
        print(json.dumps(out))
        """))
    assert "k_clear" not in out[0] and out[1] == ["k_clear"]


def test_adjoint_context_makes_the_one_launch_tables_when_asked():
    out = json.loads(run("""
        import json
        sc = scenes.dam_break(d=1.0 / 32, iters=6)
        g = capi.FlipSimC(opts_for(sc))
        a = capi.AdjointC(g, 1)
        live = [hip.host_hip_live()]
        for one in (0, 1, 0, 1):
            a.set_sor_path(one)
            live.append(hip.host_hip_live())
        print(json.dumps([live, g.dims.scap * 512 * 48]))
        """))
    live, tables = out
    assert live[0] == live[1] and live[2] == live[3] == live[4] and live[2] - live[1] >= tables
