"""The register-resident island solve (groups of wavefronts, B2G_PARAM_GROUP_LOAD) against the
team and lane paths: the same solves in the same order, so the same bits, at the edges of its
classes (62 / 63, 126 / 127, 254 / 255, 510 / 511 and 1022 / 1023 contacts an island)."""
import numpy as np
import pytest

from pypybox2d_amd import _native as N
from pypybox2d_amd import builder, layout as L, scenes
from pypybox2d_amd.scenes import _body, _fix

pytestmark = pytest.mark.gpu
DT = 1.0 / 60

PATHS = {"groups": {"group_load": 1 << 20}, "default": {}, "few": {"group_load": 3},
         "teams64": {"group_load": 0, "heavy_class": 0, "team_full_class": 0},
         "teams8": {"group_load": 0, "heavy_class": 0, "team_full_class": 16},
         "fallback": {"group_load": 0, "heavy_class": 3, "team_lds": 4096},
         "pairs": {"group_load": 0, "heavy_class": 5, "team_full_class": 9, "team_max": 32},
         "lanes": {"heavy_class": 16}}


def _run(prec, state, vel_iters=8, pos_iters=3):
    out, times = {}, {}
    for name, params in PATHS.items():
        e = N.Engine(prec)
        for k, v in params.items():
            e.set_param(k, v)
        e.set_param("island_times", 1)
        e.upload(state)
        for _ in range(2):
            e.step(DT, vel_iters, pos_iters)
        e.step_n(2, DT, vel_iters, pos_iters, graph=True)
        out[name], times[name] = e.download(), e.island_times()
        print(prec, name, "done", flush=True)
        e.close()
    ref = out["lanes"]
    for name, st in out.items():
        for f in ("body_d", "body_i", "fix_d", "con_d", "con_i"):
            assert np.array_equal(getattr(st, f), getattr(ref, f)), (name, f)
    return times


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_islands_around_the_class_limits(prec):
    """Pyramids of 2 to 34 rows: islands of 3 to over 1022 contacts, one- and two-point manifolds."""
    rows = (2, 3, 5, 7, 8, 9, 11, 12, 13, 15, 18, 19, 22, 26, 31, 34)
    e = N.Engine(prec)
    e.upload(builder.scenes_batch([dict(scenes.pyramid(n), do_sleep=n % 2 == 0) for n in rows]))
    e.step_n(40, DT, 8, 3, graph=True)
    state = e.download()
    e.close()
    times = _run(prec, state)
    n = times["groups"][:, 2]
    assert n.max() > 1022 and set(times["groups"][n <= 1022, 4].tolist()) <= {1, 64}
    assert np.all(times["groups"][(n >= 31) & (n <= 1022), 4] == 64)


@pytest.mark.parametrize("prec,iters", [("fp64", (8, 3)), ("fp32", (8, 3)), ("fp32", (1, 0)), ("fp64", (0, 1))])
def test_piles_static_sides_and_iteration_counts(prec, iters):
    """Mixed piles (circles, polygons and edges on static ground), with and without warm starting."""
    counts = [16, 40, 96, 180, 260, 420, 512]
    batch = builder.scenes_batch([scenes.batch_world(9, w, n) for w, n in enumerate(counts)])
    e = N.Engine(prec)
    e.upload(batch)
    e.step_n(150, DT, 8, 3, graph=True)
    state = e.download()
    e.close()
    state.world_i[::2, L.WI_FLAGS] &= ~L.WF_WARM_STARTING
    _run(prec, state, *iters)


@pytest.mark.parametrize("prec,iters", [("fp64", 4000), ("fp32", 4103), ("fp32", 4104)])
def test_many_iterations_on_a_body_of_many_contacts(prec, iters):
    """Each of a slab's 301 contacts waits for the one before it: 4001 sweeps are 1.2 million solves one
    after another.  Groups take a step of up to 4103 iterations, the teams one of more."""
    bodies = [_body("static", (0.0, 0.0), [_fix(("edge", (-600.0, 0.0), (600.0, 0.0)))]),
              _body("dynamic", (0.0, 0.5), [_fix(("box", 180.0, 0.5), density=2.0, friction=0.5)])]
    bodies += [_body("dynamic", (1.1 * (k - 149.5), 1.49), [_fix(("box", 0.5, 0.5), density=1.0, friction=0.5)])
               for k in range(300)]
    batch = builder.scene_batch({"gravity": (0.0, -10.0), "bodies": bodies, "do_sleep": False, "warm_starting": True})
    out = []
    for load in (1 << 20, 0):
        e = N.Engine(prec)
        e.set_param("group_load", load)
        e.set_param("island_times", 1)
        e.upload(batch)
        e.step_n(3, DT, 8, 3, graph=True)
        e.step(DT, iters, 3)
        out.append((e.download(), e.island_times()[0]))
        print(prec, iters, load, "done", flush=True)
        e.close()
    (groups, gt), (teams, tt) = out
    assert gt[2] >= 300 and gt[4] == (64 if iters <= 4103 else 32) and tt[4] == 32
    for f in ("body_d", "con_d", "con_i"):
        assert np.array_equal(getattr(groups, f), getattr(teams, f)), f


def _towers(heights):
    bodies = [_body("static", (0.0, 0.0), [_fix(("edge", (-90.0, 0.0), (90.0, 0.0)))])]
    bodies += [_body("dynamic", (2.0 * (k - 0.5 * len(heights)), 0.49 + 0.99 * r), [_fix(("box", 0.5, 0.5), density=1.0)])
               for k, h in enumerate(heights) for r in range(h)]
    return {"gravity": (0.0, -10.0), "bodies": bodies, "do_sleep": False, "warm_starting": True}


@pytest.mark.parametrize("team_lds", [16384, 24576, 32768])
def test_groups_do_not_depend_on_the_teams_memory(team_lds):
    """Towers of 115 boxes do not fit a team's share of LDS in most of its sizes; in groups they take two
    wavefronts and their load all the same (3 workgroups, of which those of 40 boxes need one)."""
    batch = builder.scene_batch(_towers([115] * 8 + [40] * 8))
    out = []
    for load in (3, 0):
        e = N.Engine("fp64")
        e.set_param("group_load", load)
        e.set_param("team_lds", team_lds)
        e.set_param("island_times", 1)
        e.upload(batch)
        e.step_n(4, DT, 8, 3, graph=True)
        out.append((e.download(), e.island_times()))
        print(team_lds, load, "done", flush=True)
        e.close()
    assert sorted(set(out[0][1][:, 2].tolist())) == [40, 115] and set(out[0][1][:, 4].tolist()) == {64}
    assert 8 in out[1][1][:, 4]
    for f in ("body_d", "con_d", "con_i"):
        assert np.array_equal(getattr(out[0][0], f), getattr(out[1][0], f)), f


def _step_ms(batch, load):
    e = N.Engine("fp32")
    e.set_param("group_load", load)
    e.set_param("island_times", 1)
    e.upload(batch)
    e.step_n(4, DT, 8, 3, graph=True)
    st, lanes = e.download(), e.island_times()[:, 4]
    ms = min(float(e.profile(1, DT, 8, 3)[N.STAGES.index("solve")]) for _ in range(9))
    e.close()
    return st, lanes, ms


@pytest.mark.parametrize("heights,copies,want", [([1] * 3, 1, 1), ([2] * 3, 700, 1), ([3] * 8, 1, 64), ([3] * 8, 256, 64),
                                                 ([3] * 8, 257, 1), ([14] * 8, 513, 1), ([15] * 8, 512, 64),
                                                 ([40, 3, 3, 1], 300, None), ([1] * 5, 3000, 1)])
def test_small_islands_take_wavefronts_only_while_those_are_few(heights, copies, want):
    """Towers of one class: of up to two contacts a lane each; of three and more a wavefront each while 256
    workgroups of eight hold them, of seven and more while 512 do.  The group solver is no slower than the lanes and teams by more than
    its launch costs."""
    batch = L.concat([builder.scene_batch(_towers(heights))] * copies)
    st, lanes, ms = _step_ms(batch, 768)
    ref, _, ref_ms = _step_ms(batch, 0)
    print(heights, copies, np.unique(lanes, return_counts=True), "%.3f ms, without groups %.3f" % (ms, ref_ms), flush=True)
    if want is None:  # 40 high and 3 high in wavefronts, 1 high in a lane
        assert np.count_nonzero(lanes == 64) == 3 * copies and np.count_nonzero(lanes == 1) == copies
    else:
        assert set(lanes.tolist()) == {want}
    for f in ("body_d", "con_d", "con_i"):
        assert np.array_equal(getattr(st, f), getattr(ref, f)), f
    assert ms < 1.15 * ref_ms + 0.03
