"""Joint islands by a wavefront with their records in LDS against one lane with them in HBM: a batch
takes the lanes when one of its worlds does not fit the LDS or when its joints are too many for a
wavefront each, and every world gets the same bits."""
import numpy as np
import pytest

from pypybox2d_amd import _native as N
from pypybox2d_amd import builder, layout as L, scenes

pytestmark = pytest.mark.gpu
DT = 1.0 / 60
LARGE = 110  # planks: 111 joints of 720 bytes do not fit 64 KB


def _run(batch, prec, iters, lds, events=0):
    e = N.Engine(prec)
    e.set_param("events", events)
    e.upload(batch)
    assert (e.get_param("joint_lds") > 0) == lds
    for _ in range(5):
        e.step(DT, *iters)
    ev = e.events() if events else None
    e.step_n(35, DT, *iters, graph=True)
    st = e.download()
    e.close()
    return st, ev


@pytest.mark.parametrize("prec,iters", [("fp64", (8, 3)), ("fp32", (8, 3)), ("fp64", (1, 0)), ("fp32", (0, 2))])
def test_records_in_lds_give_the_lanes_bits(prec, iters):
    specs = [scenes.joint_bridge(n) for n in (1, 2, 30, 63, 64, 65, 84)] + [scenes.joint_machines(), scenes.joint_gears()]
    batch = builder.scenes_batch(specs)
    batch.world_i[::2, L.WI_FLAGS] &= ~L.WF_WARM_STARTING
    lds, _ = _run(batch, prec, iters, True)
    with_large, _ = _run(L.concat([batch, builder.scene_batch(scenes.joint_bridge(LARGE))]), prec, iters, False)
    print(prec, iters, "joints", lds.n_joints, flush=True)
    for w in range(lds.n_worlds):
        a, b = lds.world(w), with_large.world(w)
        for f in ("body_d", "body_i", "con_d", "con_i", "joint_d", "joint_i"):
            assert np.array_equal(getattr(a, f), getattr(b, f)), (w, f)


def test_joint_bodies_come_to_rest_and_report_the_same():
    """Sleeping joint islands and post-solve records."""
    spec = dict(scenes.joint_bridge(6), do_sleep=True)
    batch = builder.scene_batch(spec)
    lds, ev = _run(batch, "fp64", (8, 3), True, events=15)
    large, ev2 = _run(L.concat([batch, builder.scene_batch(scenes.joint_bridge(LARGE))]), "fp64", (8, 3), False, events=15)
    part = ev2[0][:, 0] == 0
    assert np.array_equal(ev[0], ev2[0][part]) and np.array_equal(ev[1], ev2[1][part])
    assert np.array_equal(lds.body_d, large.world(0).body_d) and np.array_equal(lds.body_i, large.world(0).body_i)


@pytest.mark.parametrize("spec,copies", [(scenes.joint_bridge(12), 128), (scenes.joint_machines(), 98), (scenes.joint_gears(), 64)])
def test_batches_of_more_joints_than_the_wavefronts_hold_take_the_lanes(spec, copies):
    """The same worlds as often as wavefronts take them, once more, and so beside a large bridge, whose
    lane has more steps to hide them behind (4000 bridges took 1175 us by wavefronts, 294 by lanes)."""
    one, bridge = builder.scene_batch(spec), builder.scene_batch(scenes.joint_bridge(84))
    runs = {"few": (L.concat([one] * copies), True), "more": (L.concat([one] * (copies + 1)), False),
            "beside": (L.concat([one] * (copies + 1) + [bridge]), True)}
    first = {}
    for name, (batch, lds) in runs.items():
        st, _ = _run(batch, "fp32", (8, 3), lds)
        for w in (0, 1, copies - 1):
            got = st.world(w)
            for f in ("body_d", "con_d", "joint_d"):
                assert np.array_equal(getattr(got, f), first.setdefault(f, getattr(got, f))), (name, w, f)
        print(name, "lds", lds, flush=True)


def test_joint_sets_of_one_world_count_each():
    """Eight bridges of five planks in a world are eight islands: 16 such worlds are 128 wavefronts."""
    one = scenes.joint_bridge(5)
    bodies, joints = [one["bodies"][0]], []
    for k in range(8):
        x = 60.0 * (k + 1)
        shift = {i: i + len(bodies) - 1 if i > 0 else 0 for i in range(len(one["bodies"]))}
        joints += [dict(j, bodies=tuple(shift[i] for i in j["bodies"]), anchor=(j["anchor"][0] + x, j["anchor"][1]))
                   for j in one["joints"]]
        bodies += [dict(b, position=(b["position"][0] + x, b["position"][1])) for b in one["bodies"][1:]]
    batch = builder.scene_batch(dict(one, bodies=bodies, joints=joints))
    for n, lds in ((16, True), (17, False)):
        e = N.Engine("fp32")
        e.upload(L.concat([batch] * n))
        assert (e.get_param("joint_lds") > 0) == lds, n
        e.close()
