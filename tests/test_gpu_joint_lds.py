"""Joint islands by a wavefront with their records in LDS against one lane with them in HBM: a batch
takes the lanes when one of its worlds does not fit the LDS, and every world gets the same bits."""
import numpy as np
import pytest

from pypybox2d_amd import _native as N
from pypybox2d_amd import builder, layout as L, scenes

pytestmark = pytest.mark.gpu
DT = 1.0 / 60
LARGE = 110  # planks: 111 joints of 720 bytes do not fit 64 KB


def _run(batch, prec, iters, events=0):
    e = N.Engine(prec)
    e.set_param("events", events)
    e.upload(batch)
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
    lds, _ = _run(batch, prec, iters)
    with_large, _ = _run(L.concat([batch, builder.scene_batch(scenes.joint_bridge(LARGE))]), prec, iters)
    print(prec, iters, "joints", lds.n_joints, flush=True)
    for w in range(lds.n_worlds):
        a, b = lds.world(w), with_large.world(w)
        for f in ("body_d", "body_i", "con_d", "con_i", "joint_d", "joint_i"):
            assert np.array_equal(getattr(a, f), getattr(b, f)), (w, f)


def test_joint_bodies_come_to_rest_and_report_the_same():
    """Sleeping joint islands and post-solve records."""
    spec = dict(scenes.joint_bridge(6), do_sleep=True)
    batch = builder.scene_batch(spec)
    lds, ev = _run(batch, "fp64", (8, 3), events=15)
    large, ev2 = _run(L.concat([batch, builder.scene_batch(scenes.joint_bridge(LARGE))]), "fp64", (8, 3), events=15)
    part = ev2[0][:, 0] == 0
    assert np.array_equal(ev[0], ev2[0][part]) and np.array_equal(ev[1], ev2[1][part])
    assert np.array_equal(lds.body_d, large.world(0).body_d) and np.array_equal(lds.body_i, large.world(0).body_i)
