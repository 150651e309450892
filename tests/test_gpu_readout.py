"""The readout kernels (b2g_download): records gathered on the device, in one piece or in chunks."""
import numpy as np
import pytest

from pypybox2d_amd import _native as N
from pypybox2d_amd import builder, layout as L, scenes

pytestmark = pytest.mark.gpu
DT = 1.0 / 60
FIELDS = ("world_d", "world_i", "body_d", "body_i", "fix_d", "fix_i", "con_d", "con_i", "move", "joint_d", "joint_i")


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("copies", [1, 300])
def test_every_world_reads_as_it_does_alone(prec, copies):
    """Worlds of 62 to 65 bodies, a joint world and a larger one, once and 300 times over (above the
    32 MB staged at once): each copy's records are those of the worlds read one at a time."""
    specs = [scenes.batch_world(5, k, n) for k, n in enumerate((62, 63, 64, 65, 180))] + [scenes.joint_bridge(12)]
    batch = builder.scenes_batch(specs)
    e = N.Engine(prec)
    e.upload(L.concat([batch] * copies))
    e.step_n(30, DT, 8, 3, graph=True)
    st = e.download()
    e.close()
    print(prec, copies, "records", st.body_d.nbytes + st.con_d.nbytes >> 20, "MB", flush=True)
    alone = []
    for k in range(len(specs)):
        e = N.Engine(prec)
        e.upload(batch.world(k))
        e.step_n(30, DT, 8, 3, graph=True)
        alone.append(e.download())
        e.close()
    for w in range(st.n_worlds):
        got, want = st.world(w), alone[w % len(specs)]
        for f in FIELDS:
            assert np.array_equal(getattr(got, f), getattr(want, f)), (w, f)


def test_dropped_contacts_are_left_out_in_place():
    batch = builder.scenes_batch([scenes.pyramid(5 + k) for k in range(3)])
    batch.world_i[:, L.WI_FLAGS] |= L.WF_CUSTOM_FILTER
    e = N.Engine("fp64")
    e.upload(batch)
    e.pair_search()
    rows = e.new_contacts()
    before = e.download()
    w = rows[::3, 0]
    first = np.searchsorted(rows[:, 0], w)
    j = np.arange(len(rows))[::3] - first
    e.drop_contacts(w, j)
    after = e.download()
    e.close()
    new = np.diff(before.con_off)
    start = before.con_off[:-1] + new - np.bincount(rows[:, 0], minlength=3)
    gone = start[w] + j
    keep = np.setdiff1d(np.arange(before.con_d.shape[0]), gone)
    assert len(gone) > 3
    assert np.array_equal(after.con_i, before.con_i[keep]) and np.array_equal(after.con_d, before.con_d[keep])
    assert np.array_equal(np.diff(after.con_off), new - np.bincount(w, minlength=3))
