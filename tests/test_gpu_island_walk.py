"""The island search's wavefront walk against the large worlds' search: the same islands, contact
order, ranks and levels, and so the same bits, where a body has more contacts than a wavefront has
lanes, where two bodies touch more than once, and where many islands share a static body."""
import numpy as np
import pytest

from pypybox2d_amd import _native as N
from pypybox2d_amd import builder, layout as L, scenes
from pypybox2d_amd.scenes import _body, _fix

pytestmark = pytest.mark.gpu
DT = 1.0 / 60


def _world(bodies):
    return {"gravity": (0.0, -10.0), "bodies": bodies, "do_sleep": False, "warm_starting": True}


def _box(hx, hy, x):
    return ("polygon", [(x - hx, -hy), (x + hx, -hy), (x + hx, hy), (x - hx, hy)])


def _ground():
    return _body("static", (0.0, 0.0), [_fix(("edge", (-90.0, 0.0), (90.0, 0.0)))])


def _boxes(n, y):
    return [_body("dynamic", (1.1 * (k - 0.5 * (n - 1)), y), [_fix(("box", 0.5, 0.5), density=1.0, friction=0.5)])
            for k in range(n)]


def crowded(n, kind="dynamic"):
    """A slab under n boxes: n contacts of one body and, on the ground, one more."""
    slab = _body(kind, (0.0, 0.5), [_fix(("box", 0.6 * n, 0.5), density=2.0, friction=0.5)])
    return _world([_ground(), slab] + _boxes(n, 1.49))


def sandwich(n):
    """n boxes between two dynamic slabs, the upper one of two fixtures side by side: contacts of two
    crowded bodies, taken by the lower slab and by the boxes."""
    slab = _body("dynamic", (0.0, 0.5), [_fix(("box", 0.6 * n, 0.5), density=2.0, friction=0.5)])
    lid = _body("dynamic", (0.0, 2.47), [_fix(_box(0.3 * n, 0.5, -0.3 * n), density=0.2, friction=0.5),
                                         _fix(_box(0.3 * n, 0.5, 0.3 * n), density=0.2, friction=0.5)])
    return _world([_ground(), slab] + _boxes(n, 1.49) + [lid])


def doubled(n):
    """A row of two-footed bodies on planks of two fixtures: pairs of bodies that touch up to four times."""
    bodies = [_ground()]
    for k in range(n):
        x = 3.0 * (k - 0.5 * n)
        bodies.append(_body("dynamic", (x, 0.25), [_fix(_box(0.6, 0.25, -0.6), density=2.0, friction=0.6),
                                                    _fix(_box(0.6, 0.25, 0.6), density=2.0, friction=0.6)]))
        bodies.append(_body("dynamic", (x, 0.99), [_fix(_box(0.3, 0.5, -0.4), density=1.0, friction=0.6),
                                                    _fix(_box(0.3, 0.5, 0.4), density=1.0, friction=0.6)]))
    return _world(bodies)


def singles(n):
    """n boxes apart on one ground: an island each, all with the same static body."""
    return _world([_ground()] + [_body("dynamic", (1.5 * (k - 0.5 * n), 0.49), [_fix(("box", 0.5, 0.5), density=1.0)])
                                 for k in range(n)])


SCENES = {"crowded": [crowded(n) for n in (15, 16, 17, 62, 63, 64, 65, 130)],
          "kinematic": [crowded(n, "kinematic") for n in (16, 17, 130, 300)],
          "sandwich": [sandwich(n) for n in (7, 15, 16, 17, 130, 300)], "doubled": [doubled(n) for n in (1, 5, 28)],
          "singles": [singles(n) for n in (1, 62, 63, 64, 110)]}


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("name", sorted(SCENES))
def test_walk_agrees_with_the_large_worlds_search(prec, name):
    batch = builder.scenes_batch(SCENES[name])
    out = {}
    for path, params in (("walk", {}), ("wide", {"islands_wide": 32}), ("narrow", {"islands_wide": 0}),
                         ("teams", {"group_load": 0, "heavy_class": 0}), ("large", {"large_worlds": 1})):
        e = N.Engine(prec)
        for k, v in params.items():
            e.set_param(k, v)
        e.upload(batch)
        e.step_n(40, DT, 8, 3, graph=True)
        out[path] = e.download()
        print(prec, name, path, "done", flush=True)
        e.close()
    ref = out["large"]
    touching = ref.con_i[:, L.CI_FLAGS] & L.CF_TOUCHING != 0
    assert touching.sum() >= len(SCENES[name])
    if name == "doubled":
        w = np.repeat(np.arange(ref.n_worlds), np.diff(ref.con_off))
        fa = ref.fix_i[ref.fix_off[w] + ref.con_i[:, L.CI_FA], L.FI_BODY]
        fb = ref.fix_i[ref.fix_off[w] + ref.con_i[:, L.CI_FB], L.FI_BODY]
        pairs = np.stack([w, np.minimum(fa, fb), np.maximum(fa, fb)], 1)[touching & (fa != 0) & (fb != 0)]
        assert len(np.unique(pairs, axis=0)) < len(pairs)  # some pair of bodies touches more than once
    for path, st in out.items():
        for f in ("body_d", "body_i", "fix_d", "con_d", "con_i"):
            assert np.array_equal(getattr(st, f), getattr(ref, f)), (path, f)


def test_a_crowded_body_costs_no_more_than_as_many_apart():
    """The island search of 600 boxes on a slab against that of 600 on static ground (once 21 times it)."""
    ms = {}
    for kind in ("kinematic", "dynamic", "static"):
        e = N.Engine("fp32")
        e.upload(builder.scene_batch(crowded(600, kind)))
        e.step_n(10, DT, 8, 3, graph=True)
        ms[kind] = np.median([e.profile(1, DT, 8, 3)[N.STAGES.index("islands")] for _ in range(7)])
        print(kind, ms[kind], flush=True)
        e.close()
    assert max(ms["kinematic"], ms["dynamic"]) < 3 * ms["static"]
