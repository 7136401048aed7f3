"""D2Q9 steps several to a launch (squares of 32 x 32 nodes with a recomputed
frame) against one launch a step: the same bits in the fields, the populations
and the residuals, at box sizes around the squares, for every wall, face, force
and collision model; and against the oracle."""
import numpy as np
import pytest

from thesis_amd import lattices as LT
from thesis_amd import lbm as L
from test_gpu_parity import compare, pair

pytestmark = pytest.mark.gpu


def run(monkeypatch, multi, steps, shape, cls, bb, u0, **kw):
    if multi:
        monkeypatch.setenv("LBM_MULTI", str(multi))
    else:
        monkeypatch.delenv("LBM_MULTI", raising=False)
    s = L.Solver(9, shape, cls, bb, **kw)
    s.init(0, u=u0[0], v=u0[1])
    out = []
    for n in steps:
        s.step(n)
        out += list(s.macros()) + [s.get_f(), np.array(s.residual_l2())]
    out.append(np.array(s.run_to_residual(1e-30, every=11, max_steps=22)))
    out += list(s.macros())
    s.close()
    return out


def same(monkeypatch, shape, cls, bb, **kw):
    print(f"case: {shape} {kw.get('collision')} {kw.get('storage')} {kw.get('periodic')}", flush=True)
    rng = np.random.default_rng(shape[0])
    u0 = 0.02 * rng.standard_normal((2,) + tuple(shape))
    steps = (1, 2, 3, 17, 32)
    ref = run(monkeypatch, 1, steps, shape, cls, bb, u0, **kw)
    for multi in (None, 2, 5, 15):
        got = run(monkeypatch, multi, steps, shape, cls, bb, u0, **kw)
        for a, b in zip(ref, got):
            assert np.array_equal(a, b), multi


@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("shape", [(1, 3), (3, 2), (5, 40), (31, 33), (48, 25), (66, 130)])
@pytest.mark.parametrize("periodic", [(1, 1, 0), (1, 0, 0), (0, 1, 0)])
def test_periodic_boxes_with_solids(monkeypatch, storage, shape, periodic):
    rng = np.random.default_rng(shape[1])
    solid = rng.random(shape) < 0.1
    solid.flat[0] = False
    cls = np.where(solid, L.SOLID, L.FLUID).astype(np.uint8)
    bb = LT.bb_from_solid(solid, 9, periodic=(periodic[0], periodic[1], 1),
                          outside_is_wall=(not periodic[0], not periodic[1], False))
    same(monkeypatch, shape, cls, bb, storage=storage, collision=L.TRT, omega=1.2, periodic=periodic,
         force_model=L.FORCE_GUO, g=(1e-5, 2e-6, 0))


@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("coll", [L.BGK, L.TRT, L.MRT])
@pytest.mark.parametrize("outlet,inlet,parity", [(L.OUTLET_PRESSURE, L.INLET_ZOUHE, 0),
                                                 (L.OUTLET_REF_VELOCITY, L.INLET_REF2D, L.PARITY_OUTLET_V0),
                                                 (L.OUTLET_PRESSURE, L.INLET_ZOUHE, L.PARITY_INLET_FROZEN)])
def test_channels(monkeypatch, storage, coll, outlet, inlet, parity):
    d = LT.channel2d(141, 37, 0.05, obstacles=[(50.2, 17.1, 5.3)])
    ubc = d["ubc"].copy()
    ubc[:, -1] = 0.02
    for wall in (L.WALL_HALFWAY, L.WALL_ONNODE):
        same(monkeypatch, (37, 141), d["node_class"], d["bb"], storage=storage, collision=coll, omega=1.3, ubc=ubc,
             vbc=d["vbc"], outlet_model=outlet, inlet_model=inlet, parity=parity, wall_model=wall,
             force_model=L.FORCE_SHIFT, g=(1e-6, 0, 0))


@pytest.mark.parametrize("n", [24, 97])
@pytest.mark.parametrize("coll", [L.BGK, L.MRT])
@pytest.mark.parametrize("inlet", [L.INLET_ZOUHE, L.INLET_REF2D])
def test_cavity_and_oracle(monkeypatch, oracle, n, coll, inlet):
    d = LT.cavity2d(n, 0.08)
    kw = dict(collision=coll, omega=1.25, ubc=d["ubc"], vbc=d["vbc"], wall_model=L.WALL_ONNODE, inlet_model=inlet)
    same(monkeypatch, (n, n), d["node_class"], d["bb"], storage="f64", **kw)
    monkeypatch.delenv("LBM_MULTI", raising=False)
    g, o = pair(oracle, 9, (n, n), d["node_class"], d["bb"], **kw)
    g.init(0)
    o.init(0)
    compare(g, o, 150)
