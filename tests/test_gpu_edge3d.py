"""D3Q19 lattices large enough that extrapolating outlets and curved walls are
closed by a launch of their own (56 MiB of populations), against the FP64
oracle: every face, both orders, wet-node and curved walls beside them."""
import numpy as np
import pytest

from thesis_amd import lattices as LT
from thesis_amd import lbm as L
from lattice_checks import sphere_wall_q
from test_gpu_boundaries3d import PAIRS, open_box
from test_gpu_parity import compare, pair

pytestmark = pytest.mark.gpu
SHAPE = (70, 73, 77)   # 393 470 nodes: 57.04 MiB in FP64


@pytest.mark.parametrize("k", range(6))
@pytest.mark.parametrize("outlet,coll", [(L.OUTLET_EXTRAP2, L.TRT), (L.OUTLET_EXTRAP1, L.MRT)])
def test_extrapolating_faces(oracle, k, outlet, coll):
    vel, out, axis, g = PAIRS[k]
    cls, U, per = open_box(vel, out, axis, g, SHAPE)
    cls[30:40, 30:40, 30:40] = L.SOLID
    end = [40, 40, 40]
    end[2 - axis] = -2 if g > 0 else 1   # a solid node upstream of the outlet
    cls[tuple(end)] = L.SOLID
    bb = LT.bb_from_solid(cls == L.SOLID, 19, periodic=per)
    rng = np.random.default_rng(k)
    u0 = [0.02 * rng.standard_normal(SHAPE) for _ in range(3)]
    gg, o = pair(oracle, 19, SHAPE, cls, bb, collision=coll, omega=1 / 0.8, periodic=per, ubc=U[0], vbc=U[1],
                 wbc=U[2], outlet_model=outlet)
    gg.init(0, u=u0[0], v=u0[1], w=u0[2])
    o.init(0, u=u0[0], v=u0[1], w=u0[2])
    compare(gg, o, 6)


@pytest.mark.parametrize("coll", [L.BGK, L.MRT])
def test_duct_with_wet_node_walls(oracle, coll):
    d = LT.duct3d(101, 63, 0.05)
    gg, o = pair(oracle, 19, (63, 63, 101), d["node_class"], d["bb"], collision=coll, omega=1 / 0.8, ubc=d["ubc"],
                 vbc=d["vbc"], wbc=d["wbc"], wall_model=L.WALL_HH, outlet_model=L.OUTLET_EXTRAP1)
    gg.init(0)
    o.init(0)
    compare(gg, o, 8)


def test_curved_sphere_between_open_faces(oracle):
    vel, out, axis, g = PAIRS[0]
    cls, U, per = open_box(vel, out, axis, g, SHAPE)
    solid, bb, q = sphere_wall_q(SHAPE, (38.3, 35.7, 34.2), 9.4, q=19)
    cls[solid] = L.SOLID
    gg, o = pair(oracle, 19, SHAPE, cls, bb, collision=L.TRT, omega=1 / 0.8, periodic=per, ubc=U[0], vbc=U[1],
                 wbc=U[2], outlet_model=L.OUTLET_EXTRAP2, wall_model=L.WALL_CURVED, wall_q=q)
    gg.init(0)
    o.init(0)
    compare(gg, o, 8)
