"""Forms of the large-lattice and several-launch routes beside those their own test
files hold: extrapolating outlets and curved walls closed by a launch of their own in
FP32 and FP16, the single pass's default columns in FP32, the wide tile of the walled
step with the enhanced model, and mostly solid 2D boxes.

Tolerances against the FP64 oracle after 6 steps: FP32 rounds about 60 operations a step
to 2^-24 of deviations that sum to 0.6 at the fastest node, 6 x 2.1e-6 = 1.3e-5, taken as
3e-5.  FP16 stores these deviations to within 2^-10 of each (stochastic rounding): 6e-4 a
step, 6 of them 3.6e-3, taken as 4e-3."""
import numpy as np
import pytest

from thesis_amd import lattices as LT
from thesis_amd import lbm as L
from lattice_checks import sphere_wall_q
from test_gpu_boundaries3d import PAIRS, open_box
from test_gpu_cgw_tiles import run as walled_run
from test_gpu_multi2 import same
from test_gpu_parity import pair

pytestmark = pytest.mark.gpu

BIG = {"f32": (90, 93, 96), "f16": (115, 116, 118)}   # 58.2 and 57.0 MiB of populations: above the line of 56
TOL = {"f32": 3e-5, "f16": 4e-3}


@pytest.mark.parametrize("storage", ["f32", "f16"])
@pytest.mark.parametrize("k,outlet,coll,curved", [(0, L.OUTLET_EXTRAP2, L.TRT, False), (3, L.OUTLET_EXTRAP1, L.MRT, False),
                                                  (0, L.OUTLET_EXTRAP2, L.BGK, True)])
def test_closures_of_their_own_launch(oracle, storage, k, outlet, coll, curved):
    shape = BIG[storage]
    print(f"case {storage} {shape} pair {k} outlet {outlet} collision {coll} curved {curved}", flush=True)
    vel, out, axis, g = PAIRS[k]
    cls, U, per = open_box(vel, out, axis, g, shape)
    kw = dict(collision=coll, omega=1 / 0.8, periodic=per, ubc=U[0], vbc=U[1], wbc=U[2], outlet_model=outlet)
    bb = None
    if curved:
        solid, bb, q = sphere_wall_q(shape, (48.3, 45.7, 44.2), 9.4, q=19)
        cls[solid] = L.SOLID
        kw.update(wall_model=L.WALL_CURVED, wall_q=q)
    rng = np.random.default_rng(k)
    u0 = [0.02 * rng.standard_normal(shape) for _ in range(3)]
    gpu, ref = pair(oracle, 19, shape, cls, bb, storage=storage, **kw)
    for s in (gpu, ref):
        s.init(0, u=u0[0], v=u0[1], w=u0[2])
        s.step(6)
    for a, b in zip(gpu.macros(), ref.macros()):
        assert np.abs(a - b)[cls != L.SOLID].max() <= TOL[storage]
    gpu.close()


# 1.88 and 1.89 million nodes, above the 7/4 2^20 from which FP32 takes the single pass;
# the default columns do not divide the planes
@pytest.mark.parametrize("shape", [(128, 128, 115), (192, 128, 77)])
def test_default_columns_are_the_bits_of_two_launches(monkeypatch, shape):
    nx, ny, nz = shape
    r, b = LT.droplet3d(nx, ny, nz, 20.0, cx=60.2, cy=47.7, cz=31.3)
    out = []
    for zchunk in (None, "0"):
        print(f"case {shape} f32 zchunk {zchunk}", flush=True)
        if zchunk:
            monkeypatch.setenv("LBM_CG3_ZCHUNK", zchunk)
        g = L.CgSolver(nx, ny, nz=nz, storage="f32", beta=0.7, A=0.01125)
        g.init(r, b)
        g.step(10)
        m = g.macros()
        out.append([m[k] for k in sorted(m)] + list(g.get_f()))
        g.close()
    for a, c in zip(*out):
        assert np.array_equal(a, c)


def test_wide_walled_tile_with_the_enhanced_model(oracle):
    walled_run(oracle, 601, 437, 3, walls=1, high_order=0, enhanced=1, u_wall=0.01, g=-5e-5, external_force=1)


# squares without a live node among others, and the rule's own choice (one launch a step
# on the large box)
@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("shape", [(97, 210), (700, 900)])
def test_mostly_solid_boxes(monkeypatch, storage, shape):
    rng = np.random.default_rng(5)
    solid = np.ones(shape, bool)
    solid[: shape[0] // 3, 10:-7] = False
    solid[:, shape[1] // 2: shape[1] // 2 + 9] = False
    solid |= rng.random(shape) < 0.05
    cls = np.where(solid, L.SOLID, L.FLUID).astype(np.uint8)
    bb = LT.bb_from_solid(solid, 9, periodic=(True, True, True))
    same(monkeypatch, shape, cls, bb, storage=storage, collision=L.TRT, omega=1.2, periodic=(1, 1, 0),
         force_model=L.FORCE_GUO, g=(1e-5, 2e-6, 0))
