"""The FP64 D2Q9 step with walls or a force in one launch, at the edges of its
tiles: boxes smaller than a tile's 14 x 14 (30 x 14) own nodes, exact multiples,
one more, and the size from which the wider tile is taken, against the oracle.

Tolerance: 12 steps of about a hundred rounded operations on values of the size
of the density, each good to 1.1e-16: 1.3e-13, taken as 1e-12; the velocity is a
sum of populations over the density, the same in lattice units."""
import numpy as np
import pytest

from thesis_amd import lbm as L

pytestmark = pytest.mark.gpu

SIZES = [(3, 5), (14, 14), (15, 29), (30, 28), (31, 15), (16, 6), (43, 57)]


def run(oracle, nx, ny, steps, **kw):
    rng = np.random.default_rng(nx * 1000 + ny)
    red = rng.uniform(0.05, 0.95, (ny, nx)).ravel()
    blue = 1.0 - red
    print(f"case: cg wall step {nx}x{ny} {kw}", flush=True)
    kw = dict(beta=0.7, A=1e-3, r_nu=1 / 6, b_nu=1 / 12, r_alpha=4 / 9, b_alpha=4 / 9, **kw)
    g = L.CgSolver(nx, ny, storage=L.STORE_F64, **kw)
    o = oracle.CgSim(nx, ny, **kw)
    g.init(red, blue)
    o.init(red, blue)
    g.step(steps - 1)   # an odd and an even number of steps: both buffers
    g.step(1)
    o.step(steps)
    gm, om = g.macros(), o.get()
    for k in ("r_rho", "b_rho", "rho", "u", "v"):
        assert np.abs(gm[k] - om[k]).max() <= 1e-12, k
    for a, b in zip(g.get_f(), (om["r_f"], om["b_f"])):
        assert np.abs(a - b).max() <= 1e-12
    g.close()


@pytest.mark.parametrize("walls,ho,enh", [(0, 0, 0), (1, 0, 1), (2, 0, 0), (0, 1, 0), (1, 1, 0), (2, 1, 1)])
@pytest.mark.parametrize("nx,ny", SIZES)
def test_one_launch_wall_step_matches_the_oracle(oracle, nx, ny, walls, ho, enh):
    force = dict(g=-5e-5, external_force=int(ho != enh))
    run(oracle, nx, ny, 12, walls=walls, high_order=ho, enhanced=enh, u_wall=0.01, **force)


@pytest.mark.parametrize("nx,ny", [(512, 512), (601, 437)])
def test_wider_tile_matches_the_oracle(oracle, nx, ny):
    run(oracle, nx, ny, 3, walls=2, high_order=0, enhanced=0, g=-5e-5, external_force=0)
