"""The FP64 two-launch D3Q19 colour-gradient step (64 x 4 LDS tiles of the phase
field) at the edges of its tiles, against the oracle, and the default column
height of the single pass on a box of 2^20 nodes and more against the two
launches."""
import numpy as np
import pytest

from thesis_amd import lattices as LT
from thesis_amd import lbm as L
from test_gpu_cg3d import compare

pytestmark = pytest.mark.gpu


# boxes smaller than the frame of the large stencil, one node short of and over
# a tile in x and y, several tiles
@pytest.mark.parametrize("shape", [(3, 3, 3), (4, 5, 3), (63, 3, 4), (64, 4, 5), (65, 5, 6), (130, 9, 7), (61, 66, 8)])
@pytest.mark.parametrize("ho,enh", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_tiles_match_oracle(oracle, shape, ho, enh):
    nx, ny, nz = shape
    rng = np.random.default_rng(nx + ny)
    r = 0.2 + 0.6 * rng.random((nz, ny, nx))
    b = 0.6 * (1.0 - r)
    kw = dict(beta=0.7, A=0.01, r_nu=1 / 6, b_nu=0.1, r_alpha=0.3, b_alpha=0.4, high_order=ho, enhanced=enh)
    g = L.CgSolver(nx, ny, nz=nz, storage=L.STORE_F64, **kw)
    o = oracle.CgSim(nx, ny, nz=nz, nthreads=4, **kw)
    g.init(r, b)
    o.init(r, b)
    g.step(20)
    o.step(20)
    compare(g, o)
    g.close()


@pytest.mark.parametrize("shape", [(128, 128, 65), (192, 96, 61)])
@pytest.mark.parametrize("storage", ["f64", "f32"])
def test_default_columns_match_two_launches(monkeypatch, shape, storage):
    nx, ny, nz = shape
    r, b = LT.droplet3d(nx, ny, nz, 20.0, cx=60.2, cy=47.7, cz=31.3)
    out = []
    for zchunk in (None, "0"):
        if zchunk:
            monkeypatch.setenv("LBM_CG3_ZCHUNK", zchunk)
        g = L.CgSolver(nx, ny, nz=nz, storage=storage, beta=0.7, A=0.01125)
        g.init(r, b)
        g.step(10)
        out.append(g.macros())
        g.close()
    # ten steps from one start: FP64 rounding of populations of order 1, FP32 its
    # unit round-off 6e-8 of 38 of them a step
    tol = 1e-13 if storage == "f64" else 10 * 38 * 6e-8
    for k in out[0]:
        assert np.abs(out[0][k] - out[1][k]).max() <= tol, k


# the two launches carry the red density instead of the red populations: the same
# sum, so the same bits as the single pass
@pytest.mark.parametrize("shape", [(64, 8, 3), (64, 16, 5), (192, 24, 11)])
@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("enh", [0, 1])
def test_two_launches_are_the_bits_of_the_single_pass(monkeypatch, shape, storage, enh):
    nx, ny, nz = shape
    rng = np.random.default_rng(nx + ny)
    r = 0.2 + 0.6 * rng.random((nz, ny, nx))
    out = []
    for zchunk in ("0", "4"):
        print(f"case: {shape} {storage} enhanced={enh} zchunk={zchunk}", flush=True)
        monkeypatch.setenv("LBM_CG3_ZCHUNK", zchunk)
        g = L.CgSolver(nx, ny, nz=nz, storage=storage, beta=0.7, A=0.01, r_nu=1 / 6, b_nu=0.1, r_alpha=0.3, b_alpha=0.4,
                       enhanced=enh)
        g.init(r, 0.6 * (1.0 - r))
        g.step(10)
        m = g.macros()
        out.append([m[k] for k in sorted(m)] + list(g.get_f()))
        g.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
