"""Several steps per launch of the periodic D2Q9 colour gradient (squares of 32 x 32
nodes with a recomputed frame) against one launch a step.

The node update is the same code on the same values, so the results are the same
bits; FP16 storage keeps one launch a step, whatever is asked for."""
import numpy as np
import pytest

from thesis_amd import lbm as L

pytestmark = pytest.mark.gpu

# boxes smaller than the frame, one node around a square's inner side, several squares
SIZES = [(3, 3), (5, 70), (32, 33), (61, 47), (130, 29)]


@pytest.mark.parametrize("nx,ny", SIZES)
@pytest.mark.parametrize("storage", ["f64", "f32", "f16"])
@pytest.mark.parametrize("ho,enh,most", [(0, 0, None), (0, 1, 2), (0, 0, 8), (1, 0, None), (1, 1, 5), (1, 0, 2)])
def test_same_bits_as_single_steps(monkeypatch, nx, ny, storage, ho, enh, most):
    rng = np.random.default_rng(nx * 1000 + ny)
    red = rng.uniform(0.05, 0.95, (ny, nx))
    runs = []
    for m in (1, most):
        print(f"case: {nx}x{ny} {storage} high_order={ho} enhanced={enh} steps a launch {m}", flush=True)
        if m is None:
            monkeypatch.delenv("LBM_CG_MULTI", raising=False)
        else:
            monkeypatch.setenv("LBM_CG_MULTI", str(m))
        g = L.CgSolver(nx, ny, storage=storage, beta=0.7, A=1e-3, r_nu=1 / 6, b_nu=0.1, r_alpha=0.3, b_alpha=0.4,
                       high_order=ho, enhanced=enh)
        g.init(red, 1.0 - red)
        out = []
        for steps in (1, 2, 3, 17):   # no, one and several launches, whole and partial ones
            g.step(steps)
            out.append(g.macros())
        rf, bf = g.get_f()
        g.close()
        runs.append([o[k] for o in out for k in sorted(o)] + [rf, bf])
    assert all(np.isfinite(a).all() for a in runs[0])
    for a, b in zip(*runs):
        assert np.array_equal(a, b)
