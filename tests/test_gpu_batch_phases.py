"""Batched channels advancing several steps a barrier: any check interval and any
number of instances gives the fields of single-lattice runs, exactly the same
as a run checked after every step (one step a barrier throughout)."""
import numpy as np
import pytest

from thesis_amd import lattices as LT
from thesis_amd import lbm as L
from test_gpu_batch import check_instance, oracle_of

pytestmark = pytest.mark.gpu


def channels(shapes):
    out = []
    for k, (nx, ny) in enumerate(shapes):
        d = LT.channel2d(nx, ny, 0.04, obstacles=[(nx * 0.4, ny * 0.45, ny / 7.0)] if ny > 8 else ())
        d.update(omega=1.1 + 0.05 * k, trt_magic=3.0 / 16.0)
        out.append(d)
    return out


# a row, boxes at the squares' edges, one square and a bit, many squares
SHAPES = [(3, 1), (12, 12), (13, 25), (31, 9), (33, 32), (150, 40), (301, 77)]


@pytest.mark.parametrize("collision", [L.TRT, L.BGK])
@pytest.mark.parametrize("count", [1, 7])
@pytest.mark.parametrize("every,steps", [(2, 12), (3, 10), (5, 23), (50, 51), (100, 37)])
def test_any_check_interval(collision, count, every, steps):
    ds = channels(SHAPES[-count:])
    print(f"case phases count={count} every={every} steps={steps}", flush=True)
    out = []
    for e in (1, every):
        b = L.Batch(ds, collision=collision, storage="f64")
        for n in (steps, 7):            # the second run starts on either buffer
            got, res, _ = b.run(0.0, every=e, max_steps=n)
            assert (got == n).all()
        out.append([a for i in range(count) for a in b.macros(i) + [b.get_f(i)]])
        b.close()
    for a, c in zip(*out):
        assert np.array_equal(a, c)


def test_many_squares_against_oracle(oracle):
    ds = channels([(600, 150), (57, 31), (1024, 256)])
    b = L.Batch(ds, collision=L.TRT, storage="f64")
    b.run(0.0, every=40, max_steps=75)
    for i, d in enumerate(ds):
        o = oracle_of(oracle, d, L.TRT)
        o.init(0)
        o.step(75)
        check_instance(b, i, o, d)
    b.close()
