"""A batch whose runs check at different intervals, and so take different numbers of
steps a barrier over different squares, and the largest batch there is: the same
bits as one step a barrier."""
import numpy as np
import pytest

from thesis_amd import lbm as L
from test_gpu_batch_phases import SHAPES, channels

pytestmark = pytest.mark.gpu


def fields(b):
    return [a for i in range(b.n) for a in b.macros(i) + [b.get_f(i)]]


def same(ds, runs):
    print(f"case batch of {len(ds)}: {runs}", flush=True)
    one, several = L.Batch(ds), L.Batch(ds)
    for every, steps in runs:
        for b, e in ((one, 1), (several, every)):
            done, _, _ = b.run(0.0, every=e, max_steps=steps)
            assert (done == steps).all()
        for a, c in zip(fields(one), fields(several)):
            assert np.array_equal(a, c), (every, steps)
    one.close()
    several.close()


def test_intervals_in_turn():
    same(channels(SHAPES), [(100, 120), (1, 3), (5, 23), (100, 7), (1, 1), (3, 9), (50, 101)])


def test_most_instances():
    ds = channels([(9 + k % 40, 5 + k % 23) for k in range(512)])
    for k, d in enumerate(ds):
        d["omega"] = 1.1 + 0.05 * (k % 7)
    same(ds, [(40, 41)])
