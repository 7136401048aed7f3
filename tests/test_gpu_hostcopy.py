"""Field copies to host memory through the staging threads: every byte arrives at
sizes around the thresholds (a thread's share, the size from which buffers are
made, pieces that end inside a buffer), with several threads at once and with
no buffers left."""
import threading

import numpy as np
import pytest

from thesis_amd import lbm as L

pytestmark = pytest.mark.gpu


def solver(shape, seed):
    rng = np.random.default_rng(seed)
    f = [1.0 + 0.01 * rng.standard_normal(shape)] + [0.01 * rng.standard_normal(shape) for _ in range(3)]
    s = L.Solver(19, shape, np.ones(shape, np.uint8), None, collision=L.TRT, omega=1.2, periodic=(1, 1, 1))
    s.init(0, rho=f[0], u=f[1], v=f[2], w=f[3])   # the fields come back as they were given
    return s, f


# 4 fields of 8 bytes a node: 32 B, 4.2 MB, 8 MiB, 24 MB and one row less and more, 65 MB
@pytest.mark.parametrize("shape", [(1, 1, 1), (51, 51, 51), (64, 64, 64), (93, 90, 90), (92, 91, 94), (127, 126, 128)])
def test_fields_arrive(shape):
    print(f"case: {shape}", flush=True)
    s, f = solver(shape, shape[0])
    for _ in range(2):
        for a, b in zip(s.macros(), f):
            assert np.array_equal(a, b)
    s.close()


def test_populations_arrive():
    s, _ = solver((60, 61, 62), 3)
    s.step(1)
    a, b = s.get_f(), s.get_f()
    assert np.array_equal(a, b)
    assert np.allclose(a.sum(0), s.macros()[0], rtol=0, atol=1e-14 * 19)   # 19 additions of values below 1
    s.close()


def test_several_threads_share_the_buffers():
    made = [solver((100, 90, 90 + k), k) for k in range(6)]
    bad = []

    def work(k):
        s, f = made[k]
        for _ in range(5):
            if not all(np.array_equal(a, b) for a, b in zip(s.macros(), f)):
                bad.append(k)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
    for s, _ in made:
        s.close()
