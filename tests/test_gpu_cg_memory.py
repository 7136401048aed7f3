"""Device memory of a two-phase D3Q19 box: the fields its step reads and no more
(phase field and density, and the red density where two launches pass it on)."""
import pytest
import torch

from thesis_amd import lbm as L

pytestmark = pytest.mark.gpu
N, SLACK = 128, 12 << 20   # nodes a side; allocations are rounded up to 2 MiB each


@pytest.mark.parametrize("storage,zchunk,psi", [("f16", None, 2 * 4), ("f32", "16", 2 * 4), ("f32", "0", 3 * 4),
                                                ("f64", "16", 2 * 8), ("f64", "0", 3 * 8)])
def test_bytes_of_a_box(monkeypatch, storage, zchunk, psi):
    if zchunk:
        monkeypatch.setenv("LBM_CG3_ZCHUNK", zchunk)
    n = N ** 3
    warm = L.CgSolver(16, 16, nz=16, storage=storage)   # the context and the library's code are there
    before = torch.cuda.mem_get_info()[0]
    g = L.CgSolver(N, N, nz=N, storage=storage)
    taken = before - torch.cuda.mem_get_info()[0]
    want = n * (2 * 38 * {"f16": 2, "f32": 4, "f64": 8}[storage] + 8 * 8 + psi)
    print(f"{storage} zchunk {zchunk}: {taken} bytes, {want} wanted", flush=True)
    g.close()
    warm.close()
    assert taken <= want + SLACK
