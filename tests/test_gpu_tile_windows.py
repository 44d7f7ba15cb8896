"""Scattered tiles on both sides of the sizes where their waves go from four
windows of 64 entries in flight to two and to one; integer data, exact."""
import numpy as np
import pytest

from abhsf_amd import AbhsfMatrix, synth
from abhsf_amd.hip import DeviceArray
from oracle import pyoracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("n", [5 << 18, (5 << 18) + 7, 7 << 18, (7 << 18) + 7])
def test_tile_windows_exact(gpu, n, precision):
    rng = np.random.default_rng(n)
    r = np.repeat(np.arange(1000), 12)
    A = synth.from_triplets(1000, n, r, rng.choice(n, r.size, replace=False), rng.integers(1, 9, r.size))
    print(f"case tile windows n={n} {precision}", flush=True)
    M = AbhsfMatrix(block_size=32, variant="tiled", precision=precision)
    M.from_csr(A.m, A.n, A.rowptr, A.col, A.val)
    assert not M.stats()["tile_zs1"]
    x = rng.integers(-8, 9, n).astype(np.float64)
    dx, dy = DeviceArray.from_numpy(x), DeviceArray.zeros(A.m)
    M.spmv_async(1.0, dx, 0.0, dy)
    M.synchronize()
    assert np.array_equal(dy.numpy(), pyoracle.csr_spmv(A.rowptr, A.col, A.val, x))
