"""Rows of CSR blocks in the single-vector kernel: a row of a block is summed by
itself before it meets the strip's sum, products unrounded where its entries
follow each other in a lane; and the lengths of rows and chunks at which the
entries are taken differently."""
import numpy as np
import pytest

from abhsf_amd import AbhsfMatrix, synth
from abhsf_amd.hip import DeviceArray
from oracle import pyoracle

pytestmark = pytest.mark.gpu


def spmv(A, s, x, variant="balanced", precision="f64"):
    M = AbhsfMatrix(block_size=s, variant=variant, precision=precision)
    M.from_csr(A.m, A.n, A.rowptr, A.col, A.val)
    dx, dy = DeviceArray.from_numpy(x), DeviceArray.zeros(A.m)
    M.spmv_async(1.0, dx, 0.0, dy)
    M.synchronize()
    st = M.stats()
    M.release()
    return dy.numpy(), st


def test_products_are_not_rounded_within_a_row(gpu):
    """-1 + (1 + 2^-30)^2 is 2^-29 + 2^-60, the last bit of it only if the
    product is not rounded before it is added."""
    s, d = 64, 2.0 ** -30
    a = np.arange(s) % 30
    c = np.stack([2 * a, 2 * a + 1, 2 * a + 2, 2 * a + 3], 1)
    v = np.tile([-1.0, 1.0 + d, 0.0, 0.0], (s, 1))
    A = synth.from_triplets(s, s, np.repeat(np.arange(s), 4), c.ravel(), v.ravel())
    x = np.where(np.arange(s) % 2, 1.0 + d, 1.0)
    print("case csr fma", flush=True)
    y, st = spmv(A, s, x)
    assert st["blocks"]["csr"] == 1 and st["nnz"] == 4 * s
    assert np.all(y == 2 * d + d * d)


def test_a_row_is_summed_before_it_meets_the_strip_sum(gpu):
    """1e16 in one block and 1 + 1 + 1 in the next: the sum is 3 more, to
    within half the spacing of 2 there; each 1 by itself would be lost."""
    s = 64
    r = np.arange(s)
    rows = np.repeat(np.concatenate([r, r]), 3)
    c = np.concatenate([((r[:, None] + [0, 20, 40]) % s).ravel(), s + ((r[:, None] + [0, 20, 40]) % s).ravel()])
    v = np.concatenate([np.tile([1e16, 0.0, 0.0], s), np.ones(3 * s)])
    A = synth.from_triplets(s, 2 * s, rows, c, v)
    print("case csr row sums", flush=True)
    y, st = spmv(A, s, np.ones(2 * s))
    assert st["blocks"]["csr"] == 2
    assert np.all(np.abs(y - 1e16 - 3) <= 1)


def lengths(s, lens, seed):
    """One strip, one block: row r holds lens[r] random entries."""
    rng = np.random.default_rng(seed)
    r = np.repeat(np.arange(s), lens)
    c = np.concatenate([rng.permutation(s)[:k] for k in lens])
    return synth.from_triplets(s, s, r, c, rng.integers(1, 9, r.size) * rng.choice([-1.0, 1.0], r.size))


def tail(s, total):
    """Rows of 3 and 2 entries, `total` of them."""
    lens = np.full(s, total // s)
    lens[: total - lens.sum()] += 1
    return lens


ROWS = {
    # rows of one length, within and across lanes
    **{f"s64_rows_{k}": (64, [k] * 64) for k in (3, 4, 5, 6, 7, 8)},
    # rows that cover lanes, the 16 lanes a sum is passed in, and a whole step
    "s64_long_first": (64, [64] + [2] * 63), "s64_long_last": (64, [2] * 62 + [61, 64]),
    "s64_long_every_8": (64, [40 if i % 8 == 3 else 1 for i in range(64)]),
    "s256_whole_step": (256, [256, 255, 1, 256] + [3] * 252), "s256_odd": (256, [5, 0, 9, 0, 0, 17, 1, 2] * 32),
    # what is left after steps of 256: none, 1 to 64, more
    **{f"s128_left_{k}": (128, tail(128, 512 + k)) for k in (0, 1, 63, 64, 65, 128, 255)},
    **{f"s64_left_{k}": (64, tail(64, k)) for k in (191, 192, 193, 255, 257)},
}


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("name", list(ROWS))
def test_row_lengths_exact(gpu, name, precision):
    """Integer data: every sum is exact."""
    s, lens = ROWS[name]
    A = lengths(s, np.asarray(lens), 3)
    x = np.random.default_rng(5).integers(-8, 9, A.n).astype(np.float64)
    print(f"case csr rows {name} {precision}", flush=True)
    y, st = spmv(A, s, x, precision=precision)
    assert st["blocks"]["csr"] == 1
    assert np.array_equal(y, pyoracle.csr_spmv(A.rowptr, A.col, A.val, x))
