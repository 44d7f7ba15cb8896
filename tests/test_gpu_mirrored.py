"""One-triangle storage: the pass that applies the mirrored triangle, at its
own limits (values of x and alpha at the ends of the range, the edges of its
chunks), against products summed entry by entry in numpy."""
import numpy as np
import pytest

from abhsf_amd import AbhsfMatrix, synth
from abhsf_amd.hip import DeviceArray

pytestmark = pytest.mark.gpu


def block(s, I, J, z, seed):
    """z entries of block (I, J), at random positions: rows, columns."""
    p = np.random.default_rng(seed).permutation(s * s)[:z]
    return I * s + p // s, J * s + p % s


def product(T, x, alpha=1.0, skew=False):
    """alpha A x of the whole matrix, each product rounded as (alpha v) x."""
    r, c, v = T.triplets()
    off = r != c
    y = np.zeros(T.m)
    np.add.at(y, r, alpha * (v * x[c]))
    np.add.at(y, c[off], ((-alpha if skew else alpha) * v[off]) * x[r[off]])
    return y


def spmv(T, x, s, alpha=1.0, skew=False, variant="balanced"):
    M = AbhsfMatrix(block_size=s, variant=variant)
    M.from_csr(T.m, T.n, T.rowptr, T.col, T.val, symmetry="skew" if skew else "symmetric")
    dx, dy = DeviceArray.from_numpy(x), DeviceArray.zeros(T.m)
    M.spmv_async(alpha, dx, 0.0, dy)
    M.synchronize()
    st = M.stats()
    M.release()
    return dy.numpy(), st


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("s", [16, 32, 64])
def test_dense_padding_times_a_non_finite_x(gpu, s, bad):
    """A dense block stores a zero at a position that holds no entry: a
    non-finite x of that row does not reach the position's column."""
    r, c = block(s, 1, 0, s * s, 1)
    i = s + 5
    missing = [0, 3] if s == 16 else [0, 3, s - 1]
    keep = ~((r == i) & np.isin(c, missing))
    r, c = r[keep], c[keep]
    T = synth.from_triplets(2 * s + 3, 2 * s + 3, r, c, np.random.default_rng(2).integers(1, 9, r.size) * 1.0)
    x = np.random.default_rng(3).integers(-8, 9, T.n).astype(np.float64)
    x[i] = bad
    print(f"case mirrored dense padding s={s} x={bad}", flush=True)
    got, st = spmv(T, x, s)
    assert st["blocks"]["dense"] == 1
    ref = product(T, x)
    assert np.isfinite(ref[missing]).all() and not np.isfinite(ref[:s]).all()
    assert np.array_equal(got, ref, equal_nan=True)


@pytest.mark.parametrize("alpha,v,big", [(1e200, 1e-100, 1e150), (-1e-200, 1e200, 1e-150), (1e-200, 1e150, 1e200)])
@pytest.mark.parametrize("skew", [False, True])
def test_products_that_stay_in_range_do(gpu, alpha, v, big, skew):
    """(alpha v) x is taken as such, in all four schemes: alpha x alone would
    be infinite, or zero."""
    s = 32
    rc = [block(s, I, 0, z, I) for I, z in ((1, 40), (2, 100), (3, 500), (4, 1020))]
    r, c = np.concatenate([a for a, _ in rc]), np.concatenate([a for _, a in rc])
    T = synth.from_triplets(5 * s, 5 * s, r, c, np.full(r.size, v))
    x = np.full(T.n, big)
    x[:s] = 1.0
    print(f"case mirrored range alpha={alpha} v={v} x={big} skew={skew}", flush=True)
    got, st = spmv(T, x, s, alpha, skew)
    assert list(st["blocks"].values()) == [1, 1, 1, 1]
    ref = product(T, x, alpha, skew)
    assert np.isfinite(ref).all() and (ref[:s] != 0).all()
    # sums of at most 1660 products of one sign: 2 * 1660 roundings at most
    assert np.all(np.abs(got - ref) <= 2 * 1660 * 2.0 ** -53 * np.abs(ref))
