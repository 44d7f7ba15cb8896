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


def last_strip(s, counts, seed, diag=0):
    """Blocks (I, J) of one strip I, J = 0, 1, ... with counts[J] random
    entries, `diag` more in the strip's own block on and below the diagonal,
    and a ragged strip after it."""
    I, rng = len(counts), np.random.default_rng(seed)
    rc = [block(s, I, J, z, seed + J) for J, z in enumerate(counts) if z]
    if diag:
        r, c = np.tril_indices(s)
        p = np.sort(rng.permutation(r.size)[:diag])
        rc.append((I * s + r[p], I * s + c[p]))
    n = (I + 1) * s + 3
    rc.append((np.full(2, n - 2), np.array([0, n - 3])))
    r, c = np.concatenate([a for a, _ in rc]), np.concatenate([a for _, a in rc])
    return synth.from_triplets(n, n, r, c, rng.integers(1, 9, r.size) * rng.choice([-1.0, 1.0], r.size))


EDGES = {
    # entry by entry: chunks of 256 blocks, of 2048 entries
    "coo_s16_255": (16, [1] * 255), "coo_s16_256": (16, [2] * 256), "coo_s64_257": (64, [1, 2] * 128 + [3]),
    "coo_s256_2048": (256, [100] * 21), "coo_s4": (4, [2] * 70), "coo_s8": (8, [3, 9, 1] * 30),
    # sums by column: one chunk of blocks, one more, one less; the line at s / 2 entries
    "coo_s64_cap": (64, [64] * 8), "coo_s64_cap+1": (64, [64] * 9), "coo_s32_cap-1": (32, [40] * 15),
    "coo_s64_line": (64, [31] * 8 + [32] * 8 + [31] * 8), "coo_s16_line": (16, [7] * 32 + [8] * 32 + [7] * 32),
    "coo_s256_512": (256, [512] * 9), "coo_s256_odd": (256, [256, 1] * 5 + [200]),
    "coo_s128_4": (128, [64, 63, 64, 64, 64, 64, 65, 63]),
    # from one to the other and back, at every place within a lane's four blocks
    "coo_s64_turns": (64, [1] * 20 + [100] * 3 + [1] * 300), "coo_s128_turns": (128, [2] * 5 + [200] + [2] * 6 + [200] + [2] * 7 + [200]),
    "coo_s256_turns": (256, [3] * 7 + [400] + [3] * 2 + [400] * 3 + [3] * 260 + [400]),
    # CSR chunks of 256 rows, a block beyond one mask (2048 entries)
    "csr_s32": (32, [66, 100, 130, 70, 80, 90, 67, 120, 110]), "csr_s64": (64, [140, 500, 130, 200, 300]),
    "csr_s256_7000": (256, [2049, 7000, 2048]),
    "bm_s8": (8, [20, 60, 30]), "bm_s16": (16, [60, 250] * 3), "bm_s64": (64, [600, 4000]),
    "dense_s16": (16, [253, 256] * 3), "dense_s32": (32, [1020]),
}


@pytest.mark.parametrize("skew", [False, True])
@pytest.mark.parametrize("variant", ["strip", "balanced"])
@pytest.mark.parametrize("name", list(EDGES))
def test_mirrored_chunk_edges_exact(gpu, name, variant, skew):
    """Integer data: every sum is exact."""
    s, counts = EDGES[name]
    T = last_strip(s, counts, 1, 0 if skew else min(s, 30))
    x = np.random.default_rng(5).integers(-8, 9, T.n).astype(np.float64)
    print(f"case mirrored {name} {variant} skew={skew}", flush=True)
    got, st = spmv(T, x, s, 1.0, skew, variant)
    own = {"coo": "coo", "csr": "csr", "bm": "bitmap", "dense": "dense"}[name.split("_")[0]]
    extra = 2 if skew else 3  # the ragged strip's blocks, the diagonal one (s = 4: in one scheme or another)
    assert len(counts) <= st["blocks"][own] <= len(counts) + extra
    assert np.array_equal(got, product(T, x, 1.0, skew))
