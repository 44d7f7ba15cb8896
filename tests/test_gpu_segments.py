"""The single-vector COO and CSR walks at the edges of their chunks: 256
segments (COO blocks, rows of CSR blocks) and 2048 entries per chunk, four
windows of 64 entries per step, rows without entries, long rows, and the
tiles' one-window sweep (n above 2^21).

Integer values and x keep every product and partial sum exact, so y must equal
the oracle's CSR SpMV bit for bit, in FP64 and in FP32 value storage."""
import numpy as np
import pytest

from abhsf_amd import AbhsfMatrix, synth
from abhsf_amd.hip import DeviceArray
from oracle import pyoracle

pytestmark = pytest.mark.gpu


def strip_of_blocks(s, counts, gap, seed, tall_row=False):
    """One strip plus a ragged second one: block J = 0, gap, 2 gap, ... holds
    counts[J] random entries (tall_row: its first row is full)."""
    rng = np.random.default_rng(seed)
    rows, cols = [], []
    for i, z in enumerate(counts):
        p = rng.permutation(s * s)[:z]
        if tall_row:
            p = np.unique(np.concatenate([np.arange(s), p]))[:max(z, s)]
        rows.append(p // s)
        cols.append(i * gap * s + p % s)
    n = len(counts) * gap * s + 3
    rows.append([s + 1, s + 1])
    cols.append([0, n - 1])
    r, c = np.concatenate(rows), np.concatenate(cols)
    v = rng.integers(1, 9, r.size) * rng.choice([-1.0, 1.0], r.size)
    return synth.from_triplets(s + 3, n, r, c, v)


CASES = {
    # COO: windows 1..4 with and without a remainder
    "coo_1": lambda: (strip_of_blocks(16, [1], 1, 1), 16),
    "coo_63_64_65": lambda: (strip_of_blocks(64, [63, 64, 65], 2, 2), 64),
    "coo_320": lambda: (strip_of_blocks(64, [64] * 5, 1, 3), 64),
    "coo_255_blocks": lambda: (strip_of_blocks(16, [1] * 255, 1, 4), 16),
    "coo_256_blocks": lambda: (strip_of_blocks(16, [2] * 256, 1, 5), 16),
    "coo_257_blocks": lambda: (strip_of_blocks(16, [1, 2] * 128 + [3], 1, 6), 16),
    # COO at the largest count per block: chunks end at 2048 entries
    "coo_512_each": lambda: (strip_of_blocks(256, [512] * 9, 1, 7), 256),
    "coo_2047_2049": lambda: (strip_of_blocks(256, [511, 512, 512, 512, 2, 500, 512, 512], 1, 8), 256),
    # CSR: several blocks per chunk, empty rows, a row across windows
    "csr_s32": lambda: (strip_of_blocks(32, [66, 100, 130, 70, 80, 90, 67, 120, 110], 1, 9), 32),
    "csr_s64": lambda: (strip_of_blocks(64, [140, 500, 130, 200, 300], 3, 10), 64),
    "csr_s64_tall": lambda: (strip_of_blocks(64, [200, 300, 400], 1, 11, True), 64),
    "csr_s128": lambda: (strip_of_blocks(128, [300, 2000, 1100], 1, 12, True), 128),
    # CSR beyond one mask (2048 entries)
    "csr_s256_7000": lambda: (strip_of_blocks(256, [2048, 7000, 2049, 600], 1, 13, True), 256),
}


def check(A, s, variant, precision):
    M = AbhsfMatrix(block_size=s, variant=variant, precision=precision)
    M.from_csr(A.m, A.n, A.rowptr, A.col, A.val)
    x = np.random.default_rng(5).integers(-8, 9, A.n).astype(np.float64)
    y0 = np.random.default_rng(6).integers(-8, 9, A.m).astype(np.float64)
    dx, dy = DeviceArray.from_numpy(x), DeviceArray.from_numpy(y0)
    M.spmv_async(1.0, dx, 1.0, dy)
    M.synchronize()
    assert np.array_equal(dy.numpy(), pyoracle.csr_spmv(A.rowptr, A.col, A.val, x, 1.0, 1.0, y0))
    return M.stats()


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("variant", ["strip", "balanced", "tiled"])
@pytest.mark.parametrize("name", list(CASES))
def test_chunk_edges_exact(gpu, name, variant, precision):
    A, s = CASES[name]()
    print(f"case {name} s={s} {variant} {precision}", flush=True)
    st = check(A, s, variant, precision)
    scheme = name.split("_")[0]
    assert st["blocks"][scheme] > 0


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("n", [1 << 21, (1 << 21) + 7])
def test_tile_sweep_exact(gpu, n, precision):
    """Scattered tiles on both sides of the sweep's line (2^21 columns)."""
    rng = np.random.default_rng(n)
    r = np.repeat(np.arange(1000), 12)
    A = synth.from_triplets(1000, n, r, rng.choice(n, r.size, replace=False), rng.integers(1, 9, r.size))
    print(f"case sweep n={n} {precision}", flush=True)
    st = check(A, 32, "tiled", precision)
    assert not st["tile_zs1"]


def with_integers(A, seed):
    rng = np.random.default_rng(seed)
    return synth.Csr(A.m, A.n, A.rowptr, A.col, (rng.integers(1, 9, A.nnz) * 1.0), A.name)


def gaps(n, seed):
    """Strips without entries, strips of one entry, and one long strip."""
    rng = np.random.default_rng(seed)
    r = np.concatenate([rng.choice(n, n // 40, replace=False), np.full(6000, n // 2), [0, n - 1]])
    c = np.concatenate([rng.integers(0, n, n // 40), rng.choice(n, 6000, replace=False), [n - 1, 0]])
    key = np.unique(r.astype(np.int64) * n + c)
    return synth.from_triplets(n, n, key // n, key % n, np.ones(key.size))


GROUPS = {  # matrices with several times 2048 strips (groups leave that many items)
    "laplacian_301_s4": lambda: (synth.laplacian2d(301), 4),      # T up to 11, ragged last strip
    "laplacian_700_s32": lambda: (synth.laplacian2d(700), 32),    # COO and CSR blocks, T up to 7
    "laplacian_700_s64": lambda: (synth.laplacian2d(700), 64),
    "rmat_17_s16": lambda: (synth.rmat(17, 8, seed=3), 16),       # bitmap strips and heavy strips between
    "rmat_16_s2": lambda: (synth.rmat(16, 4, seed=4), 2),         # 16 strips per group
    "gaps_s16": lambda: (gaps(100001, 5), 16),
    "gaps_s2": lambda: (gaps(150001, 6), 2),
}


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("variant", ["balanced", "tiled", "panel"])
@pytest.mark.parametrize("name", list(GROUPS))
def test_groups_exact(gpu, name, variant, precision):
    A, s = GROUPS[name]()
    A = with_integers(A, 1)
    print(f"case groups {name} {variant} {precision}", flush=True)
    st = check(A, s, variant, precision)
    if variant != "panel":  # (panels also split every strip that spans several)
        assert st["work_items"] < st["M"]
