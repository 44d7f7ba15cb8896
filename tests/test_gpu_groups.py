"""Groups of strips at their limits (64 strips, 256 rows), and the block counts
that the chunk-edge matrices of test_gpu_segments are meant to have."""
import numpy as np
import pytest

from abhsf_amd import AbhsfMatrix, synth
from test_gpu_segments import CASES, check, strip_of_blocks, with_integers

pytestmark = pytest.mark.gpu

FULL = {  # grid, block size: strips per group (a matrix of 2048 groups or more)
    "s2_64_strips": (520, 2, 64),
    "s4_64_strips": (730, 4, 64),
    "s32_256_rows": (730, 32, 8),
    "s16_bitmaps": (900, 16, 16), "s16_bitmaps_f32": (1460, 16, 16),  # (grouped in large matrices only)
}


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("variant", ["balanced", "tiled"])
@pytest.mark.parametrize("name", list(FULL))
def test_full_groups_exact(gpu, name, variant, precision):
    grid, s, strips = FULL[name]
    if name == "s16_bitmaps" and precision == "f32":
        strips = 1
    A = with_integers(synth.laplacian2d(grid), 1)
    print(f"case full groups {name} {variant} {precision}", flush=True)
    st = check(A, s, variant, precision)
    if strips == 1:
        assert st["work_items"] > st["M"] // 16
    elif variant == "balanced":
        assert st["work_items"] == -(-st["M"] // strips)


@pytest.mark.parametrize("name", list(CASES))
def test_chunk_edge_matrices_hold_their_blocks(gpu, name):
    """The first strip's blocks are all of the named scheme; the two of the
    second strip are COO blocks."""
    A, s = CASES[name]()
    r, c, _ = A.triplets()
    first = np.unique(c[r < s] // s).size
    M = AbhsfMatrix(block_size=s)
    M.from_csr(A.m, A.n, A.rowptr, A.col, A.val)
    blocks = M.stats()["blocks"]
    M.release()
    print(f"case blocks {name} {blocks}", flush=True)
    own = name.split("_")[0]
    assert blocks == {"coo": 2, "csr": 0, "bitmap": 0, "dense": 0, **{own: first + (2 if own == "coo" else 0)}}


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("counts,units", [
    ([1500] * 4, 4),               # two do not fit 2048 entries
    ([2048] * 3, 3), ([2049, 2047, 600], 3),
    ([7000], 1),                   # one block is never cut
    ([1100] * 6, 6),               # the even ones reach into the next multiple, the odd ones begin there
    ([1020] * 6, 3), ([300] * 20, 3),  # blocks below 1024 entries stay with the unit they begin in
])
def test_units_of_a_heavy_strip(gpu, counts, units, precision):
    """CSR blocks of one heavy strip: how many units it is cut into, and the
    exact product."""
    A = strip_of_blocks(256, counts, 1, 3)
    print(f"case units {counts} {precision}", flush=True)
    st = check(A, 256, "balanced", precision)
    assert st["work_items"] == units + 1  # (the ragged second strip)
