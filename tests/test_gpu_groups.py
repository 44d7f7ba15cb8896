"""Groups of strips at their limits (64 strips, 256 rows), and the block counts
that the chunk-edge matrices of test_gpu_segments are meant to have."""
import numpy as np
import pytest

from abhsf_amd import AbhsfMatrix, synth
from test_gpu_segments import CASES, check, with_integers

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
