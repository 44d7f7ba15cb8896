"""The scratch a conversion keeps goes back to the device on request."""
import pytest

import abhsf_amd
from abhsf_amd import AbhsfMatrix, synth

pytestmark = pytest.mark.gpu


def test_trim_returns_the_memory(gpu):
    A = synth.rmat(17, 16, seed=1)
    print("case scratch trim", flush=True)
    M = AbhsfMatrix(block_size=64)
    M.from_csr(A.m, A.n, A.rowptr, A.col, A.val)
    M.release()
    # (what the runtime does with freed memory is its own: the free memory it
    # reports rises by less.  That the buffers are freed is test_scratch_cpu's.)
    freed = abhsf_amd.scratch_trim()
    assert freed > 20 * A.nnz  # rows, keys and their order alone
    assert abhsf_amd.scratch_trim() == 0
    M = AbhsfMatrix(block_size=64)  # and the next conversion works
    M.from_csr(A.m, A.n, A.rowptr, A.col, A.val)
    assert M.stats()["nnz"] == A.nnz
    M.release()
