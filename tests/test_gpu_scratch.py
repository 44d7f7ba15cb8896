"""The conversion's scratch, kept from one build to the next: builds of
changing sizes, and builds from several threads on streams of their own, give
the oracle's arrays byte for byte and exact products (heavy strips' units are
cut on the device)."""
import threading

import numpy as np
import pytest

from abhsf_amd import AbhsfMatrix, hip, synth
from abhsf_amd.hip import DeviceArray
from oracle import pyoracle

pytestmark = pytest.mark.gpu


def check(A, s, stream=None, variant="balanced"):
    M = AbhsfMatrix(block_size=s, variant=variant, stream=stream)
    M.from_csr(A.m, A.n, A.rowptr, A.col, A.val)
    if variant == "balanced":
        oa, ga = pyoracle.Abhsf(A.m, A.n, A.rowptr, A.col, A.val, s.bit_length() - 1).arrays(), M.export_all()
        assert [k for k in oa if not np.array_equal(oa[k], ga[k])] == []
    x = np.random.default_rng(s).integers(-8, 9, A.n).astype(np.float64)
    dx, dy = DeviceArray.from_numpy(x), DeviceArray.zeros(A.m)
    M.spmv_async(1.0, dx, 0.0, dy)
    M.synchronize()
    ok = np.array_equal(dy.numpy(), pyoracle.csr_spmv(A.rowptr, A.col, A.val, x))
    M.release()
    assert ok


def integers(A, seed):
    v = np.random.default_rng(seed).integers(1, 9, A.nnz).astype(np.float64)
    return synth.Csr(A.m, A.n, A.rowptr, A.col, v, A.name)


@pytest.mark.parametrize("variant", ["balanced", "tiled"])
def test_sizes_up_and_down(gpu, variant):
    """4095 / 4096 / 4097 entries (one workgroup of the key pass and its
    edges), heavy strips, few entries over many rows."""
    mats = [integers(synth.rmat(16, 16, seed=1), 1), integers(synth.random_sparse(50, 60, 0.3, seed=2), 2)]
    for z in (4095, 4096, 4097):
        key = np.sort(np.random.default_rng(z).choice(3000 * 3000, z, replace=False))
        mats.append(integers(synth.from_triplets(3000, 3000, key // 3000, key % 3000, np.ones(z)), z))
    key = np.sort(np.random.default_rng(9).choice(200000 * 1000, 9000, replace=False))
    mats.append(integers(synth.from_triplets(200000, 1000, key // 1000, key % 1000, np.ones(9000)), 3))
    mats.append(integers(synth.rmat(15, 16, seed=4), 4))
    for A in mats:
        for s in (16, 64, 256):
            print(f"case scratch {A.m}x{A.n} nnz={A.nnz} s={s} {variant}", flush=True)
            check(A, s, variant=variant)


def test_threads(gpu):
    mats = [integers(synth.rmat(14, 16, seed=i), i) for i in range(4)]
    failed = []

    def work(i):
        try:
            st = hip.Stream()
            for rep in range(4):
                check(mats[(i + rep) % 4], (32, 64)[rep % 2], st)
        except BaseException as e:  # noqa: BLE001 (reported below)
            failed.append(repr(e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert failed == []
