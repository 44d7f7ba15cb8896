"""Performance cases: what a program does with this library through its public
classes (AbhsfMatrix, AbhsfBatch, DeltaMatrix), from one small SpMV to the
largest matrices of the benchmark.

A case is a dict: "op" (what is called), "family" and its size (the matrix),
and the options a program picks (block size, variant, precision, right-hand
sides, codec, beta).  The matrices are the families of abhsf_amd.synth
(5-point Laplacian, 27-point stencil, R-MAT, block mix, banded, random
blocks), generated on the GPU from the case and the seed; x, y and the values
are drawn as the benchmark draws them.

  spmv     y = A x + beta y on a built matrix
  spmm     Y = A X + beta Y, k right-hand sides, row-major
  sym      the same product with one stored triangle of a symmetric matrix
  delta    the delta-coded formats' product
  batch    one launch (a replayed graph) over many matrices
  convert  CSR -> ABHSF and the first product with the new matrix
"""
import math
import os

import torch

# A program that has loaded torch shares torch's HIP runtime with the library
# (two runtimes in one process do not see each other's streams); the package
# takes the runtime under ROCM_PATH/lib.
os.environ["ROCM_PATH"] = os.path.dirname(torch.__file__)

from abhsf_amd import AbhsfBatch, AbhsfMatrix, DeltaMatrix  # noqa: E402

DEV = "cuda"


# ---- the cases ---------------------------------------------------------------

def listed():
    return [
        # the smallest call: the 256^2 Laplacian of the reference's CPU path,
        # default block size; launch latency counts
        {"name": "laplacian256_spmv", "op": "spmv", "family": "laplacian", "size": 256, "s": 64, "variant": "auto",
         "precision": "f64", "beta": 0.0},
        # a 2-D grid in the fastest format for it (the tuner's pick)
        {"name": "laplacian1024_delta", "op": "delta", "family": "laplacian", "size": 1024, "codec": "u32_block",
         "beta": 0.0},
        # a 3-D grid operator inside a Krylov solver, default options
        {"name": "stencil160_spmv", "op": "spmv", "family": "stencil", "size": 160, "s": 64, "variant": "auto",
         "precision": "f64", "beta": 0.0},
        # the headline benchmark: R-MAT scale 22 at the tuner's pick, accumulating
        {"name": "rmat22_spmv", "op": "spmv", "family": "rmat", "size": 22, "ef": 16, "s": 256, "variant": "tiled",
         "precision": "f64", "beta": 1.0},
        # a graph with default options (no tuner)
        {"name": "rmat20_spmv_default", "op": "spmv", "family": "rmat", "size": 20, "ef": 16, "s": 64,
         "variant": "auto", "precision": "f64", "beta": 0.0},
        # the block-structured matrix at the tuner's pick, all four schemes' work
        {"name": "blockmix22_spmv", "op": "spmv", "family": "blockmix", "size": 1 << 22, "s": 32, "variant": "tiled",
         "precision": "f64", "beta": 1.0},
        # single-precision values with compensated sums
        {"name": "rmat20_spmv_f32", "op": "spmv", "family": "rmat", "size": 20, "ef": 16, "s": 256,
         "variant": "tiled", "precision": "f32", "beta": 0.0},
        # a symmetric operator, one triangle stored; an odd grid
        {"name": "stencil99_sym", "op": "sym", "family": "stencil", "size": 99, "s": 64, "variant": "auto",
         "precision": "f64", "beta": 0.0},
        # a block Krylov / multi-source step: 32 right-hand sides
        {"name": "stencil160_spmm_k32", "op": "spmm", "family": "stencil", "size": 160, "s": 64, "variant": "auto",
         "precision": "f64", "k": 32, "beta": 0.0},
        # a few right-hand sides on mixed structure, ragged size
        {"name": "blockmix_spmm_k8", "op": "spmm", "family": "blockmix", "size": 1000003, "s": 32, "variant": "auto",
         "precision": "f64", "k": 8, "beta": 1.0},
        # many small and medium matrices in one launch (the batch workload)
        {"name": "batch100_spmv", "op": "batch", "count": 100, "s": 32, "variant": "balanced", "beta": 0.0},
        # a matrix that is converted, used and dropped
        {"name": "rmat20_convert", "op": "convert", "family": "rmat", "size": 20, "ef": 16, "s": 64,
         "variant": "auto", "precision": "f64", "beta": 0.0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _matrix(rng, most):
    """A family and a size of at most `most` entries."""
    fam = rng.choice(["laplacian", "stencil", "rmat", "blockmix", "banded", "blocks"])
    if fam == "laplacian":
        return {"family": fam, "size": _log(rng, 32, min(2048, math.isqrt(most // 5)))}
    if fam == "stencil":
        return {"family": fam, "size": _log(rng, 16, min(160, int((most / 27) ** (1 / 3))))}
    if fam == "rmat":
        ef = rng.choice([8, 16])
        return {"family": fam, "size": rng.randint(12, min(22, int(math.log2(most / ef)))), "ef": ef}
    if fam == "blockmix":
        return {"family": fam, "size": _log(rng, 4096, min(1 << 22, int(most / 32.5)))}
    if fam == "banded":
        bw = rng.randint(4, 64)
        return {"family": fam, "size": _log(rng, 1000, min(1 << 20, most // (2 * bw + 1))), "bw": bw}
    bs, nbr = rng.choice([4, 8, 16, 32]), rng.randint(2, 8)
    return {"family": fam, "size": _log(rng, 1000, min(1 << 20, most // (bs * nbr))), "bs": bs, "nbr": nbr,
            "density": round(rng.uniform(0.05, 0.30), 3)}


def draw(rng):
    op = rng.choice(["spmv"] * 9 + ["spmm"] * 4 + ["sym"] * 2 + ["delta"] * 2 + ["batch"] + ["convert"] * 2)
    beta = float(rng.choice([0, 1]))
    if op == "batch":
        return {"op": op, "count": rng.randint(20, 100), "s": rng.choice([16, 32, 64]),
                "variant": rng.choice(["balanced", "tiled"]), "beta": 0.0}
    if op == "delta":  # the encoder runs on the host: smaller matrices
        return {"op": op, **_matrix(rng, 8 << 20), "codec": rng.choice(["varint", "u32_row", "u32_block"]),
                "beta": beta}
    s = rng.choice([8, 16, 32, 64, 128, 256])
    if op == "sym":
        fam = rng.choice(["laplacian", "stencil", "banded"])
        size = {"laplacian": _log(rng, 64, 2048), "stencil": _log(rng, 16, 120), "banded": _log(rng, 1000, 1 << 19)}
        return {"op": op, "family": fam, "size": size[fam], "bw": rng.randint(4, 64), "s": s, "variant": "auto",
                "precision": "f64", "beta": beta}
    precision = rng.choice(["f64"] * 4 + ["f32"])
    if op == "spmm":
        k = _log(rng, 2, 64)
        c = _matrix(rng, min(40 << 20, (100 << 25) // k))
        return {"op": op, **c, "s": min(s, 128), "variant": "auto", "precision": precision, "k": k, "beta": beta}
    if op == "convert":
        return {"op": op, **_matrix(rng, 16 << 20), "s": s, "variant": rng.choice(["auto", "tiled"]),
                "precision": precision, "beta": 0.0}
    return {"op": op, **_matrix(rng, 100 << 20), "s": s, "variant": rng.choice(["auto"] * 3 + ["tiled"] * 2 + ["panel"]),
            "precision": precision, "beta": beta}


# ---- matrices (CSR on the GPU) -------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _uniform(n, g):
    return torch.rand(n, device=DEV, dtype=torch.float64, generator=g) * 2.0 - 1.0


def _from_keys(m, n, key, g, normal):
    """CSR of the distinct keys r * n + c, with random values."""
    key = torch.unique(key)
    rows = torch.div(key, n, rounding_mode="floor")
    col = (key - rows * n).to(torch.int32)
    rp = torch.zeros(m + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(torch.bincount(rows, minlength=m), 0, out=rp[1:])
    nnz = key.numel()
    val = torch.randn(nnz, device=DEV, dtype=torch.float64, generator=g) if normal else _uniform(nnz, g)
    return m, n, rp, col, val


def _grid(dims, offsets, diag, lower):
    """A grid operator in natural ordering: `diag` on the diagonal, -1 else;
    lower: only the entries on and below the diagonal."""
    n = math.prod(dims)
    p = torch.arange(n, device=DEV)
    coord, q = [], p
    for d in reversed(dims):
        coord.insert(0, q % d)
        q = torch.div(q, d, rounding_mode="floor")
    cols, ok = [], []
    for off in offsets:
        step, inside = 0, torch.ones(n, dtype=torch.bool, device=DEV)
        for a, o, d in zip(coord, off, dims):
            step = step * d + o
            if o:
                inside &= (a + o >= 0) & (a + o < d)
        if lower and step > 0:
            continue
        cols.append((p + step).to(torch.int32))
        ok.append(inside)
    ok, cols = torch.stack(ok, 1), torch.stack(cols, 1)
    rp = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(ok.sum(1), 0, out=rp[1:])
    val = torch.where(cols == p.to(torch.int32)[:, None], diag, -1.0).to(torch.float64)
    return n, n, rp, cols[ok], val[ok]


def _rmat(scale, ef, g):
    n, ne = 1 << scale, ef << scale
    r = torch.zeros(ne, dtype=torch.int64, device=DEV)
    c = torch.zeros(ne, dtype=torch.int64, device=DEV)
    for _ in range(scale):
        u = torch.rand(ne, device=DEV, generator=g)
        r.mul_(2).add_(u >= 0.76)
        c.mul_(2).add_(((u >= 0.57) & (u < 0.76)) | (u >= 0.95))
    return _from_keys(n, n, r.mul_(n).add_(c), g, False)


def _block_mix(n, g):
    strips = (n + 31) // 32
    u = torch.rand(strips, device=DEV, generator=g)
    t32 = torch.arange(32, device=DEV)
    dense = torch.nonzero(u < 0.2).flatten()
    bc = torch.randint(0, strips, (dense.numel(), 3), device=DEV, generator=g)
    bc[:, 0] = dense
    r = (dense[:, None] * 32 + t32)[:, None, :, None]
    c = (bc[:, :, None] * 32 + t32)[:, :, None, :]
    keys = [torch.where((r < n) & (c < n), r * n + c, -1).flatten()]
    band = torch.nonzero((u >= 0.2) & (u < 0.5)).flatten()
    r = (band[:, None] * 32 + t32).flatten()[:, None]
    c = (torch.div(r, 8, rounding_mode="floor") - 1) * 8 + torch.arange(24, device=DEV)
    keys.append(torch.where((r < n) & (c >= 0) & (c < n), r * n + c, -1).flatten())
    scatter = torch.nonzero(u >= 0.5).flatten()
    r = (scatter[:, None] * 32 + t32).flatten()[:, None]
    c = torch.randint(0, n, (r.numel(), 12), device=DEV, generator=g)
    keys.append(torch.where(r < n, r * n + c, -1).flatten())
    key = torch.cat(keys)
    return _from_keys(n, n, key[key >= 0], g, True)


def _banded(n, bw, g, lower):
    r = torch.arange(n, device=DEV)[:, None]
    c = r + torch.arange(-bw, 1 if lower else bw + 1, device=DEV)
    ok = (c >= 0) & (c < n)
    rp = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(ok.sum(1), 0, out=rp[1:])
    col = c[ok].to(torch.int32)
    return n, n, rp, col, torch.randn(col.numel(), device=DEV, dtype=torch.float64, generator=g)


def _random_blocks(n, bs, nbr, density, g):
    nb = (n + bs - 1) // bs
    bc = torch.randint(0, nb, (nb, nbr), device=DEV, generator=g)
    bc[:, 0] = torch.arange(nb, device=DEV)
    t = torch.arange(bs, device=DEV)
    r = (torch.arange(nb, device=DEV)[:, None] * bs + t)[:, None, :, None]
    c = (bc[:, :, None] * bs + t)[:, :, None, :]
    keep = torch.rand(nb, nbr, bs, bs, device=DEV, generator=g) < density
    key = torch.where((r < n) & (c < n) & (keep | (r == c)), r * n + c, -1).flatten()
    return _from_keys(n, n, key[key >= 0], g, True)


def _csr(case, g, lower=False):
    fam, size = case["family"], case["size"]
    if fam == "laplacian":
        A = _grid([size] * 2, [(-1, 0), (0, -1), (0, 0), (0, 1), (1, 0)], 4.0, lower)
    elif fam == "stencil":
        A = _grid([size] * 3, [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)], 26.0, lower)
    elif fam == "rmat":
        A = _rmat(size, case["ef"], g)
    elif fam == "blockmix":
        A = _block_mix(size, g)
    elif fam == "banded":
        A = _banded(size, case["bw"], g, lower)
    else:
        A = _random_blocks(size, case["bs"], case["nbr"], case["density"], g)
    if case.get("precision") == "f32":  # a program with single-precision data
        A = A[:4] + (A[4].to(torch.float32).to(torch.float64),)
    return A


def _batch_members(case, seed, g):
    """Matrices of the batch workload: n log-uniform in [1e3, 2e5], one of
    four families.  Sizes and families are the same for every seed, so that
    the work is."""
    import random
    rng = random.Random(case["count"])
    for _ in range(case["count"]):
        n = _log(rng, 1e3, 2e5)
        fam = rng.choice(["laplacian", "banded", "rmat", "blocks"])
        yield _csr({"family": fam, "ef": 8, "bw": rng.randint(4, 64), "bs": rng.choice([4, 8, 16, 32]),
                    "nbr": rng.randint(2, 8), "density": rng.uniform(0.01, 0.30),
                    "size": {"laplacian": round(math.sqrt(n)), "rmat": round(math.log2(n))}.get(fam, n)}, g)


# ---- prepare and run ------------------------------------------------------------

def _abhsf(case, A):
    m, n, rp, col, val = A
    M = AbhsfMatrix(block_size=case["s"], variant=case["variant"], precision=case.get("precision", "f64"))
    M.from_csr(m, n, rp.data_ptr(), col.data_ptr(), val.data_ptr(), on_device=True, nnz=col.numel(),
               symmetry="symmetric" if case["op"] == "sym" else "general")
    return M


def _inputs(case, seed):
    """(A, x, y): the CSR arrays and the vectors (row-major n x k for spmm)."""
    g = _gen(seed)
    A = _csr(case, g, lower=case["op"] == "sym")
    k = case.get("k", 0)
    x = _uniform((A[1], k) if k else A[1], g)
    y = _uniform((A[0], k) if k else A[0], g)
    return A, x, y


def _batch_inputs(case, seed):
    """Members with x and y as slices of one array each (256-byte aligned)."""
    g = _gen(seed)
    mats = list(_batch_members(case, seed, g))
    at = [0]
    for A in mats:
        at.append(at[-1] + (A[0] + 31) // 32 * 32)
    return mats, at, _uniform(at[-1], g)


def prepare(case, seed):
    op = case["op"]
    if op == "batch":
        mats, at, x = _batch_inputs(case, seed)
        y = torch.zeros_like(x)
        torch.cuda.synchronize()
        members = [_abhsf(case, A) for A in mats]
        B = AbhsfBatch(members)
        B.set_vectors([x.data_ptr() + 8 * o for o in at[:-1]], [y.data_ptr() + 8 * o for o in at[:-1]])
        return {"case": case, "batch": B, "x": x, "y": y}
    A, x, y = _inputs(case, seed)
    state = {"case": case, "x": x, "y": y}
    torch.cuda.synchronize()  # the conversion reads the arrays
    if op == "convert":
        state["A"] = A
    elif op == "delta":
        M = DeltaMatrix(codec=case["codec"])
        M.from_csr(A[0], A[1], A[2].data_ptr(), A[3].data_ptr(), A[4].data_ptr(), on_device=True, nnz=A[3].numel())
        state["M"] = M
    else:
        state["M"] = _abhsf(case, A)
    return state


def run(state):
    case, y = state["case"], state["y"]
    op = case["op"]
    if op == "batch":
        state["batch"].spmv_async(1.0, case["beta"], graph=True)
        return y
    x = state["x"]
    if op == "spmm":
        k = case["k"]
        state["M"].spmm_async(k, 1.0, x.data_ptr(), k, case["beta"], y.data_ptr(), k)
        return y
    if op == "convert":
        M = _abhsf(case, state["A"])
        M.spmv_async(1.0, x.data_ptr(), case["beta"], y.data_ptr())
        st = M.stats()
        return {"y": y, "blocks": [int(v) for v in st["blocks"].values()],
                "bits": [int(st["smf_bits_preproc"]), int(st["smf_bits_msmf"])]}
    state["M"].spmv_async(1.0, x.data_ptr(), case["beta"], y.data_ptr())
    return y


# ---- work and exact results ------------------------------------------------------

def _entries(case):
    """(rows, stored entries); the random families' expected counts."""
    fam, size = case["family"], case["size"]
    if fam == "laplacian":
        m, nnz = size * size, 5 * size * size - 4 * size
    elif fam == "stencil":
        m, nnz = size ** 3, (3 * size - 2) ** 3
    elif fam == "rmat":
        m, nnz = 1 << size, 0.97 * (case["ef"] << size)
    elif fam == "blockmix":
        m, nnz = size, 32.4 * size
    elif fam == "banded":
        m, nnz = size, size * (2 * case["bw"] + 1)
    else:
        m, nnz = size, size * case["nbr"] * case["bs"] * case["density"]
    return m, (nnz + m) / 2 if case["op"] == "sym" else nnz


def work(case):
    """Values, one local index per entry and the vectors, once each; for a
    conversion the CSR arrays read and the new storage written."""
    if case["op"] == "batch":
        import random
        rng = random.Random(case["count"])
        m = nnz = 0
        for _ in range(case["count"]):
            n = _log(rng, 1e3, 2e5)
            fam = rng.choice(["laplacian", "banded", "rmat", "blocks"])
            bw, bs, nbr, d = rng.randint(4, 64), rng.choice([4, 8, 16, 32]), rng.randint(2, 8), rng.uniform(0.01, 0.30)
            size = {"laplacian": round(math.sqrt(n)), "rmat": round(math.log2(n))}.get(fam, n)
            mi, zi = _entries({"op": "spmv", "family": fam, "size": size, "ef": 8, "bw": bw, "bs": bs, "nbr": nbr,
                               "density": d})
            m, nnz = m + mi, nnz + zi
    else:
        m, nnz = _entries(case)
    k = case.get("k", 1)
    index = 1 if case.get("s", 64) <= 16 else 2
    entry = (4 if case.get("precision") == "f32" else 8) + (4 if case["op"] == "delta" else index)
    vectors = m * k * 8 * (2 + (case["beta"] != 0.0))
    flops = 2 * nnz * k * (2 if case["op"] == "sym" else 1)
    if case["op"] == "convert":
        return {"bytes": 8 * m + 12 * nnz + nnz * entry + vectors, "flops": flops}
    return {"bytes": nnz * entry + vectors, "flops": flops}


def _product(A, x, transposed=False):
    """A x in 64 bits (transposed: A^T x without the diagonal)."""
    m, n, rp, col, val = A
    rows = torch.repeat_interleave(torch.arange(m, device=DEV), rp[1:] - rp[:-1])
    c = col.long()
    if transposed:
        off = rows != c
        rows, c, val = c[off], rows[off], val[off]
    if x.dim() == 1:
        return torch.zeros(m, dtype=torch.float64, device=DEV).index_add_(0, rows, val * x[c])
    return torch.stack([torch.zeros(m, dtype=torch.float64, device=DEV).index_add_(0, rows, val * x[:, j].contiguous()[c])
                        for j in range(x.shape[1])], 1)


def exact(case, seed):
    if case["op"] == "batch":
        mats, at, x = _batch_inputs(case, seed)
        y = torch.zeros_like(x)
        for A, o in zip(mats, at):
            y[o:o + A[0]] = _product(A, x[o:o + A[1]])
        return y
    A, x, y = _inputs(case, seed)
    out = _product(A, x)
    if case["op"] == "sym":
        out += _product(A, x, transposed=True)
    if case["beta"] != 0.0:
        out += case["beta"] * y
    if case["op"] == "convert":
        return {"y": out, "blocks": [None] * 4, "bits": [None] * 2}
    return out
