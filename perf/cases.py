"""The work that users of this library have it do, as measurable cases.

``listed()`` names the cases, ``draw()`` gives further ones of the same
ranges, ``prepare()`` builds what a program holds before the call (matrix
uploaded, vectors on the GPU), ``run()`` is one pass through the public entry
points and ``exact()`` the same result in 64 bits from plain torch / numpy.

Kinds of case (every SpMV is y += A x, FP32 accumulation):

  dia       27-point stencil of a structured grid as a DIA part, in FP32 or
            with one of the value codecs
  bsr       3x3-block matrix (three unknowns per mesh node) as a BSR part, in
            FP32 or with a codec
  ell       scattered columns, equal row lengths, as an x-tiled ELL part
  csr       irregular rows as a CSR part: power-law rows with scattered
            columns x-tiled, mesh-like rows near the diagonal as adaptive row
            blocks
  coo       mesh-like rows as a COO part (triplets straight from assembly)
  block44   dense 4x4 blocks in one of the reference's block formats
  cocktail  a matrix through the analyzer: partition, upload, do_spmv
  iterate   power_iterate: the matrix-power loop of the reference's example,
            here explicit heat steps on a 2D grid
  batch     many matrices with 1, 4 or 16 right-hand sides in one launch
  mlp       training steps of the format selector's network
"""
import ctypes
import math

import numpy as np
import torch

from clspmv_amd import _lib as L
from clspmv_amd import cocktail as K
from clspmv_amd import matrix as M
from clspmv_amd.batch import Batch
from clspmv_amd.selector import Mlp

CODECS = {"fp32": 0, "bf16x2": L.VAL_BF16X2, "fp16": L.VAL_FP16_ROW, "fp8": L.VAL_FP8_SLICE, "int16": L.VAL_I16_ROW}
VALUE_BYTES = {"fp32": 4, "bf16x2": 4, "fp16": 2, "fp8": 1, "int16": 2}
TABLES = {"mi355x": K.MI355X_TABLES, "reference": K.REFERENCE_TABLES}


def listed():
    return [
        # the smallest calls: a short matrix-power loop on a 256 x 256 grid
        {"name": "iterate_heat_256", "kind": "iterate", "nx": 256, "ny": 256, "iterations": 16},
        # a 128^3 27-point stencil with two-byte values
        {"name": "dia_stencil_int16", "kind": "dia", "n": 128, "codec": "int16"},
        # a smaller stencil through the analyzer (ordinary size, odd edge)
        {"name": "cocktail_stencil_75", "kind": "cocktail", "matrix": "stencil", "n": 75, "tables": "mi355x"},
        # the widest scattered matrix of the benchmark: 4M rows of 32
        {"name": "ell_uniform_4m", "kind": "ell", "rows": 4194304, "per_row": 32},
        # power-law rows (graphs), one of them 50,000 entries long
        {"name": "csr_zipf_2m", "kind": "csr", "matrix": "zipf", "rows": 2097152, "mean": 16, "longest": 50000, "method": 4},
        # an irregular mesh in CSR, the default format of such matrices
        {"name": "csr_mesh_1m", "kind": "csr", "matrix": "mesh", "rows": 1000003, "mean": 18, "method": 1},
        # the same kind of matrix as row-sorted triplets
        {"name": "coo_mesh_500k", "kind": "coo", "rows": 500009, "mean": 12},
        # three unknowns per node: 1M block rows of 9 dense 3x3 blocks
        {"name": "bsr_blocks_1m", "kind": "bsr", "block_rows": 1048576, "blocks": 9, "band": 5000, "codec": "fp32"},
        # 4x4 blocks in the reference's BCSR
        {"name": "bcsr_blocks_100k", "kind": "block44", "block_rows": 100003, "blocks": 9, "band": 2000, "format": "bcsr"},
        # a composite (band, blocks, power-law rows) through the analyzer's plan
        {"name": "cocktail_composite_4m", "kind": "cocktail", "matrix": "composite", "n": 4194304, "tables": "mi355x"},
        # a service's mixed batch: 24 matrices of 2^10 .. 2^18 rows, k = 1, 4, 16
        {"name": "batch_24", "kind": "batch", "count": 24, "log2_min": 10, "log2_max": 18},
        # training the selector's network on its own dataset's shape
        {"name": "mlp_train_1920", "kind": "mlp", "samples": 1920, "features": 24, "hidden": 128, "classes": 22, "steps": 20},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dia", "bsr", "ell", "csr", "csr", "coo", "block44", "cocktail", "cocktail", "iterate", "batch", "mlp"])
    if kind == "dia":
        return {"kind": kind, "n": _log(rng, 12, 128), "codec": rng.choice(sorted(CODECS))}
    if kind == "bsr":
        return {"kind": kind, "block_rows": _log(rng, 2000, 1048576), "blocks": rng.randint(3, 9),
                "band": rng.choice([16, 200, 5000]), "codec": rng.choice(sorted(CODECS))}
    if kind == "ell":
        return {"kind": kind, "rows": _log(rng, 60000, 4194304), "per_row": rng.randint(8, 32)}
    if kind == "csr":
        if rng.random() < 0.4:
            rows = _log(rng, 60000, 2097152)
            return {"kind": kind, "matrix": "zipf", "rows": rows, "mean": rng.randint(6, 16),
                    "longest": min(50000, rows // 4), "method": 4}
        return {"kind": kind, "matrix": "mesh", "rows": _log(rng, 2000, 1500000), "mean": rng.randint(4, 40), "method": 1}
    if kind == "coo":
        return {"kind": kind, "rows": _log(rng, 2000, 1000000), "mean": rng.randint(3, 30)}
    if kind == "block44":
        return {"kind": kind, "block_rows": _log(rng, 2000, 200000), "blocks": rng.randint(3, 16),
                "band": rng.choice([16, 200, 2000]), "format": rng.choice(["bcsr", "bell", "sbell"])}
    if kind == "cocktail":
        matrix = rng.choice(["stencil", "composite", "mesh", "blocks4", "blocks3"])
        n = {"stencil": lambda: _log(rng, 12, 100), "composite": lambda: 16 * _log(rng, 256, 131072),
             "mesh": lambda: _log(rng, 2000, 500000), "blocks4": lambda: _log(rng, 1000, 100000),
             "blocks3": lambda: _log(rng, 1000, 200000)}[matrix]()
        return {"kind": kind, "matrix": matrix, "n": n, "tables": rng.choice(sorted(TABLES))}
    if kind == "iterate":
        return {"kind": kind, "nx": _log(rng, 20, 700), "ny": _log(rng, 20, 700), "iterations": rng.randint(4, 40)}
    if kind == "batch":
        lo = rng.randint(8, 12)
        return {"kind": kind, "count": _log(rng, 3, 24), "log2_min": lo, "log2_max": rng.randint(lo + 2, 18)}
    return {"kind": kind, "samples": _log(rng, 50, 2400), "features": 24, "hidden": rng.choice([64, 96, 128]),
            "classes": rng.randint(12, 22), "steps": rng.randint(5, 20)}


# ------------------------------------------------------------------ matrices

_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = M.Context(0)
    return _ctx


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _mesh(rows, mean, seed):
    """Rows of mean/2 .. 3 mean/2 distinct sorted columns around the diagonal
    (a mesh in a bandwidth-reducing order), N(0,1) values."""
    g = _generator(seed)
    lo, hi = max(1, mean // 2), max(2, mean + mean // 2)
    count = torch.randint(lo, hi + 1, (rows,), device="cuda", generator=g)
    row = torch.repeat_interleave(torch.arange(rows, device="cuda"), count)
    reach = max(4, int(4 * rows ** 0.5 / mean))
    step = torch.cumsum(torch.randint(1, reach, row.shape, device="cuda", generator=g), 0)
    first = torch.cumsum(count, 0) - count
    col = row - (mean * reach) // 4 + step - step[first][row]
    keep = (col >= 0) & (col < rows)
    row, col = row[keep], col[keep]
    val = torch.randn(row.shape, device="cuda", generator=g)
    return M.CooMatrix.from_arrays(row.int().cpu().numpy(), col.int().cpu().numpy(), val.cpu().numpy(), rows, rows)


def _heat(nx, ny):
    """Explicit heat step on an nx x ny grid: y += A x with A = -0.2 times
    the 5-point Laplacian, so that the iteration stays bounded."""
    coo = M.gen_laplacian2d(nx, ny)
    coo.data[:] *= np.float32(-0.2)
    return coo


def _batch_matrices(case, seed):
    out = []
    n, lo, hi = case["count"], case["log2_min"], case["log2_max"]
    for i in range(n):
        rows = int(2 ** (lo + (hi - lo) * ((7 * i) % n + 0.5) / n))
        k = (1, 4, 16)[i % 3]
        kind = ("stencil", "uniform", "zipf", "blocks")[i % 4]
        s = seed * 1009 + i
        if kind == "stencil":
            coo = M.gen_stencil27(max(4, round(rows ** (1 / 3))), s)
        elif kind == "uniform":
            coo = M.gen_uniform_rows(rows, min(32, rows), s)
        elif kind == "zipf":
            coo = M.gen_zipf_rows(rows, 1.8, 16.0, max(1, min(50000, rows // 2)), s)
        else:
            coo = M.gen_block_rows(max(16, rows // 3), 3, 9, 5000, s)
        out.append((kind, coo, k))
    return out


def _matrix(case, seed):
    kind = case["kind"]
    if kind == "dia":
        return M.gen_stencil27(case["n"], seed)
    if kind == "bsr":
        return M.gen_block_rows(case["block_rows"], 3, case["blocks"], case["band"], seed)
    if kind == "ell":
        return M.gen_uniform_rows(case["rows"], case["per_row"], seed)
    if kind == "csr" and case["matrix"] == "zipf":
        return M.gen_zipf_rows(case["rows"], 1.8, float(case["mean"]), case["longest"], seed)
    if kind in ("csr", "coo"):
        return _mesh(case["rows"], case["mean"], seed)
    if kind == "block44":
        return M.gen_block_rows(case["block_rows"], 4, case["blocks"], case["band"], seed)
    if kind == "iterate":
        return _heat(case["nx"], case["ny"])
    assert kind == "cocktail"
    if case["matrix"] == "stencil":
        return M.gen_stencil27(case["n"], seed)
    if case["matrix"] == "composite":
        return M.gen_cocktail_composite(case["n"], seed)
    if case["matrix"] == "mesh":
        return _mesh(case["n"], 14, seed)
    if case["matrix"] == "blocks4":
        return M.gen_block_rows(case["n"], 4, 9, 1000, seed)
    return M.gen_block_rows(case["n"], 3, 9, 1000, seed)


def _vectors(coo, seed):
    return M.gen_vector(coo.width, seed + 1), M.gen_vector(coo.height, seed + 2)


def _training_set(case, seed):
    """Standardised features, labels that depend on them, He-uniform
    initial parameters (W1, b1, W2, b2, W3, b3)."""
    r = np.random.default_rng(seed)
    n, d, h, c = case["samples"], case["features"], case["hidden"], case["classes"]
    x = r.standard_normal((n, d)).astype(np.float32)
    label = np.argmax(x @ r.standard_normal((d, c)) + r.standard_normal((n, c)), axis=1).astype(np.int32)

    def weights(a, b):
        return r.uniform(-1.0, 1.0, a * b) * math.sqrt(6.0 / a)

    p = np.concatenate([weights(d, h), np.zeros(h), weights(h, h), np.zeros(h), weights(h, c), np.zeros(c)])
    return x, label, p.astype(np.float32)


# ------------------------------------------------------------------ states


class _DeviceFloats:
    """A device buffer of a library object as torch sees it; keeps the object,
    whose memory it is."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (int(ptr.value), False),
                                         "version": 2}


def _tensor(owner, ptr, *shape):
    t = torch.as_tensor(_DeviceFloats(owner, ptr, shape), device="cuda")
    t.owner = owner  # the buffer lives as long as the tensor that shows it
    return t


def _part(case, coo):
    kind, ctx = case["kind"], _context()
    if kind == "dia":
        if case["codec"] == "fp32":
            return M.Part(ctx, L.FMT_DIA, M.coo2dia(coo))
        return M.MixedPart(ctx, L.FMT_DIA, M.coo2dia(coo, 256), CODECS[case["codec"]])
    if kind == "bsr":
        bsr = M.coo2bsr(coo, 3, 3)
        if case["codec"] == "fp32":
            return M.Part(ctx, L.FMT_BSR, bsr)
        return M.MixedPart(ctx, L.FMT_BSR, bsr, CODECS[case["codec"]])
    if kind == "ell":
        return M.Part(ctx, L.FMT_ELL, M.coo2ell(coo), 4)
    if kind == "csr":
        return M.Part(ctx, L.FMT_CSR_VECTOR, M.coo2csr(coo), case["method"])
    if kind == "coo":
        return M.Part(ctx, L.FMT_COO, coo)
    if case["format"] == "bcsr":
        return M.Part(ctx, L.FMT_BCSR, M.coo2b4csr(coo, 4, 4))
    if case["format"] == "bell":
        return M.Part(ctx, L.FMT_BELL, M.coo2b4ell(coo, 4, 4))
    return M.Part(ctx, L.FMT_SBELL, M.coo2sbell(coo, 4, 4))


def prepare(case, seed):
    kind, ctx = case["kind"], _context()
    if kind == "mlp":
        x, label, p = _training_set(case, seed)
        net = Mlp(ctx, case["features"], case["hidden"], case["classes"])
        net.set_params(p)
        return {"kind": kind, "net": net, "x": x, "label": label, "steps": case["steps"]}
    if kind == "batch":
        mats, ks, data = [], [], []
        for name, coo, k in _batch_matrices(case, seed):
            # dense blocks with several right-hand sides go to the matrix cores
            mats.append(M.coo2bsr(coo, 3, 3) if name == "blocks" and k > 1 else M.coo2csr(coo))
            ks.append(k)
            data.append((coo.width, coo.height))
        b = Batch(ctx, mats, ks)
        ys = []
        for i, (w, h) in enumerate(data):
            b.set_x(i, M.gen_vector(w * ks[i], seed + 2 * i + 1))
            b.set_y(i, M.gen_vector(h * ks[i], seed + 2 * i + 2))
            px, py = ctypes.c_void_p(), ctypes.c_void_p()
            L.check(L.lib().clspmv_batch_buffers(b.h, i, ctypes.byref(px), ctypes.byref(py)), "batch_buffers")
            ys.append(_tensor(b, py, h, ks[i]))
        return {"kind": kind, "batch": b, "y": ys}
    coo = _matrix(case, seed)
    x, y = _vectors(coo, seed)
    if kind in ("cocktail", "iterate"):
        tables = K.BenchTables(TABLES[case.get("tables", "mi355x")])
        gpu = K.GpuCocktail(ctx, K.Plan.analyze(coo, tables), x, x if kind == "iterate" else y)
        return {"kind": kind, "gpu": gpu, "y": _tensor(gpu, gpu.buffers()[1], coo.height),
                "iterations": case.get("iterations", 1)}
    part = _part(case, coo)
    return {"kind": kind, "part": part, "x": torch.from_numpy(x).cuda(), "y": torch.from_numpy(y).cuda()}


def run(state):
    kind = state["kind"]
    if kind == "mlp":
        loss = state["net"].train(state["x"], state["label"], steps=state["steps"])
        return {"loss": float(loss), "params": state["net"].get_params()}
    if kind == "batch":
        state["batch"].run(1)
    elif kind == "cocktail":
        state["gpu"].do_spmv(1)
    elif kind == "iterate":
        L.check(L.lib().clspmv_power_iterate(state["gpu"].h, state["iterations"]), "power_iterate")
    else:
        L.check(L.lib().clspmv_part_spmv(state["part"].h, state["x"].data_ptr(), state["y"].data_ptr(), 1), "part_spmv")
    return state["y"]


# ------------------------------------------------------------------ work


def _entries(case):
    """(rows, nonzeros) of the case's matrix; random row lengths by their mean."""
    kind = case["kind"]
    matrix = case.get("matrix")
    if kind == "dia" or matrix == "stencil":
        return case["n"] ** 3, (3 * case["n"] - 2) ** 3
    if kind in ("bsr", "block44"):
        b = 3 if kind == "bsr" else 4
        return b * case["block_rows"], b * b * case["blocks"] * case["block_rows"]
    if kind == "ell":
        return case["rows"], case["rows"] * case["per_row"]
    if kind in ("csr", "coo"):
        return case["rows"], case["rows"] * case["mean"]
    if kind == "iterate":
        return case["nx"] * case["ny"], 5 * case["nx"] * case["ny"]
    n = case["n"]
    if matrix == "composite":
        return n, n // 4 * 9 + n // 4 * 24 + n // 2 * 12
    if matrix == "mesh":
        return n, 14 * n
    b = 4 if matrix == "blocks4" else 3
    return b * n, 9 * b * b * n


def work(case):
    """Bytes of the matrix as its format has to hold it (values, and columns
    where they are not implied), of x once and of y read and written."""
    kind = case["kind"]
    if kind == "mlp":
        d, h, c = case["features"], case["hidden"], case["classes"]
        weights = d * h + h * h + h * c
        steps = case["steps"]
        return {"bytes": 4 * (case["samples"] * (d + 1) + steps * 7 * (weights + 2 * h + c)),
                "flops": 6 * case["samples"] * weights * (steps + 1)}
    if kind == "batch":
        n, lo, hi = case["count"], case["log2_min"], case["log2_max"]
        total, flops = 0, 0
        for i in range(n):
            rows = int(2 ** (lo + (hi - lo) * ((7 * i) % n + 0.5) / n))
            k, nnz = (1, 4, 16)[i % 3], rows * (27, 32, 16, 27)[i % 4]
            matrix = nnz * (40 / 9) if i % 4 == 3 and k > 1 else 8 * nnz + 4 * rows
            total += matrix + 12 * rows * k
            flops += 2 * nnz * k
        return {"bytes": total, "flops": flops}
    rows, nnz = _entries(case)
    vectors = 12 * rows
    if kind == "dia":
        matrix = nnz * VALUE_BYTES[case["codec"]]
    elif kind == "bsr":
        matrix = nnz * VALUE_BYTES[case["codec"]] + nnz // 9 * 2
    elif kind == "block44":
        matrix = 4 * nnz + nnz // 16 * 4
    elif kind == "coo":
        matrix = 12 * nnz
    elif kind in ("ell", "csr"):
        matrix = 8 * nnz + (4 * rows if kind == "csr" else 0)
    elif kind == "iterate":
        return {"bytes": case["iterations"] * (4 * nnz + vectors), "flops": case["iterations"] * 2 * nnz}
    elif case["matrix"] == "stencil":
        matrix = 4 * nnz
    elif case["matrix"] == "composite":
        matrix = rows // 4 * 9 * 8 + rows // 4 * 24 * 4 + rows // 4 * 6 + rows // 2 * 12 * 8
    elif case["matrix"] == "mesh":
        matrix = 8 * nnz + 4 * rows
    else:
        b = 4 if case["matrix"] == "blocks4" else 3
        matrix = 4 * nnz + nnz // (b * b) * 4
    return {"bytes": matrix + vectors, "flops": 2 * nnz}


# ------------------------------------------------------------------ 64 bits


def _product(coo, x):
    """A x in 64 bits; x (width) or (width, k)."""
    row = torch.from_numpy(np.array(coo.row_id)).cuda().long()
    col = torch.from_numpy(np.array(coo.col_id)).cuda().long()
    val = torch.from_numpy(np.array(coo.data)).cuda().double()
    x = x if isinstance(x, torch.Tensor) else torch.from_numpy(np.array(x, np.float64)).cuda()
    y = torch.zeros((coo.height,) + tuple(x.shape[1:]), dtype=torch.float64, device="cuda")
    step = 1 << 24
    for a in range(0, row.numel(), step):
        s = slice(a, a + step)
        p = val[s].reshape((-1,) + (1,) * (x.dim() - 1)) * x[col[s]]
        y.index_add_(0, row[s], p)
    return y


def _train_exact(case, seed):
    x, label, p = _training_set(case, seed)
    n, d, h, c = case["samples"], case["features"], case["hidden"], case["classes"]
    x, p = x.astype(np.float64), p.astype(np.float64)
    lr, b1, b2, eps = (float(np.float32(v)) for v in (2e-3, 0.9, 0.999, 1e-8))  # the defaults, as the call takes them
    at = np.cumsum([0, d * h, h, h * h, h, h * c, c])
    shape = [(d, h), (h,), (h, h), (h,), (h, c), (c,)]

    def both(p):
        w1, a1, w2, a2, w3, a3 = (p[at[i]:at[i + 1]].reshape(shape[i]) for i in range(6))
        h1 = np.maximum(x @ w1 + a1, 0.0)
        h2 = np.maximum(h1 @ w2 + a2, 0.0)
        z = h2 @ w3 + a3
        z = z - z.max(axis=1, keepdims=True)
        log_sum = np.log(np.exp(z).sum(axis=1, keepdims=True))
        loss = float(np.mean(log_sum[:, 0] - z[np.arange(n), label]))
        dz = np.exp(z - log_sum)
        dz[np.arange(n), label] -= 1.0
        dz /= n
        d2 = (dz @ w3.T) * (h2 > 0)
        d1 = (d2 @ w2.T) * (h1 > 0)
        g = [x.T @ d1, d1.sum(0), h1.T @ d2, d2.sum(0), h2.T @ dz, dz.sum(0)]
        return loss, np.concatenate([v.reshape(-1) for v in g])

    m, v = np.zeros_like(p), np.zeros_like(p)
    for t in range(1, case["steps"] + 1):
        _, g = both(p)
        m = b1 * m + (1 - b1) * g
        v = b2 * v + (1 - b2) * g * g
        p = p - lr * (m / (1 - b1 ** t)) / (np.sqrt(v / (1 - b2 ** t)) + eps)
    return {"loss": both(p)[0], "params": p}


def exact(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        return _train_exact(case, seed)
    if kind == "batch":
        out = []
        for i, (_, coo, k) in enumerate(_batch_matrices(case, seed)):
            x = M.gen_vector(coo.width * k, seed + 2 * i + 1).astype(np.float64).reshape(coo.width, k)
            y = M.gen_vector(coo.height * k, seed + 2 * i + 2).astype(np.float64).reshape(coo.height, k)
            out.append(torch.from_numpy(y).cuda() + _product(coo, x))
        return out
    coo = _matrix(case, seed)
    x, y = (torch.from_numpy(v.astype(np.float64)).cuda() for v in _vectors(coo, seed))
    if kind != "iterate":
        return y + _product(coo, x)
    y = x.clone()
    for _ in range(case["iterations"]):
        y = y + _product(coo, x)
        x = y
    return y
