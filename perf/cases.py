"""The work users have this package do, as cases that can be timed and compared.

Every case goes through the public entry points the way a program calls them: an operand that a
program keeps (a graph, a mask, a weight matrix) is made in ``prepare``, one pass over it is ``run``.
The kinds are the applications the package serves: neighbourhood aggregation and graph convolution,
weight-sparse and activation-sparse layers, sampled products, sparse attention (fused in bf16 and fp32,
and composed of its three steps for masks the fused kernels do not take), sparse x sparse products and
matrix-vector products of iterative solvers.  ``draw`` spreads the sizes over the range of each kind.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import scorch_amd as scorch
from scorch_amd import STensor
from scorch_amd import scorch_ops_hip as ops

ZIPF = 2.1              # exponent of the graphs' out-degrees
MAX_DEGREE = 50_000


# ---- the cases --------------------------------------------------------------------------------
def listed():
    return [
        # aggregation over a citation-sized graph: one short launch, latency is everything
        {"name": "spmm_small_graph", "kind": "spmm", "pattern": "graph", "rows": 2708, "per_row": 4, "width": 16,
         "dtype": "f32", "format": "csr"},
        # a product of ordinary size with a uniformly sparse matrix
        {"name": "spmm_uniform_4096", "kind": "spmm", "pattern": "uniform", "rows": 4096, "per_row": 41, "width": 64,
         "dtype": "f32", "format": "csr"},
        # an edge list in coordinate form, ragged in every size
        {"name": "spmm_edge_list_odd", "kind": "spmm", "pattern": "graph", "rows": 50_021, "per_row": 11, "width": 37,
         "dtype": "f32", "format": "coo"},
        # aggregation over a power-law graph of a million nodes
        {"name": "spmm_graph_1m", "kind": "spmm", "pattern": "graph", "rows": 1 << 20, "per_row": 16, "width": 128,
         "dtype": "f32", "format": "csr"},
        # a two-layer graph convolution through the fusing decorator, narrow odd classifier at the end
        {"name": "gcn_two_layers", "kind": "gcn", "rows": 19_717, "per_row": 4, "features": 500, "hidden": 16,
         "classes": 3},
        # an autoencoder whose two weight matrices are 95 % sparse: matrix times transposed activations
        {"name": "sparse_weight_layers", "kind": "sparse_weights", "wide": 4096, "narrow": 1024, "batch": 256,
         "density": 0.05},
        # decoder of a sparse autoencoder: new top-k activations on every call, the same weights
        {"name": "topk_decoder", "kind": "decoder", "batch": 4096, "latents": 16_384, "width": 4096, "active": 32},
        # dot products of two embeddings at the stored positions of a mask
        {"name": "sddmm_65536", "kind": "sddmm", "rows": 65_536, "cols": 65_536, "per_row": 64, "depth": 64,
         "format": "csr", "unit": True},
        # long-context attention in bf16, local window and strided blocks
        {"name": "attention_bf16_8192", "kind": "attention", "mask": "blocks", "tokens": 8192, "heads": 16, "dim": 64,
         "dtype": "bf16", "fused": True},
        # a sequence of odd length with a sliding window and a global token: the three steps, fp32
        {"name": "attention_steps_odd", "kind": "attention", "mask": "window", "tokens": 3001, "heads": 8, "dim": 64,
         "dtype": "f32", "fused": False},
        # two-hop neighbourhoods of a power-law graph
        {"name": "spgemm_two_hop", "kind": "spgemm", "rows": 131_072, "per_row": 16, "dtype": "f32"},
        # one step of an iterative method in double precision on a large graph
        {"name": "spmv_f64_1m", "kind": "spmv", "pattern": "graph", "rows": 1 << 20, "per_row": 16, "dtype": "f64"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("spmm", "spmm", "gcn", "sparse_weights", "decoder", "sddmm", "attention", "attention", "spgemm",
                       "spmv"))
    if kind == "spmm":
        rows, per_row = _log(rng, 500, 1 << 20), _log(rng, 3, 64)
        form = rng.choice(("csr", "csr", "csr", "coo"))
        dtype = "f32" if form == "coo" else rng.choice(("f32", "f32", "f64"))
        most = (2.2e9 if dtype == "f32" else 1.1e9) / (rows * (per_row + 1))
        width = min(_log(rng, 1, 512), max(1, int(most)))
        return {"kind": kind, "pattern": rng.choice(("graph", "uniform")), "rows": rows, "per_row": min(per_row, rows // 8),
                "width": width if form == "coo" or rng.random() < 0.5 else _round(width),
                "dtype": dtype, "format": form}
    if kind == "gcn":
        rows = _log(rng, 1000, 1 << 19)
        return {"kind": kind, "rows": rows, "per_row": _log(rng, 3, 24), "features": _log(rng, 32, 512 if rows < 1 << 17 else 160),
                "hidden": rng.choice((16, 32, 64, 100, 128)), "classes": rng.randint(2, 64)}
    if kind == "sparse_weights":
        wide = _log(rng, 256, 8192)
        return {"kind": kind, "wide": wide, "narrow": max(32, wide // rng.choice((2, 4, 8))), "batch": _log(rng, 1, 1024),
                "density": rng.choice((0.02, 0.05, 0.1))}
    if kind == "decoder":
        latents = _log(rng, 1024, 16_384)
        return {"kind": kind, "batch": _log(rng, 1, 4096), "latents": latents, "width": _round(_log(rng, 256, 4096)),
                "active": rng.choice((8, 16, 32, 64))}
    if kind == "sddmm":
        rows, cols = _log(rng, 500, 131_072), _log(rng, 500, 131_072)
        depth = rng.choice((16, 32, 50, 64, 64, 100, 128, 256))
        return {"kind": kind, "rows": rows, "cols": cols,
                "per_row": min(_log(rng, 4, 128), cols // 8, max(4, int(1.0e9 / (rows * depth)))),
                "depth": depth, "format": rng.choice(("csr", "csr", "coo")),
                "unit": rng.random() < 0.5}
    if kind == "attention":
        fused = rng.random() < 0.7
        tokens = _log(rng, 256, 8192)
        if fused:
            tokens = max(256, tokens // 64 * 64)
        mask = rng.choice(("blocks", "window")) if fused else "window"
        return {"kind": kind, "mask": mask, "tokens": tokens, "heads": rng.choice((1, 4, 8, 12, 16)),
                "dim": rng.choice((32, 64, 64, 128)), "dtype": rng.choice(("bf16", "bf16", "f32")) if fused else "f32",
                "fused": fused}
    if kind == "spgemm":
        return {"kind": kind, "rows": _log(rng, 1000, 131_072), "per_row": _log(rng, 2, 16),
                "dtype": rng.choice(("f32", "f32", "f64"))}
    return {"kind": kind, "pattern": rng.choice(("graph", "uniform")), "rows": _log(rng, 1000, 1 << 20), "per_row": _log(rng, 3, 32),
            "dtype": rng.choice(("f32", "f64"))}


def _round(n):
    """A width as models have it: a multiple of 16 (of 4 below 16)."""
    return max(4, n // 4 * 4) if n < 16 else n // 16 * 16


# ---- inputs -----------------------------------------------------------------------------------
_DTYPE = {"f32": torch.float32, "f64": torch.float64, "bf16": torch.bfloat16}


def _rand(gen, *shape, dtype=torch.float32):
    return torch.rand(shape, generator=gen, device="cuda", dtype=dtype)


def _randn(gen, *shape, dtype=torch.float32):
    return torch.randn(shape, generator=gen, device="cuda", dtype=dtype)


def _row_ptr(rows, n_rows):
    pos = torch.zeros(n_rows + 1, dtype=torch.int64, device="cuda")
    pos[1:] = torch.cumsum(torch.bincount(rows, minlength=n_rows), 0)
    return pos.to(torch.int32)


def _scale_to_mean(z, mean, cap):
    """Factor by which positive weights `z` have the given mean after a cap (numpy or torch)."""
    clip = np.minimum if isinstance(z, np.ndarray) else lambda a, c: torch.clamp(a, max=c)
    lo, hi = 0.0, 64.0 * mean
    for _ in range(40):
        mid = 0.5 * (lo + hi)
        lo, hi = (mid, hi) if float(clip(z * mid, float(cap)).mean()) < mean else (lo, mid)
    return hi


def _graph(gen, n, mean):
    """Rows and columns (sorted, distinct) of a graph of n nodes with power-law out-degrees and a loop
    at every node."""
    cap = min(MAX_DEGREE, n - 1)
    z = torch.clamp(torch.floor((1.0 - _rand(gen, n, dtype=torch.float64)) ** (-1.0 / (ZIPF - 1.0))), max=float(cap))
    deg = torch.clamp(z * _scale_to_mean(z, mean, cap), max=float(cap))
    deg = torch.floor(deg + _rand(gen, n, dtype=torch.float64)).to(torch.int64)
    nodes = torch.arange(n, device="cuda")
    rows = torch.repeat_interleave(nodes, deg)
    cols = torch.randint(n, (rows.numel(),), generator=gen, device="cuda")
    key = torch.unique(torch.cat([rows * n + cols, nodes * n + nodes]))
    return key // n, key % n


def _uniform(gen, n_rows, n_cols, mean):
    count = int(n_rows * mean)
    rows = torch.randint(n_rows, (count,), generator=gen, device="cuda")
    cols = torch.randint(n_cols, (count,), generator=gen, device="cuda")
    key = torch.unique(rows * n_cols + cols)
    return key // n_cols, key % n_cols


def _relabelled(gen, rows, cols, n_rows, n_cols):
    """The entries with rows and columns renumbered at random (a square matrix's alike)."""
    p = torch.randperm(n_rows, generator=gen, device="cuda")
    q = p if n_rows == n_cols else torch.randperm(n_cols, generator=gen, device="cuda")
    key = torch.sort(p[rows] * n_cols + q[cols])[0]
    return key // n_cols, key % n_cols


def _matrix(gen, pattern, n, mean, dtype):
    """(rows, columns, values): a normalised graph or a uniformly sparse matrix with values in (-1, 1)."""
    if pattern == "graph":
        rows, cols = _graph(gen, n, mean)
        inv = torch.bincount(rows, minlength=n).to(dtype).rsqrt()
        return rows, cols, inv[rows] * inv[cols]
    rows, cols = _uniform(gen, n, n, mean)
    return rows, cols, _rand(gen, rows.numel(), dtype=dtype) * 2 - 1


def _csr(rows, cols, vals, shape):
    return STensor.from_csr_arrays(_row_ptr(rows, shape[0]), cols.to(torch.int32), vals, shape)


def _window_mask(tokens, window=64):
    """Sliding window on either side and one global token, as CSR arrays."""
    i = torch.arange(tokens, device="cuda")[:, None]
    span = torch.arange(-window, window + 1, device="cuda")[None, :]
    cols = i + span
    fine = (cols >= 0) & (cols < tokens)
    key = torch.cat([(i * tokens + cols)[fine], i[:, 0] * tokens, i[:, 0]]).unique()
    return _row_ptr(key // tokens, tokens), (key % tokens).to(torch.int32)


def _active_blocks(n, window=4, stride=8):
    i, j = np.arange(n)[:, None], np.arange(n)[None, :]
    return (j <= i) & ((i - j < window) | ((i - j) % stride == 0))


def _block_mask(tokens, block=64):
    """Causal local window and strided pattern of 64 x 64 blocks, as CSR arrays."""
    active = torch.from_numpy(_active_blocks(tokens // block)).cuda()
    lens = active.sum(1).repeat_interleave(block) * block
    pos = torch.zeros(tokens + 1, dtype=torch.int64, device="cuda")
    pos[1:] = torch.cumsum(lens, 0)
    br, bc = active.nonzero(as_tuple=True)
    cols = (bc[:, None] * block + torch.arange(block, device="cuda")).reshape(-1)       # of one row per block row
    first = torch.cat([torch.zeros(1, dtype=torch.int64, device="cuda"), torch.cumsum(active.sum(1) * block, 0)])
    row = torch.repeat_interleave(torch.arange(tokens, device="cuda"), lens)
    at = torch.arange(row.numel(), device="cuda") - pos[row] + first[row // block]
    return pos.to(torch.int32), cols[at].to(torch.int32)


# The layers of a graph convolution network as a program writes them.
@scorch.compile
def _hidden_layer(a, h, bias):
    return torch.relu(scorch.matmul(a, h) + bias)


@scorch.compile
def _output_layer(a, h, bias):
    return scorch.matmul(a, h) + bias


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind, s = case["kind"], {"case": case}
    if kind in ("spmm", "spmv"):
        n, dtype = case["rows"], _DTYPE[case["dtype"]]
        rows, cols, vals = _matrix(gen, case["pattern"], n, case["per_row"], dtype)
        if case.get("format") == "coo":
            s["A"] = STensor.from_coo(indices=torch.stack([rows, cols]), values=vals, shape=(n, n))
        else:
            s["A"] = _csr(rows, cols, vals, (n, n))
        s["B"] = _randn(gen, *((n, case["width"]) if kind == "spmm" else (n,)), dtype=dtype)
    elif kind == "gcn":
        n, f, h, c = case["rows"], case["features"], case["hidden"], case["classes"]
        rows, cols, vals = _matrix(gen, "graph", n, case["per_row"], torch.float32)
        s["A"] = _csr(rows, cols, vals, (n, n))
        s["X"] = _randn(gen, n, f)
        s["W1"], s["b1"] = _randn(gen, f, h) / math.sqrt(f), _randn(gen, h)
        s["W2"], s["b2"] = _randn(gen, h, c) / math.sqrt(h), _randn(gen, c)
    elif kind == "sparse_weights":
        wide, narrow = case["wide"], case["narrow"]
        for name, (m, k) in (("W1", (narrow, wide)), ("W2", (wide, narrow))):
            rows, cols = _uniform(gen, m, k, case["density"] * k)
            s[name] = _csr(rows, cols, _randn(gen, rows.numel()) / math.sqrt(case["density"] * k), (m, k))
        s["b1"], s["b2"] = _randn(gen, narrow), _randn(gen, wide)
        s["X"] = _randn(gen, case["batch"], wide)
    elif kind == "decoder":
        b, k, active = case["batch"], case["latents"], case["active"]
        s["W"] = _randn(gen, k, case["width"]) * 0.125
        # what torch.topk of the rectified latents hands over: (batch, active) values, largest first, and int64 indices
        s["vals"], s["idx"] = torch.topk(torch.relu(_randn(gen, b, k)), active, dim=1)
        s["row_ptr"] = torch.arange(0, b * active + 1, active, dtype=torch.int32, device="cuda")
    elif kind == "sddmm":
        m, n, k = case["rows"], case["cols"], case["depth"]
        # results come in the mask's own sparsity: as many entries whatever the seed
        rows, cols = _relabelled(gen, *_uniform(torch.Generator("cuda").manual_seed(m), m, n, case["per_row"]), m, n)
        vals = torch.ones(rows.numel(), device="cuda") if case["unit"] else _rand(gen, rows.numel()) * 2 - 1
        s["mask"] = STensor.from_coo(indices=torch.stack([rows, cols]), values=vals, shape=(m, n)) \
            if case["format"] == "coo" else _csr(rows, cols, vals, (m, n))
        s["Q"], s["K"] = _randn(gen, m, k) * math.sqrt(0.125), _randn(gen, n, k) * math.sqrt(0.125)
    elif kind == "attention":
        t, dtype = case["tokens"], _DTYPE[case["dtype"]]
        s["row_ptr"], s["col_idx"] = _block_mask(t) if case["mask"] == "blocks" else _window_mask(t)
        for name in "QKV":
            s[name] = _randn(gen, case["heads"], t, case["dim"]).to(dtype)
        s["scale"] = 1.0 / math.sqrt(case["dim"])
    elif kind == "spgemm":
        n = case["rows"]
        rows, cols = _relabelled(gen, *_graph(torch.Generator("cuda").manual_seed(n), n, case["per_row"]), n, n)
        s["A"] = _csr(rows, cols, _rand(gen, rows.numel(), dtype=_DTYPE[case["dtype"]]) + 0.5, (n, n))
    return s


# ---- one pass ---------------------------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("spmm", "spmv"):
        return scorch.matmul(s["A"], s["B"])
    if kind == "gcn":
        hidden = _hidden_layer(s["A"], s["X"] @ s["W1"], s["b1"])
        return _output_layer(s["A"], hidden @ s["W2"], s["b2"])
    if kind == "sparse_weights":
        code = torch.relu(scorch.matmul(s["W1"], s["X"].t()).t() + s["b1"])
        return code, scorch.matmul(s["W2"], code.t()).t() + s["b2"]
    if kind == "decoder":
        acts = STensor.from_csr_arrays(s["row_ptr"], s["idx"].reshape(-1), s["vals"].reshape(-1),
                                       (case["batch"], case["latents"]))
        return scorch.matmul(acts, s["W"])
    if kind == "sddmm":
        out = scorch.einsum("ij,ik,jk->ij", s["mask"], s["Q"], s["K"])
        return out.values, out.index.mode_indices
    if kind == "attention":
        if not case["fused"]:
            return ops.sparse_attention_csr(s["row_ptr"], s["col_idx"], s["Q"], s["K"], s["V"], s["scale"])
        fused = ops.sparse_attention_bf16 if case["dtype"] == "bf16" else ops.sparse_attention_f32
        return fused(s["Q"], s["K"], s["V"], s["row_ptr"], s["col_idx"], s["scale"])
    out = scorch.matmul(s["A"], s["A"])
    return out.values, out.index.mode_indices[1]


# ---- what a pass cannot do without --------------------------------------------------------------
def _graph_rows(n, mean):
    """Row lengths of a graph, loop included, at 4,096 evenly spaced quantiles."""
    cap = min(MAX_DEGREE, n - 1)
    u = (np.arange(4096) + 0.5) / 4096
    z = np.minimum(np.floor((1.0 - u) ** (-1.0 / (ZIPF - 1.0))), cap)
    deg = np.minimum(z * _scale_to_mean(z, mean, cap), cap)
    return n * (1.0 - np.exp(-deg / n)) + 1


def _entries(case, n):
    if case.get("pattern", "graph") == "graph":
        return n * float(_graph_rows(n, case["per_row"]).mean())
    return n * n * (1.0 - math.exp(-case["per_row"] / n))


def work(case):
    kind = case["kind"]
    size = {"f64": 8, "bf16": 2}.get(case.get("dtype"), 4)
    if kind in ("spmm", "spmv"):
        n, w = case["rows"], case.get("width", 1)
        nnz = _entries(case, n)
        index = 8 * nnz if case.get("format") == "coo" else 4 * nnz + 4 * (n + 1)
        return {"bytes": index + size * (nnz + 2 * n * w), "flops": 2 * nnz * w}
    if kind == "gcn":
        n, f, h, c = case["rows"], case["features"], case["hidden"], case["classes"]
        nnz = _entries(case, n)
        return {"bytes": 8 * nnz + 4 * (n + 1) + 4 * (n * f + f * h + h * c + h + c + n * c),
                "flops": 2 * n * (f * h + h * c) + 2 * nnz * (h + c)}
    if kind == "sparse_weights":
        a, b, m, d = case["wide"], case["narrow"], case["batch"], case["density"]
        nnz = a * b * (1.0 - math.exp(-d))
        return {"bytes": 2 * 8 * nnz + 4 * (a + b) * (m + 2) + 4 * m * a, "flops": 2 * 2 * nnz * m}
    if kind == "decoder":
        b, k, n, t = case["batch"], case["latents"], case["width"], case["active"]
        used = k * (1.0 - math.exp(-b * t / k))          # rows of the weights that some activation names
        return {"bytes": 12 * b * t + 4 * (b + 1) + 4 * n * (used + b), "flops": 2 * b * t * n}
    if kind == "sddmm":
        m, n, k = case["rows"], case["cols"], case["depth"]
        nnz = m * n * (1.0 - math.exp(-case["per_row"] / n))
        index = 8 * nnz if case["format"] == "coo" else 4 * nnz + 4 * (m + 1)
        return {"bytes": index + 8 * nnz + 4 * k * (m + n), "flops": 2 * nnz * k}
    if kind == "attention":
        t, h, d = case["tokens"], case["heads"], case["dim"]
        nnz = float(_active_blocks(t // 64).sum()) * 4096 if case["mask"] == "blocks" else 131.0 * t
        return {"bytes": size * 4 * h * t * d + 4 * (t + 1) + 4 * nnz, "flops": 4 * nnz * h * d}
    n = case["rows"]
    rows = _graph_rows(n, case["per_row"])
    products = rows * rows.mean()
    nnz, out = n * float(rows.mean()), n * float((n * (1.0 - np.exp(-products / n))).mean())
    return {"bytes": (4 + size) * (nnz + out) + 4 * 2 * (n + 1), "flops": 2 * n * float(products.mean())}


def tolerance(case):
    if case.get("dtype") == "bf16":
        return {"rel": 1e-2}                 # probabilities and results are rounded to eight bits
    if case.get("dtype") == "f64":
        return {"rel": 1e-13}
    return {"rel": 1e-5}
