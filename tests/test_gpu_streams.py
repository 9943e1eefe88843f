"""What is kept with an operand between calls is made on the stream of the call that needed it first, and read
by calls on any other: each call here follows one on another stream that is still waiting for its turn."""
import numpy as np
import pytest
import torch

import scorch_amd as scorch
from conftest import random_csr
from gpu_util import dev
from scorch_amd import STensor, native, workloads
from scorch_amd import scorch_ops_hip as H

pytestmark = pytest.mark.gpu


class _behind:
    """``with _behind(stream):`` runs its body on a stream that is busy for some 50 ms."""

    def __init__(self, stream):
        self.stream, self.context = stream, torch.cuda.stream(stream)

    def __enter__(self):
        self.context.__enter__()
        torch.cuda._sleep(100_000_000)

    def __exit__(self, *exc):
        return self.context.__exit__(*exc)


def _graph(rng, n, long_row, dtype=np.float32):
    lens = rng.integers(0, 9, n)
    lens[3] = long_row
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    return rp, rng.integers(0, n, rp[-1]).astype(np.int32), rng.uniform(-1, 1, rp[-1]).astype(dtype)


@pytest.mark.parametrize("form", ["csr", "coo", "coo_unsorted"])
@pytest.mark.parametrize("N", [None, 24, 200, 1024])
def test_products_on_a_stream_that_did_not_make_what_they_read(form, N):
    if form != "csr" and N is None:
        pytest.skip("coordinate operands have no matrix-vector kernel")
    rng = np.random.default_rng(5)
    n = 700
    rp, ci, v = _graph(rng, n, 3000)
    rows = np.repeat(np.arange(n), np.diff(rp)).astype(np.int32)
    if form == "coo_unsorted":
        order = rng.permutation(rows.size)
        rows, ci, v = rows[order], ci[order], v[order]
    A = STensor.from_csr_arrays(dev(rp), dev(ci), dev(v), (n, n)) if form == "csr" else \
        STensor._coo((n, n), [dev(rows), dev(ci)], dev(v), "A")
    dense = torch.zeros(n, n, dtype=torch.float64)
    dense.index_put_((torch.from_numpy(rows).long(), torch.from_numpy(ci).long()), torch.from_numpy(v).double(), accumulate=True)
    b = torch.randn(n, N or 1, device="cuda") if N else torch.randn(n, device="cuda")
    want = dense @ b.double().cpu()

    def check(out):
        torch.cuda.synchronize()
        assert float((out.double().cpu() - want).norm()) <= 1e-5 * float(want.norm())

    scorch.matmul(A, torch.randn(n, 5, device="cuda"))            # the inspection, which waits for its stream
    torch.cuda.synchronize()
    one, two = torch.cuda.Stream(), torch.cuda.Stream()
    for turn in range(4):                                         # (a copy by column tiles is made on the second use)
        with _behind(one):
            first = scorch.matmul(A, b)
        with torch.cuda.stream(two):
            second = scorch.matmul(A, b)
        check(second)
        check(first)
    for stream in (one, two) if form != "coo_unsorted" else ():    # (coordinates out of row order are never decided)
        with torch.cuda.stream(stream):
            assert native.host().spmm(A, b, None, 0) is not None
    assert native.host().spmm(A, b, None, 0) is None              # nothing has been decided on this stream
    check(scorch.matmul(A, b))


@pytest.mark.parametrize("form", ["csr", "coo"])
@pytest.mark.parametrize("pattern", ["blocks", "uniform", "wide"])
def test_sampled_products_on_another_stream(form, pattern):
    rng = np.random.default_rng(6)
    n, K, n_cols = (256, 64, 256) if pattern == "blocks" else (300, 64, 300) if pattern == "uniform" else (8192, 256, 8192)
    if pattern == "blocks":
        rp, ci = workloads.longformer_mask(n)
    elif pattern == "uniform":
        rp, ci, _ = random_csr(rng, n, n_cols, 0.05)
    else:
        rp = np.arange(0, n * 8 + 1, 8).astype(np.int32)
        ci = rng.integers(0, n_cols, n * 8).astype(np.int32)
    rows = np.repeat(np.arange(n), np.diff(rp)).astype(np.int32)
    values = dev(rng.uniform(0.5, 1.5, ci.size).astype(np.float32))
    S = STensor.from_csr_arrays(dev(rp), dev(ci), values, (n, n_cols)) if form == "csr" else \
        STensor._coo((n, n_cols), [dev(rows), dev(ci)], values, "S")
    q, k = torch.randn(n, K, device="cuda"), torch.randn(n_cols, K, device="cuda")
    want = (values.double() * (q.double()[dev(rows).long()] * k.double()[dev(ci).long()]).sum(1)).cpu()
    torch.cuda.synchronize()
    one, two = torch.cuda.Stream(), torch.cuda.Stream()
    for turn in range(5):
        with _behind(one):
            first = scorch.einsum("ij,ik,jk->ij", S, q, k)
        with torch.cuda.stream(two):
            second = scorch.einsum("ij,ik,jk->ij", S, q, k)
            second_rows = second.index.mode_indices[0][0].clone()
        torch.cuda.synchronize()
        for out in (second, first):
            assert float((out.values.double().cpu() - want).norm()) <= 1e-5 * float(want.norm())
        assert np.array_equal(second_rows.cpu().numpy(), rows)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads", [1, 8])
def test_attention_on_another_stream(dtype, heads):
    S, D = 1024, 64
    fn = H.sparse_attention_bf16 if dtype == torch.bfloat16 else H.sparse_attention_f32
    blocks = workloads.blocksparse_pattern(S // 64)
    for mask in (workloads.longformer_mask(S), workloads.blocks_to_csr(*blocks, 64)):
        rp, ci = (dev(x) for x in mask)
        q, k, v = (torch.randn(heads, S, D, device="cuda").to(dtype) for _ in range(3))
        want = fn(q, k, v, rp.clone(), ci.clone(), 0.125)
        torch.cuda.synchronize()
        one, two = torch.cuda.Stream(), torch.cuda.Stream()
        for turn in range(3):
            with _behind(one):
                first = fn(q, k, v, rp, ci, 0.125)
            with torch.cuda.stream(two):
                second = fn(q, k, v, rp, ci, 0.125)
            torch.cuda.synchronize()
            assert torch.equal(first, want) and torch.equal(second, want)


def test_kept_memory_is_not_handed_out_while_another_stream_reads_it():
    """The operand is dropped while a product on a second stream is still queued: what was kept with it must not
    become another tensor's memory on the stream it came from before that product has run."""
    rng = np.random.default_rng(7)
    n, N = 3000, 48
    rp, ci, v = _graph(rng, n, 20_000)
    operands = [dev(x) for x in (rp, ci, v)]
    b = torch.randn(n, N, device="cuda")
    A = STensor.from_csr_arrays(*operands, (n, n))
    want = scorch.matmul(A, b)
    two = torch.cuda.Stream()
    two.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(two):
        scorch.matmul(A, b)
    torch.cuda.synchronize()
    bounds = operands[0]._scorch_plan.bounds[(N, 4)]
    size = bounds.numel()
    with _behind(two):
        late = scorch.matmul(A, b)
    operands[0].__dict__.clear()                                  # what forget() and the end of the operand do
    A.storage.__dict__.pop("_routes", None)
    where = bounds.data_ptr()
    del bounds
    fresh = [torch.full((size,), 0x7F, dtype=torch.uint8, device="cuda") for _ in range(8)]
    assert all(t.data_ptr() != where for t in fresh)
    torch.cuda.synchronize()
    assert torch.equal(late, want)


@pytest.mark.parametrize("N", [None, 24, 200])
@pytest.mark.parametrize("pin", ["auto", "merge"])
def test_what_a_capture_would_make_is_not_kept(N, pin, monkeypatch):
    """A product of a planned operand at a width that is new, recorded first and replayed never: the eager product
    after it does not read what the recording alone would have filled.  Then the replays."""
    monkeypatch.setattr(H, "SPMM_PATH", pin)
    rng = np.random.default_rng(8)
    n = 900
    rp, ci, v = _graph(rng, n, 4000)
    A = STensor.from_csr_arrays(dev(rp), dev(ci), dev(v), (n, n))
    b = torch.randn(n, N, device="cuda") if N else torch.randn(n, device="cuda")
    dense = torch.zeros(n, n, dtype=torch.float64)
    dense.index_put_((torch.from_numpy(np.repeat(np.arange(n), np.diff(rp))), torch.from_numpy(ci).long()),
                     torch.from_numpy(v).double(), accumulate=True)
    want = dense @ b.double().cpu()
    scorch.matmul(A, torch.randn(n, 5, device="cuda"))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        recorded = scorch.matmul(A, b)
    assert ((N, 4) if N else "spmv") not in A.index.mode_indices[1][0]._scorch_plan.bounds
    eager = scorch.matmul(A, b)
    for _ in range(3):
        assert float((eager.double().cpu() - want).norm()) <= 1e-5 * float(want.norm())
        graph.replay()
        torch.cuda.synchronize()
        assert float((recorded.double().cpu() - want).norm()) <= 1e-5 * float(want.norm())
        recorded.zero_()
        eager = scorch.matmul(A, b)


@pytest.mark.parametrize("kind", ["csr", "coo", "vector", "sddmm", "attention"])
def test_a_recording_holds_what_it_reads(kind):
    """forget() drops what is kept with an operand; a recorded step goes on reading it."""
    from scorch_amd import graphs
    rng = np.random.default_rng(9)
    n, N = 640, 48
    rp, ci, v = _graph(rng, n, 5000)
    rows = np.repeat(np.arange(n), np.diff(rp)).astype(np.int32)
    A = STensor._coo((n, n), [dev(rows), dev(ci)], dev(v), "A") if kind == "coo" else \
        STensor.from_csr_arrays(dev(rp), dev(ci), dev(v), (n, n))
    X = torch.randn(n, device="cuda") if kind == "vector" else torch.randn(n, N, device="cuda")
    forgotten, X2 = A, torch.randn_like(X)
    if kind == "sddmm":
        step = lambda x: scorch.einsum("ij,ik,jk->ij", A, x, X2).values
    elif kind == "attention":
        X, X2 = torch.randn(2, n, 64, device="cuda"), torch.randn(2, n, 64, device="cuda")
        mask = forgotten = tuple(dev(x) for x in workloads.longformer_mask(n))
        step = lambda x: H.sparse_attention_f32(x, X2, X2, *mask, 0.125)
    else:
        step = lambda x: scorch.matmul(A, x)
    recorded = graphs.capture(step, X, warmup=4)
    want = step(X)
    # (fp32 sums by another kernel, or in another order)
    close = lambda got: float((got - want).norm()) <= 2e-5 * float(want.norm())
    assert close(recorded())
    H.forget(forgotten)
    junk = [torch.full((size,), 0x7F, dtype=torch.uint8, device="cuda") for size in (512, 2048, 8192, 65_536, 1 << 20)
            for _ in range(40)]
    for _ in range(3):
        recorded.result.zero_()
        assert close(recorded())
        torch.cuda.synchronize()
    del junk
