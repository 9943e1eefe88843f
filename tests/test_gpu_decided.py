"""Products that have been decided are served by the native call path (scorch_amd/csrc/host.cpp): same
results as the general way, and nothing stale after a write, a replaced tensor or forget()."""
import numpy as np
import pytest
import torch

import scorch_amd as scorch
from conftest import random_csr
from gpu_util import dev, host
from scorch_amd import STensor, native
from scorch_amd import scorch_ops_hip as H

pytestmark = pytest.mark.gpu


def _operand(rng, M, K, dtype, form, long_row=0):
    rp, ci, v = random_csr(rng, M, K, 0.05, dtype)
    if long_row:
        lens = np.diff(rp); lens[3] = long_row
        rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        ci = rng.integers(0, K, rp[-1]).astype(np.int32)
        v = rng.uniform(-1, 1, rp[-1]).astype(dtype)
    rows = np.repeat(np.arange(M), np.diff(rp))
    dense = torch.zeros(M, K, dtype=torch.float64)
    dense.index_put_((torch.from_numpy(rows), torch.from_numpy(ci).long()), torch.from_numpy(v).double(), accumulate=True)
    if form == "coo":
        return STensor._coo((M, K), [dev(rows.astype(np.int32)), dev(ci)], dev(v), "A"), dense
    return STensor.from_csr_arrays(dev(rp), dev(ci), dev(v), (M, K)), dense


def _close(got, want, dtype):
    tol = 1e-5 if dtype == np.float32 else 1e-12
    return float((got.double().cpu() - want).norm()) <= tol * max(float(want.norm()), 1e-30)


@pytest.mark.parametrize("form, dtype", [("csr", np.float32), ("csr", np.float64), ("coo", np.float32)])
@pytest.mark.parametrize("long_row", [0, 700])
@pytest.mark.parametrize("N", [None, 1, 37, 128])
def test_decided_products_follow_their_operands(form, dtype, long_row, N):
    if form == "coo" and N is None:
        pytest.skip("coordinate operands have no matrix-vector kernel")
    rng = np.random.default_rng(7)
    M, K = 330, 290
    A, dense = _operand(rng, M, K, dtype, form, long_row)
    b = dev(rng.standard_normal((K, N) if N else K).astype(dtype))
    for _ in range(3):
        assert _close(scorch.matmul(A, b), dense @ b.double().cpu(), dtype)
    decided = native.host().spmm
    assert decided(A, b, None, 0) is not None
    A.values.mul_(2)                                              # values are read on every call
    assert _close(decided(A, b, None, 0), 2 * dense @ b.double().cpu(), dtype)
    assert decided(A, b.float() if dtype == np.float64 else b.double(), None, 0) is None
    assert decided(A, b[:-1], None, 0) is None
    if N and N > 1:
        turned = decided(A, b.t().contiguous().t(), None, 0)          # the transpose of a stored operand (fp32)
        assert turned is None if dtype == np.float64 else torch.equal(turned, decided(A, b, None, 0))
        assert decided(A, torch.cat([b, b], 1)[:, ::2], None, 0) is None    # any other view goes the general way
        assert _close(scorch.matmul(A, b.t().contiguous().t()), 2 * dense @ b.double().cpu(), dtype)
    H.forget(A)
    assert decided(A, b, None, 0) is None
    for _ in range(2):                                            # (whether a pattern is made of blocks: from the second on)
        assert _close(scorch.matmul(A, b), 2 * dense @ b.double().cpu(), dtype)
    assert decided(A, b, None, 0) is not None
    crd = A.index.mode_indices[1][-1]
    crd[0] = K + 5                                                # a write to the pattern: inspected again, refused
    assert decided(A, b, None, 0) is None
    with pytest.raises(ValueError, match="column"):
        scorch.matmul(A, b)


def test_a_decided_product_keeps_to_pinned_paths_and_to_its_storage():
    rng = np.random.default_rng(8)
    A, dense = _operand(rng, 256, 256, np.float32, "csr")
    b = torch.randn(256, 24, device="cuda")
    scorch.matmul(A, b)
    decided = native.host().spmm
    assert decided(A, b, None, 0) is not None
    H.SPMM_PATH = "merge"
    try:
        assert decided(A, b, None, 0) is None
    finally:
        H.SPMM_PATH = "auto"
    assert decided(A, b, None, 0) is not None
    A.storage._value = A.values * 3                               # another tensor in its place
    assert decided(A, b, None, 0) is None
    assert _close(scorch.matmul(A, b), 3 * dense @ b.double().cpu(), np.float32)


@pytest.mark.parametrize("form", ["csr", "coo"])
@pytest.mark.parametrize("unit", [True, False])
def test_a_decided_sddmm_notices_new_mask_values(form, unit):
    rng = np.random.default_rng(9)
    M, n, K = 200, 170, 48
    S, dense = _operand(rng, M, n, np.float32, form)
    if unit:
        S.values.fill_(1.0)
        dense = (dense != 0).double()
    q, k = torch.randn(M, K, device="cuda"), torch.randn(n, K, device="cuda")
    want = (q.double() @ k.double().t()).cpu()
    for _ in range(4):
        out = scorch.einsum("ij,ik,jk->ij", S, q, k)
    assert native.host().sddmm(S, q, k) is not None

    def check(out, scale):
        r, c = (out.index.mode_indices[i][0].long().cpu() for i in (0, 1))
        assert torch.allclose(out.values.double().cpu(), scale * (dense * want)[r, c], rtol=1e-4, atol=1e-4)
    check(scorch.einsum("ij,ik,jk->ij", S, q, k), 1)
    S.values.mul_(0.5)
    assert native.host().sddmm(S, q, k) is None                   # what was known about the values no longer holds
    for _ in range(4):
        check(scorch.einsum("ij,ik,jk->ij", S, q, k), 0.5)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_decided_attention_is_the_general_ways_bit_for_bit(dtype):
    from scorch_amd import workloads
    S, Hn, D = 512, 4, 32
    rp, ci = (dev(x) for x in workloads.longformer_mask(S))
    q, k, v = (torch.randn(Hn, S, D, device="cuda").to(dtype) for _ in range(3))
    fn = H.sparse_attention_bf16 if dtype == torch.bfloat16 else H.sparse_attention_f32
    first = fn(q, k, v, rp, ci, 0.2)
    f32 = int(dtype == torch.float32)
    assert torch.equal(native.host().attention(q, k, v, rp, ci, 0.2, f32), first)
    assert native.host().attention(q, k, v, rp, ci.clone(), 0.2, f32) is None
    assert native.host().attention(q, k, v, rp, ci, 0.2, 1 - f32) is None
    rp.add_(0)                                                    # written to, if only with what it held
    assert native.host().attention(q, k, v, rp, ci, 0.2, f32) is None
    assert torch.equal(fn(q, k, v, rp, ci, 0.2), first)


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int32, np.int64])
@pytest.mark.parametrize("N", [1, 2, 3, 5, 16, 61, 65, 130, 300])
@pytest.mark.parametrize("relu", [None, True])
def test_rows_folded_in_one_launch_are_the_second_launchs_bit_for_bit(dtype, N, relu):
    """The decided product lets the last of the chunks that share a row add their parts up; the general way
    makes a second launch for it.  Rows that end at, just before and just after a chunk's boundary,
    over two chunks and over hundreds; many launches one after the other on the same counters."""
    if relu and dtype != np.float32:
        pytest.skip("the fused epilogue is fp32")
    rng = np.random.default_rng(N)
    K = 500
    lens = rng.integers(0, 9, 4000)
    lens[[3, 700, 701, 2500, 3999]] = [20_000, 300, 31, 5000, 2000]
    lens[1000:1040] = np.arange(225, 265)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    integer = np.issubdtype(dtype, np.integer)
    ci = rng.integers(0, K, rp[-1]).astype(np.int32)
    v = (rng.integers(-9, 9, rp[-1]) if integer else rng.uniform(-1, 1, rp[-1])).astype(dtype)
    A = STensor.from_csr_arrays(dev(rp), dev(ci), dev(v), (lens.size, K))
    b = dev((rng.integers(-9, 9, (K, N)) if integer else rng.standard_normal((K, N))).astype(dtype))
    bias = torch.randn(N, device="cuda") if relu else None
    general = (lambda: scorch.spmm_bias_act(A, b, bias, relu=True)) if relu else (lambda: scorch.matmul(A, b))
    want = general()
    for _ in range(20):
        got = native.host().spmm(A, b, bias, 2 if relu else 0)
        assert got is not None and torch.equal(got, want)
    assert all(int(c.abs().sum()) == 0 for c in H._counter_buffers.values())


@pytest.mark.parametrize("dtype, N", [(np.float32, 129), (np.float32, 257), (np.float32, 258), (np.float32, 259), (np.float32, 513),
                                      (np.float32, 771), (np.int32, 257), (np.float64, 129), (np.float64, 257), (np.float64, 385),
                                      (np.int64, 513)])
@pytest.mark.parametrize("act", [0, 1])
def test_folded_rows_of_widths_whose_last_column_tile_is_one_ragged_vector(dtype, N, act, monkeypatch):
    """A last vector that is moved back from the row's end shares columns with the one before it: were that
    another column tile's, the tiles' folds would read one another's sums, and count a part or the
    bias twice.  Rows of two to sixteen chunks, of more than sixteen, and many such rows at once."""
    if act and dtype != np.float32:
        pytest.skip("the fused epilogue is fp32")
    monkeypatch.setenv("SCORCH_HIP_TILED", "0")                   # (a copy by column tiles would take the wide ones)
    rng = np.random.default_rng(N)
    K = 300
    lens = rng.integers(0, 5, 1500)
    lens[::50] = rng.integers(300, 900, 30)
    lens[[7, 702, 1499]] = [30_000, 12_000, 9000]
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    integer = np.issubdtype(dtype, np.integer)
    ci = rng.integers(0, K, rp[-1]).astype(np.int32)
    v = (rng.integers(-9, 9, rp[-1]) if integer else rng.uniform(-1, 1, rp[-1])).astype(dtype)
    b = (rng.integers(-9, 9, (K, N)) if integer else rng.standard_normal((K, N))).astype(dtype)
    A = STensor.from_csr_arrays(dev(rp), dev(ci), dev(v), (lens.size, K))
    bd, bias = dev(b), torch.randn(N, device="cuda") if act else None
    general = (lambda: scorch.spmm_bias_act(A, bd, bias)) if act else (lambda: scorch.matmul(A, bd))
    first = general()
    dense = np.zeros((lens.size, K))
    np.add.at(dense, (np.repeat(np.arange(lens.size), lens), ci), v.astype(np.float64))
    want = dense @ b.astype(np.float64) + (host(bias).astype(np.float64) if act else 0)
    # a row's error is below its entries' count, in fp32's or fp64's unit, times the sum of magnitudes (first
    # 1, then n additions); integers are exact
    unit = 0.0 if integer else np.finfo(dtype).eps
    bound = np.zeros_like(dense)
    np.add.at(bound, (np.repeat(np.arange(lens.size), lens), ci), np.abs(v.astype(np.float64)))
    bound = unit * (lens[:, None] + 2) * (bound @ np.abs(b.astype(np.float64)) + 10)
    assert (np.abs(host(first).astype(np.float64) - want) <= bound).all()
    for _ in range(30):
        got = native.host().spmm(A, bd, bias, act)
        assert got is not None and torch.equal(got, first)
    assert all(int(c.abs().sum()) == 0 for c in H._counter_buffers.values())


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int32, np.int64])
@pytest.mark.parametrize("rows, entries", [(1, 0), (1, 447), (1, 448), (3, 1500), (5000, 20_000), (900_000, 5_000_000)])
def test_vector_product_from_a_plans_boundaries(dtype, rows, entries):
    """One short chunk, a row that ends at a chunk's end, rows over many chunks, and the larger chunks of
    large matrices: against float64, and launch after launch on the same counters."""
    rng = np.random.default_rng(rows)
    K = 3000
    lens = rng.multinomial(entries // 2, np.full(rows, 1 / rows))
    lens[rows // 2] += entries - entries // 2
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    integer = np.issubdtype(dtype, np.integer)
    ci = rng.integers(0, K, entries).astype(np.int32)
    v = (rng.integers(-9, 9, entries) if integer else rng.uniform(-1, 1, entries)).astype(dtype)
    x = (rng.integers(-9, 9, K) if integer else rng.standard_normal(K)).astype(dtype)
    A = STensor.from_csr_arrays(dev(rp), dev(ci), dev(v), (rows, K))
    xd = dev(x)
    want = np.bincount(np.repeat(np.arange(rows), lens), v.astype(np.float64) * x[ci], minlength=rows)
    got = scorch.matmul(A, xd)
    if integer:
        assert np.array_equal(host(got), want.astype(dtype))
    else:
        tol = 1e-5 if dtype == np.float32 else 1e-12
        assert np.linalg.norm(host(got) - want) <= tol * max(np.linalg.norm(want), 1e-30)
    for _ in range(10):
        assert torch.equal(scorch.matmul(A, xd), got)
    assert all(int(c.abs().sum()) == 0 for c in H._counter_buffers.values())


@pytest.mark.parametrize("rows, K, N, per_row", [(1, 1, 3, 1), (37, 50, 5, 7), (64, 500, 64, 300), (4096, 2048, 1024, 8)])
def test_new_columns_under_known_row_pointers(rows, K, N, per_row):
    """New column indices with every product, the same row pointers: each product is its own, a column out
    of range is refused after any number of good ones (and leaves the next one alone), columns multiplied
    a second time are planned, and a rewritten row pointer is looked at again."""
    gen = torch.Generator(device="cuda").manual_seed(rows)
    rp = torch.arange(0, rows * per_row + 1, per_row, dtype=torch.int32, device="cuda")
    b = torch.randn(K, N, device="cuda", generator=gen)

    def product(ci, vals):
        return scorch.matmul(STensor.from_csr_arrays(rp, ci, vals, (rows, K)), b)

    def check(ci, vals):
        want = torch.zeros(rows, K, dtype=torch.float64)
        at = torch.arange(rows).repeat_interleave(per_row)
        want.index_put_((at, ci.long().cpu()), vals.double().cpu(), accumulate=True)
        assert _close(product(ci, vals), want @ b.double().cpu(), np.float32)

    for turn in range(6):
        ci = torch.randint(K, (rows * per_row,), device="cuda", generator=gen, dtype=torch.int32 if turn % 2 else torch.int64)
        vals = torch.randn(rows * per_row, device="cuda", generator=gen)
        check(ci, vals)
        if turn == 2:
            for outside in (K, -1, 2**31 - 1):
                bad = ci.to(torch.int32)
                bad[-1] = outside
                with pytest.raises(ValueError, match="column"):
                    product(bad, vals)
    first = rp._scorch_plan
    ci = ci.to(torch.int32)
    for _ in range(3):
        check(ci, vals)
    assert rp._scorch_plan is not first and H._plan_at_hand(rp, ci, rows, K) is rp._scorch_plan
    rp[-1] += 1
    with pytest.raises(ValueError, match="row_ptr"):
        product(torch.zeros_like(ci), vals)


@pytest.mark.parametrize("rows, K, N, longest", [(4099, 2048, 1000, 40), (1500, 16_384, 2050, 70), (90, 3000, 8200, 1500)])
def test_new_columns_with_a_dense_operand_stored_by_column_tiles(rows, K, N, longest, monkeypatch):
    """The kernel looks at the columns itself: the same bits as with columns that were checked before, columns out of range at the
    first, some and the last entry refused, rows without entries and rows that chunks cut, several streams."""
    rng = np.random.default_rng(rows)
    lens = rng.integers(0, longest + 1, rows)
    lens[[0, rows // 2]] = [longest, 0]
    rp = dev(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32))
    nnz = int(lens.sum())
    assert native.lib().scorch_hip_spmm_csr_tiled_recommended(rows, K, N, nnz)
    b = torch.randn(K, N, device="cuda")
    vals = torch.randn(nnz, device="cuda")
    product = lambda ci: scorch.matmul(STensor.from_csr_arrays(rp, ci, vals, (rows, K)), b)
    columns = lambda: dev(rng.integers(0, K, nnz).astype(np.int32))
    for _ in range(3):
        product(columns())                                # (the copy by column tiles is made for the second one)
    for at in (0, nnz // 3, nnz - 1):
        for outside in (K, -1, 2**31 - 1, -2**31):
            bad = columns()
            bad[at] = outside
            with pytest.raises(ValueError, match="column"):
                product(bad)
        ci = columns()
        got = product(ci)
        with monkeypatch.context() as m:
            m.setattr(H, "SPMM_PATH", "tiled")
            assert torch.equal(got, scorch.matmul(STensor.from_csr_arrays(rp.clone(), ci, vals, (rows, K)), b))
    streams = [torch.cuda.Stream() for _ in range(3)]
    torch.cuda.synchronize()
    some = [(s, columns()) for s in streams for _ in range(3)]
    results = []
    for s, ci in some:
        with torch.cuda.stream(s):
            s.wait_stream(torch.cuda.default_stream())
            results.append(product(ci))
    torch.cuda.synchronize()
    for (_, ci), got in zip(some, results):
        at = torch.repeat_interleave(torch.arange(rows), torch.from_numpy(lens))
        want = torch.zeros(rows, K, dtype=torch.float64).index_put_((at, ci.long().cpu()), vals.double().cpu(), accumulate=True)
        assert _close(got, want @ b.double().cpu(), np.float32)


def test_no_memory_for_a_decided_products_result_is_an_error_to_catch(monkeypatch):
    """The native call path allocates the result itself: without memory for it the caller gets torch's
    OutOfMemoryError, as from the general way, and the next product works."""
    monkeypatch.setattr(H, "_empty", H._torch_empty)              # (the allocation in native code, not the tests' poisoned one)
    rows, N = 1 << 19, 512                                        # a result of 1 GiB, from operands of a few MB
    rp = torch.arange(rows + 1, dtype=torch.int32, device="cuda")
    ci = torch.arange(rows, dtype=torch.int32, device="cuda") % 64
    A = STensor.from_csr_arrays(rp, ci, torch.ones(rows, device="cuda"), (rows, 64))
    b = torch.randn(64, N, device="cuda")
    S = 1 << 14
    mask = (torch.arange(0, S + 1, dtype=torch.int32, device="cuda") * 64,
            torch.arange(S * 64, dtype=torch.int32, device="cuda") % 64 + torch.arange(S, dtype=torch.int32, device="cuda").div(
                64, rounding_mode="floor").repeat_interleave(64) * 64)
    q = torch.randn(128, S, 64, device="cuda").to(torch.bfloat16)     # 256 MiB
    for _ in range(3):
        scorch.matmul(A, b)
        H.sparse_attention_bf16(q, q, q, *mask, 0.125)
    assert native.host().spmm(A, b, None, 0) is not None and native.host().attention(q, q, q, *mask, 0.125, 0) is not None
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (64 << 20)) / total)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            native.host().spmm(A, b, None, 0)
        with pytest.raises(torch.OutOfMemoryError):
            scorch.matmul(A, b)
        with pytest.raises(torch.OutOfMemoryError):
            H.sparse_attention_bf16(q, q, q, *mask, 0.125)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(scorch.matmul(A, b)[:64], b)


@pytest.mark.parametrize("N", [8, 512])
def test_decided_products_of_inference_and_of_wrapped_tensors(N, monkeypatch):
    """A dense operand without a version counter is multiplied like any other (and never copied by column
    tiles); one without storage -- torch.vmap, torch.func.grad -- is an error to catch, not an abort."""
    monkeypatch.setattr(H, "_empty", H._torch_empty)
    rng = np.random.default_rng(3)
    A, dense = _operand(rng, 400, 300, np.float32, "csr")
    b = torch.randn(300, N, device="cuda")
    for _ in range(3):
        scorch.matmul(A, b)
    with torch.inference_mode():
        inner = torch.randn(300, N, device="cuda")
        for _ in range(4):
            assert _close(scorch.matmul(A, inner), dense @ inner.double().cpu(), np.float32)
            inner.mul_(0.5)
    for _ in range(2):
        assert _close(scorch.matmul(A, inner), dense @ inner.double().cpu(), np.float32)
    with pytest.raises(RuntimeError):
        torch.vmap(lambda x: scorch.matmul(A, x))(torch.stack([b, b]))
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda x: scorch.matmul(A, x).sum())(b)
    assert native.host().spmm(A, torch.randn(300, N, device="cuda"), None, 0) is not None


def test_forget_and_mark_volatile_concern_the_tensors_they_name():
    """What is forgotten, or marked, is decided anew; another operand's decisions stand."""
    from scorch_amd import workloads
    rng = np.random.default_rng(11)
    (A, _), (other, _) = (_operand(rng, 300, 300, np.float32, "csr") for _ in range(2))
    b = torch.randn(300, 20, device="cuda")
    S = _operand(rng, 200, 170, np.float32, "csr")[0]
    q, k = torch.randn(200, 48, device="cuda"), torch.randn(170, 48, device="cuda")
    rp, ci = (dev(x) for x in workloads.longformer_mask(256))
    h = torch.randn(2, 256, 64, device="cuda")
    stands = {
        "spmm": lambda: native.host().spmm(A, b, None, 0) is not None,
        "other": lambda: native.host().spmm(other, b, None, 0) is not None,
        "sddmm": lambda: native.host().sddmm(S, q, k) is not None,
        "attention": lambda: native.host().attention(h, h, h, rp, ci, 0.2, 1) is not None,
    }

    def decide():
        for _ in range(4):
            scorch.matmul(A, b), scorch.matmul(other, b), scorch.einsum("ij,ik,jk->ij", S, q, k)
            H.sparse_attention_f32(h, h, h, rp, ci, 0.2)
        assert all(check() for check in stands.values())

    a_pos, a_crd = A.index.mode_indices[1]
    for act, gone in ((lambda: H.forget(b), ""), (lambda: H.forget(torch.zeros(3, device="cuda")), ""),
                      (lambda: H.mark_volatile(b), ""), (lambda: H.mark_volatile(b, volatile=False), ""),
                      (lambda: H.forget(A), "spmm"), (lambda: H.forget(A.values), "spmm"), (lambda: H.forget(a_pos), "spmm"),
                      (lambda: H.forget(a_crd), "spmm"), (lambda: H.forget(S.values), "sddmm"),
                      (lambda: H.mark_volatile(S.values), "sddmm"), (lambda: H.forget(rp), "attention"),
                      (lambda: H.forget(ci), "attention"), (lambda: H.forget(rp, ci, S, A, other), "spmm other sddmm attention")):
        decide()
        act()
        assert [name for name, check in stands.items() if not check()] == gone.split()
        H.mark_volatile(S.values, volatile=False)
    # values rewritten while they were volatile, behind the version counter's back
    S.values.fill_(1.0)
    decide()
    H.mark_volatile(S.values)
    S.values.data.fill_(2.0)
    H.mark_volatile(S.values, volatile=False)
    twice = scorch.einsum("ij,ik,jk->ij", S, q, k).values
    for _ in range(4):
        assert torch.equal(scorch.einsum("ij,ik,jk->ij", S, q, k).values, twice)
    at = [x[0].long().cpu() for x in scorch.einsum("ij,ik,jk->ij", S, q, k).index.mode_indices]
    assert torch.allclose(twice.cpu(), 2 * (q.double() @ k.double().t()).float().cpu()[at[0], at[1]], rtol=1e-4, atol=1e-4)


def test_a_wide_operand_that_is_rewritten_before_every_product_is_served_by_the_native_path():
    """A width at which a dense operand that stays as it is gets a copy by column tiles: one that does not is
    multiplied as it lies, without asking Python; left alone, it gets its copy on the second product."""
    rng = np.random.default_rng(12)
    A, dense = _operand(rng, 1024, 256, np.float32, "csr")
    b = torch.randn(256, 1024, device="cuda")
    for _ in range(2):
        scorch.matmul(A, b)
    for step in range(4):
        b.mul_(0.5)
        out = native.host().spmm(A, b, None, 0)
        assert out is not None and _close(out, dense @ b.double().cpu(), np.float32)
    copied = native.lib().scorch_hip_dense_tiled_recommended(256, 1024, A.values.numel(), 4)
    assert (native.host().spmm(A, b, None, 0) is None) == bool(copied)      # unchanged since: the general path's turn
    for _ in range(3):
        assert _close(scorch.matmul(A, b), dense @ b.double().cpu(), np.float32)
    assert copied and b._scorch_tiled[0] == b._version and native.host().spmm(A, b, None, 0) is not None
