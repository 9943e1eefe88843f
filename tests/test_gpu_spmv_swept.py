"""Matrix-vector products over the copy of the entries that a matrix gets when it comes back unchanged
(csrc/spmv_swept.hip): the kernel at the edges of its bands, parts, batches and cut rows, and when the copy is made,
used and dropped."""
import numpy as np
import pytest
import torch

import scorch_amd as scorch
from gpu_util import dev, host
from scorch_amd import STensor, native
from scorch_amd import scorch_ops_hip as H

pytestmark = pytest.mark.gpu


def _pattern(name, rng):
    """(row lengths, columns): bands hold 512 entries or a 1,024th of all, 2,048 rows to a part, batches 512 entries."""
    if name == "one_entry":
        return np.array([1]), 5
    if name == "one_row":                                  # cut into a piece for every band
        return np.array([3001]), 7001
    if name == "one_long_row_among_empty":
        lens = np.zeros(9000, np.int64)
        lens[4500] = 20_011
        return lens, 1 << 17
    if name == "batches":                                  # 511, 512, 513, 1,024 entries to a row
        return np.tile([511, 512, 513, 1024, 0, 1, 3], 40), 70_000
    if name == "parts":                                    # bands of more rows than have sums in LDS
        lens = (rng.random(40_000) < 0.02).astype(np.int64)
        lens[:3] = 700
        return lens, 2048
    if name == "empty_head_and_tail":
        lens = np.zeros(30_000, np.int64)
        lens[14_000:16_000] = rng.integers(0, 60, 2000)
        return lens, 300_000
    if name == "short_rows":
        return rng.integers(0, 6, 60_000), 1 << 21
    if name == "hubs":
        lens = rng.integers(1, 9, 5000)
        lens[[0, 17, 4999]] = 9000, 40_003, 1700
        return lens, 500_000
    raise KeyError(name)


def _matrix(name, dtype, seed=3):
    rng = np.random.default_rng(seed)
    lens, K = _pattern(name, rng)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ci = np.concatenate([np.sort(rng.integers(0, K, n)) for n in lens] + [np.zeros(0, np.int64)]).astype(np.int32)
    return rp, ci, rng.uniform(-1, 1, rp[-1]).astype(dtype), rng.uniform(-1, 1, K).astype(dtype)


def _check(got, rp, ci, v, x):
    """Products and sums in fp64: n roundings of 2^-53 of the sum of moduli, whatever the order, and ten for parts of a cut row;
    the result is rounded to its type once, that of a cut row twice."""
    terms = v.astype(np.longdouble) * x.astype(np.longdouble)[ci]
    rows = np.repeat(np.arange(rp.size - 1), np.diff(rp))
    want, moduli = np.zeros(rp.size - 1, np.longdouble), np.zeros(rp.size - 1, np.longdouble)
    np.add.at(want, rows, terms)
    np.add.at(moduli, rows, np.abs(terms))
    lens = np.diff(rp)
    unit = 2.0 ** (-24 if v.dtype == np.float32 else -53)
    bound = (lens + 12) * 2.0 ** -53 * moduli + 4 * unit * moduli
    assert np.all(np.abs(got.astype(np.longdouble) - want) <= bound)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("name", ["one_entry", "one_row", "one_long_row_among_empty", "batches", "parts", "empty_head_and_tail",
                                  "short_rows", "hubs"])
def test_kernel_against_wide_sums(name, dtype):
    rp, ci, v, x = _matrix(name, dtype)
    L, M, K, nnz, size = native.lib(), rp.size - 1, x.size, v.size, v.itemsize
    t_rp, t_ci, t_v, t_x = dev(rp), dev(ci), dev(v), dev(x)
    suffix, stream = ("f32" if size == 4 else "f64"), torch.cuda.current_stream().cuda_stream
    copy = H._empty(L.scorch_hip_spmv_csr_listed_bytes(M, nnz, size), dtype=torch.uint8, device="cuda")
    native.check(getattr(L, "scorch_hip_spmv_csr_listed_copy_" + suffix)(
        M, K, nnz, t_rp.data_ptr(), t_ci.data_ptr(), t_v.data_ptr(), copy.data_ptr(), copy.numel(), stream))
    longest, results = int(np.diff(rp).max()), []
    for known in (longest, 0, longest):
        y = H._empty(M, dtype=t_v.dtype, device="cuda")
        ws = H._empty(L.scorch_hip_spmv_csr_listed_workspace_bytes(M, nnz), dtype=torch.uint8, device="cuda")
        native.check(getattr(L, "scorch_hip_spmv_csr_listed_" + suffix)(
            M, K, nnz, t_rp.data_ptr(), copy.data_ptr(), copy.numel(), t_x.data_ptr(), y.data_ptr(), ws.data_ptr(), ws.numel(), known,
            stream))
        results.append(host(y))
    _check(results[0], rp, ci, v, x)
    assert all(np.array_equal(r, results[0]) for r in results)


def _operand(dtype=np.float64, K=420_000, M=3000, per_row=300):
    rng = np.random.default_rng(8)
    rp = np.arange(0, M * per_row + 1, per_row, dtype=np.int32)
    ci = np.sort(rng.integers(0, K, (M, per_row)), axis=1).reshape(-1).astype(np.int32)
    v, x = rng.uniform(-1, 1, ci.size).astype(dtype), rng.uniform(-1, 1, K).astype(dtype)
    return rp, ci, v, x


def _copy_of(values):
    kept = H._kept(values, "_scorch_swept")
    return kept[2] if kept is not None and isinstance(kept[2], torch.Tensor) else None


def test_the_copy_follows_the_matrix():
    rp, ci, v, x = _operand()
    t_rp, t_ci, t_v, t_x = dev(rp), dev(ci), dev(v), dev(x)
    A = STensor.from_csr_arrays(t_rp, t_ci, t_v, (rp.size - 1, x.size))

    def products(scale, n, served=True):
        """`n` products, the last of them from the copy or not."""
        for _ in range(n):
            _check(host(scorch.matmul(A, t_x)), rp, ci, v * scale, x)
        assert (_copy_of(A.values) is not None) == served

    products(1.0, H.SWEPT_AFTER, served=False)
    products(1.0, 1)
    first = _copy_of(A.values)
    y = scorch.matmul(A, t_x)                               # the native call path's
    assert _copy_of(A.values) is first and torch.equal(y, scorch.matmul(A, t_x))
    A.values.mul_(2.0)                                      # written to: not served from the copy
    products(2.0, 1, served=False)
    products(2.0, H.SWEPT_AFTER + 1)
    A.values.data.mul_(2.0)                                 # unseen: the caller says so
    H.forget(A)
    products(4.0, 1, served=False)
    products(4.0, H.SWEPT_AFTER + 1)
    H.mark_volatile(A.values)                               # nothing derived from them is kept or used any more
    A.values.data.mul_(0.5)
    products(2.0, H.SWEPT_AFTER + 2, served=False)
    H.mark_volatile(A.values, volatile=False)
    ci = np.roll(ci.reshape(-1, 300), 1, axis=0).reshape(-1)
    A.index.mode_indices[1][1].copy_(dev(ci))               # another pattern
    products(2.0, H.SWEPT_AFTER + 2)


def test_the_copy_on_another_stream_under_a_capture_and_without_memory(monkeypatch):
    rp, ci, v, x = _operand(np.float32, K=900_000, M=7000)
    A = STensor.from_csr_arrays(dev(rp), dev(ci), dev(v), (rp.size - 1, x.size))
    t_x = dev(x)
    real = H._empty

    def refuse(*size, **kw):
        if kw.get("dtype") is torch.uint8 and size[0] > (4 << 20):
            raise torch.OutOfMemoryError("refused")
        return real(*size, **kw)
    monkeypatch.setattr(H, "_empty", refuse)
    for _ in range(H.SWEPT_AFTER + 3):
        _check(host(scorch.matmul(A, t_x)), rp, ci, v, x)
        assert _copy_of(A.values) is None
    monkeypatch.setattr(H, "_empty", real)
    for _ in range(H.SWEPT_AFTER + 1):
        _check(host(scorch.matmul(A, t_x)), rp, ci, v, x)
    assert _copy_of(A.values) is not None
    side = torch.cuda.Stream()
    for _ in range(3):
        with torch.cuda.stream(side):
            torch.cuda._sleep(20_000_000)
            out = scorch.matmul(A, t_x)
        torch.cuda.synchronize()
        _check(host(out), rp, ci, v, x)
    from scorch_amd.graphs import capture
    step = capture(lambda b: scorch.matmul(A, b), t_x)
    for scale in (1.0, 2.0, 4.0):                           # a replay reads the values that are there then
        _check(host(step()), rp, ci, v * np.float32(scale), x)
        A.values.mul_(2.0)
        torch.cuda.synchronize()


def test_refusals():
    L = native.lib()
    assert L.scorch_hip_spmv_csr_listed_recommended(1 << 20, 1 << 20, 1 << 24, 8) == 1
    assert L.scorch_hip_spmv_csr_listed_recommended(1 << 20, 1 << 22, 1 << 24, 8) == 0      # columns do not fit an entry's word
    assert L.scorch_hip_spmv_csr_listed_recommended(4096, 4096, 1 << 24, 8) == 0            # x fits an L2
    assert L.scorch_hip_spmv_csr_listed_bytes(10, 100, 2) == 0
    x = torch.zeros(1024, dtype=torch.float64, device="cuda")
    args = (10, 1 << 22, 100, x.data_ptr(), x.data_ptr(), 8192, x.data_ptr(), x.data_ptr(), x.data_ptr(), 8192, 0, None)
    assert L.scorch_hip_spmv_csr_listed_f64(*args) == native.EUNSUPPORTED
    assert L.scorch_hip_spmv_csr_listed_f64(*((10, 512) + args[2:5] + (64,) + args[6:])) == native.EWORKSPACE
    assert L.scorch_hip_spmv_csr_listed_f64(*((10, 512) + args[2:9] + (4,) + args[10:])) == native.EWORKSPACE
