"""Fused block-sparse attention in fp32 on the MI355X through the C ABI.

Tolerance: relative Frobenius error <= 1e-5 against an fp64 recomputation of the textbook masked
softmax (the reference's "dense" mode, bench/bench_sparse_transformer.py:330-335) on the same
inputs -- the fp32 bar -- and the same bound against this package's own fp32 SDDMM -> softmax ->
SpMM pipeline, the form in which the reference composes sparse attention (:354-372).  The reference
has no fused kernel, so nothing of its own pins this one beyond that composition.
"""
import numpy as np
import pytest
import torch

from gpu_util import dev, three_step_attention
from scorch_amd import workloads
from scorch_amd import scorch_ops_hip as H

pytestmark = pytest.mark.gpu
TOL = 1e-5


def csr_of(mask_bool):
    rp = np.concatenate([[0], np.cumsum(mask_bool.sum(1))]).astype(np.int32)
    return rp, np.nonzero(mask_bool)[1].astype(np.int32)


def case(oracle, mask_bool, heads, D, seed, scale=None, spread=1.0):
    S = mask_bool.shape[0]
    rng = np.random.default_rng(seed)
    q, k, v = (rng.standard_normal((heads, S, D)).astype(np.float32) * spread for _ in range(3))
    scale = D ** -0.5 if scale is None else scale
    rp, ci = csr_of(mask_bool)
    out = H.sparse_attention_f32(dev(q), dev(k), dev(v), dev(rp), dev(ci), scale)
    assert out.dtype == torch.float32 and out.shape == (heads, S, D)
    ref = np.stack([oracle.attention_dense_fp64(q[h], k[h], v[h], mask_bool, scale) for h in range(heads)])
    return out.cpu().numpy(), ref


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("density", [0.03, 0.6])
def test_random_entry_masks(oracle, D, density):
    rng = np.random.default_rng(50 + D)
    mask = rng.random((320, 320)) < density
    mask[17, :] = False                                   # a query without any key: a zero row
    out, ref = case(oracle, mask, 3, D, 51)
    assert oracle.rel_fro(out, ref) <= TOL
    assert np.all(out[:, 17] == 0)


@pytest.mark.parametrize("D", [32, 64, 128])
def test_causal_mask(oracle, D):
    out, ref = case(oracle, np.tril(np.ones((448, 448), bool)), 2, D, 52)
    assert oracle.rel_fro(out, ref) <= TOL


@pytest.mark.parametrize("scale", [-0.7, 0.0, 3.0])
def test_negative_zero_and_large_scales(oracle, scale):
    rng = np.random.default_rng(53)
    mask = rng.random((256, 256)) < 0.3
    out, ref = case(oracle, mask, 2, 64, 54, scale=scale, spread=3.0)
    assert np.isfinite(out).all() and oracle.rel_fro(out, ref) <= TOL


def test_whole_blocks_without_bit_masks(oracle):
    """A pattern of whole 64 x 64 blocks handed over as such (no mask index, no bit masks): the
    benchmark's block pattern at a small size, with an empty block row."""
    w = workloads.attention_blocksparse(S=512, H=3, D=64, seed=55)
    brp, bci = w["block_row_ptr"].copy(), w["block_col_idx"]
    bm = H.BlockMask(512, 64, dev(brp), dev(bci), None, None, int(bci.size) * 4096)
    out = H.attn_blocksparse_f32(dev(w["q"]), dev(w["k"]), dev(w["v"]), bm, float(w["scale"])).cpu().numpy()
    rp, ci = workloads.blocks_to_csr(brp, bci, 64)
    dense = np.zeros((512, 512), bool)
    dense[np.repeat(np.arange(512), np.diff(rp)), ci] = True
    ref = np.stack([oracle.attention_dense_fp64(w["q"][h], w["k"][h], w["v"][h], dense, float(w["scale"]))
                    for h in range(3)])
    assert oracle.rel_fro(out, ref) <= TOL


def test_longformer_mask_reference_shape_against_the_three_launch_form():
    """The reference's attention benchmark at its own shape (S = 4096, 8 heads, D = 32, window 64 +
    one global token: bench/bench_sparse_transformer.py:117-141,194-209), whose global token's block
    row is shared out among workgroups: the fused fp32 kernel against the fp64 dense masked softmax
    and against SDDMM -> softmax -> SpMM in fp32."""
    S, heads, D = 4096, 8, 32
    rp, ci = workloads.longformer_mask(S)
    rng = np.random.default_rng(56)
    q, k, v = (torch.from_numpy(rng.standard_normal((heads, S, D)).astype(np.float32)).cuda() for _ in range(3))
    scale = D ** -0.5
    drp, dci = dev(rp), dev(ci)
    out = H.sparse_attention_f32(q, k, v, drp, dci, scale)
    assert H.attention_block_mask(drp, dci, S).schedule32[1].numel() > 0     # the shared-out row is exercised
    assert torch.equal(out, H.sparse_attention_f32(q, k, v, drp, dci, scale))
    dense = torch.zeros(S, S, dtype=torch.bool)
    dense[torch.from_numpy(np.repeat(np.arange(S), np.diff(rp))), torch.from_numpy(ci).long()] = True
    dense = dense.cuda()
    for h in range(heads):
        s = (q[h].double() @ k[h].double().T) * scale
        s.masked_fill_(~dense, float("-inf"))
        ref = torch.softmax(s, dim=-1) @ v[h].double()
        assert (torch.linalg.norm(out[h].double() - ref) / torch.linalg.norm(ref)).item() <= TOL
    unfused = three_step_attention(drp, dci, q, k, v, scale)
    assert not torch.equal(out, unfused)                 # (another kernel's sums)
    assert (torch.linalg.norm(out - unfused) / torch.linalg.norm(unfused)).item() <= TOL


def test_arguments_are_checked():
    bm = H.BlockMask(128, 64, dev(np.array([0, 1, 2], np.int32)), dev(np.array([0, 1], np.int32)), None, None, 8192)
    q = torch.zeros(1, 128, 64, device="cuda")
    with pytest.raises(TypeError, match="float32"):
        H.attn_blocksparse_f32(q.bfloat16(), q.bfloat16(), q.bfloat16(), bm, 1.0)
    with pytest.raises(ValueError, match="another sequence length"):
        H.attn_blocksparse_f32(q[:, :64], q[:, :64], q[:, :64], bm, 1.0)
    q48 = torch.zeros(1, 128, 48, device="cuda")
    with pytest.raises(RuntimeError, match="head dimensions 32, 64 and 128"):
        H.attn_blocksparse_f32(q48, q48, q48, bm, 1.0)


def test_keys_the_mask_leaves_out_may_hold_anything_in_k(oracle):
    """Padding keys that no query attends to: their rows of K may be NaN (their scores are replaced
    before they are looked at); their rows of V are multiplied by zero probabilities, so V has to be
    finite there.  Both fused kernels, against the fp64 result on clean operands."""
    S, heads, D = 256, 2, 64
    rng = np.random.default_rng(21)
    i, j = np.arange(S)[:, None], np.arange(S)[None, :]
    mask = j <= i
    padded = np.r_[50:64, 130:131, 192:256]         # part of a block, one key, a whole block column
    mask[:, padded] = False
    mask[padded, 0] = True                           # (the padded queries attend to the first key)
    q, k, v = (rng.standard_normal((heads, S, D)).astype(np.float32) for _ in range(3))
    k_bad = k.copy()
    k_bad[:, padded] = np.nan
    rp, ci = csr_of(mask)
    ref = np.stack([oracle.attention_dense_fp64(q[h], k[h], v[h], mask, D ** -0.5) for h in range(heads)])
    out32 = H.sparse_attention_f32(dev(q), dev(k_bad), dev(v), dev(rp), dev(ci), D ** -0.5).cpu().numpy()
    assert np.isfinite(out32).all() and oracle.rel_fro(out32, ref) <= TOL
    to16 = lambda a: dev(a).to(torch.bfloat16)
    out16 = H.sparse_attention_bf16(to16(q), to16(k_bad), to16(v), dev(rp), dev(ci), D ** -0.5).float().cpu().numpy()
    assert np.isfinite(out16).all() and oracle.rel_fro(out16, ref) <= 1e-2


@pytest.mark.parametrize("S", [1, 63, 65, 130, 447, 513])
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("kind", ["window", "causal", "dense"])
def test_sequences_of_any_length_through_the_three_step_call(oracle, S, D, kind):
    """sparse_attention_csr over a mask that fills its blocks goes to the fused kernel when the mask comes
    back, whatever the sequence length: the last block row and column are live up to S only, nothing
    beyond S is read or written, and rows no query refers to may hold anything."""
    i, j = np.arange(S)[:, None], np.arange(S)[None, :]
    mask = {"window": (abs(i - j) <= 40) | (i == 0) | (j == 0), "causal": j <= i, "dense": j >= 0}[kind] & np.ones((S, S), bool)
    unused = S // 2 if S > 3 else None
    if unused is not None:
        mask[:, unused] = False
        mask[unused, :] = False                           # a query without keys: a zero row
    rng = np.random.default_rng(S + D)
    q, k, v = (rng.standard_normal((3, S, D)).astype(np.float32) for _ in range(3))
    rp, ci = (dev(x) for x in csr_of(mask))
    ref = np.stack([oracle.attention_dense_fp64(q[h], k[h], v[h], mask, D ** -0.5) for h in range(3)])
    if unused is not None:
        k[:, unused] = v[:, unused] = np.nan
    def followed_by_nan(x):
        buffer = torch.full((x.size + 64 * D,), float("nan"), device="cuda")
        buffer[:x.size] = dev(x).reshape(-1)
        return buffer[:x.size].view(x.shape)
    dq, dk, dv = (followed_by_nan(x) for x in (q, k, v))
    for call in range(3):
        out = H.sparse_attention_csr(rp, ci, dq, dk, dv, D ** -0.5)
        assert oracle.rel_fro(out.cpu().numpy(), ref) <= TOL
    assert isinstance(rp._scorch_plan.attention, H.BlockMask) == (S > 1)    # (one entry fills no block)


@pytest.mark.parametrize("S", [65, 130, 447, 512, 1500])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_a_non_finite_row_of_v_reaches_the_queries_that_attend_to_it_and_no_others(S, D):
    """From the first call (three steps) to the later ones (the fused kernel, whose tiles hold the row for all
    64 queries of a block): NaN, either infinity, both in one sum, values whose products overflow; a
    key that every query attends to, one that few do, one in a whole block."""
    i, j = np.arange(S)[:, None], np.arange(S)[None, :]
    mask = (abs(i - j) <= 40) | (i == 0)
    mask[: S // 2] |= j[:, :] == 5
    rng = np.random.default_rng(S + D)
    q, k, v = (rng.standard_normal((2, S, D)).astype(np.float32) for _ in range(3))
    v[0, 5, 3] = np.inf
    v[0, S // 2] = np.nan
    v[0, S - 1, ::2] = -np.inf
    v[0, S - 2, 1::3] = np.inf                            # (with the row before: NaN where both meet)
    v[1, S // 3, D - 1] = -np.inf
    v[1, 7] = 3e38                                        # finite, though a product of two is not
    v[1, 9] = -3e38
    scale = 0.5 * D ** -0.5                               # (no probability underflows)
    want = np.empty((2, S, D))
    with np.errstate(all="ignore"):
        for h in range(2):
            for row in range(S):
                keys = np.flatnonzero(mask[row])
                s = scale * (k[h, keys].astype(np.float64) @ q[h, row].astype(np.float64))
                p = np.exp(s - s.max())
                want[h, row] = (p / p.sum()) @ v[h, keys].astype(np.float64)
    rp, ci = (dev(x) for x in csr_of(mask))
    dq, dk, dv = (dev(x) for x in (q, k, v))
    finite = np.isfinite(want)
    assert not finite.all() and finite.mean() > 0.3
    size = np.abs(want[finite])
    for call in range(3):
        out = H.sparse_attention_csr(rp, ci, dq, dk, dv, scale).cpu().numpy()
        if call == 0 and S % 64 == 0:
            continue                                      # (the first call's SpMM is by blocks: a block's rows share)
        np.testing.assert_array_equal(np.isnan(out), np.isnan(want))
        np.testing.assert_array_equal(np.isposinf(out), np.isposinf(want))
        np.testing.assert_array_equal(np.isneginf(out), np.isneginf(want))
        # sums of up to S terms that may cancel, each rounded a few times: against the magnitudes that go in
        assert (np.abs(out[finite] - want[finite]) <= 1e-5 * np.maximum(size, np.where(size > 1e6, 3e38, 4.0))).all()
    assert isinstance(rp._scorch_plan.attention, H.BlockMask)
    if S % 64 == 0:
        assert np.array_equal(H.sparse_attention_f32(dq, dk, dv, rp, ci, scale).cpu().numpy(), out, equal_nan=True)


# seven block rows: 7 workgroups of a block row to a head, more with the global token's row in stretches
@pytest.mark.parametrize("heads", [1, 24, 40, 50, 90])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_teams_of_four_two_and_one_wavefront_to_sixteen_queries(oracle, heads, D):
    """Launches of more and more workgroups: the tiles of sixteen queries are shared out to fewer and fewer
    wavefronts.  Sixteen queries without any key, sixteen with a single one, and a NaN that reaches one head's queries of key 99."""
    S = 447
    i, j = np.arange(S)[:, None], np.arange(S)[None, :]
    mask = (abs(i - j) <= 40) | (i == 0) | (j == 0)
    mask[160:192] = False
    mask[176:192, 300] = True
    rng = np.random.default_rng(heads + D)
    q, k, v = (rng.standard_normal((heads, S, D)).astype(np.float32) for _ in range(3))
    scale = D ** -0.5
    ref = {h: oracle.attention_dense_fp64(q[h], k[h], v[h], mask, scale) for h in {0, heads // 2, heads - 1}}
    v[heads - 1, 99, D - 1] = np.nan
    rp, ci = (dev(x) for x in csr_of(mask))
    dq, dk, dv = (dev(x) for x in (q, k, v))
    for call in range(3):
        out = H.sparse_attention_csr(rp, ci, dq, dk, dv, scale).cpu().numpy()
    assert isinstance(rp._scorch_plan.attention, H.BlockMask)
    reached = np.zeros((S, D), bool)
    reached[mask[:, 99], D - 1] = True
    for h, want in ref.items():
        hit = reached if h == heads - 1 else np.zeros_like(reached)
        assert np.isnan(out[h][hit]).all()
        assert oracle.rel_fro(np.where(hit, 0, out[h]), np.where(hit, 0, want)) <= TOL
        assert np.all(out[h, 160:176] == 0)


# twenty block rows, and five or so stretches of the row with the global token: 384 to 800 workgroups of a block row
@pytest.mark.parametrize("heads, token", [(16, 0), (24, 40), (25, 17), (32, 1100), (33, 1218)])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_a_few_long_rows_in_stretches_of_four_workgroups_each(oracle, heads, token, D):
    """One query that attends to everything, in every sixteen of its block row: its stretches go to more wavefronts than the
    other rows, whatever the order of the items."""
    S = 1219
    i, j = np.arange(S)[:, None], np.arange(S)[None, :]
    mask = (abs(i - j) <= 40) | (i == token) | (j == token)
    rng = np.random.default_rng(heads + D)
    q, k, v = (rng.standard_normal((heads, S, D)).astype(np.float32) for _ in range(3))
    scale = D ** -0.5
    rp, ci = (dev(x) for x in csr_of(mask))
    dq, dk, dv = (dev(x) for x in (q, k, v))
    for call in range(3):
        out = H.sparse_attention_csr(rp, ci, dq, dk, dv, scale).cpu().numpy()
    for h in {0, heads // 2, heads - 1}:
        assert oracle.rel_fro(out[h], oracle.attention_dense_fp64(q[h], k[h], v[h], mask, scale)) <= TOL
    bm = rp._scorch_plan.attention
    items, split_rows, n_slots = H._fp32_launch_schedule(bm, heads, D)
    rows = items.view(-1, 4)
    assert 0 < 3 * n_slots <= rows.shape[0] and bool((rows[:n_slots, 3] >= 0).all())
    bm.pairing["fp32", heads, D] = (rows.flip(0).contiguous().view(-1), split_rows, n_slots)
    turned = H.attn_blocksparse_f32(dq, dk, dv, bm, scale).cpu().numpy()
    assert oracle.rel_fro(turned, out) <= TOL


@pytest.mark.parametrize("heads, token", [(16, 0), (33, 700)])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_non_finite_values_in_stretches_of_four_workgroups_each(heads, token, D):
    """NaN, either infinity, both in one sum, values whose products overflow and a NaN in K: in keys that only the query that attends to
    everything and a window's queries refer to, and in the key that every query does."""
    S = 1219
    i, j = np.arange(S)[:, None], np.arange(S)[None, :]
    mask = (abs(i - j) <= 40) | (i == token) | (j == token)
    rng = np.random.default_rng(heads + D)
    q, k, v = (rng.standard_normal((heads, S, D)).astype(np.float32) for _ in range(3))
    last = heads - 1
    v[0, token, 3] = np.inf
    v[0, S // 2] = np.nan
    v[0, S - 1, ::2] = -np.inf
    v[0, S - 2, 1::3] = np.inf
    v[1, 7], v[1, 9] = 3e38, -3e38                        # finite, though a product of two is not
    v[1, S // 3, D - 1] = -np.inf
    k[last, 300, D // 2] = np.nan                         # a score of NaN: the whole row
    scale = 0.5 * D ** -0.5                               # (no probability underflows)
    rp, ci = (dev(x) for x in csr_of(mask))
    dq, dk, dv = (dev(x) for x in (q, k, v))
    for call in range(3):
        out = H.sparse_attention_csr(rp, ci, dq, dk, dv, scale).cpu().numpy()
    n_items, n_slots = (lambda items, split_rows, slots: (items.numel() // 4, slots))(
        *H._fp32_launch_schedule(rp._scorch_plan.attention, heads, D))
    assert 0 < 3 * n_slots <= n_items and heads * n_items > (160 if D == 128 else 320)
    for h in (0, 1, 2, last):
        want = np.empty((S, D))
        with np.errstate(all="ignore"):
            for row in range(S):
                keys = np.flatnonzero(mask[row])
                x = scale * (k[h, keys].astype(np.float64) @ q[h, row].astype(np.float64))
                p = np.exp(x - x.max())
                want[row] = (p / p.sum()) @ v[h, keys].astype(np.float64)
        finite = np.isfinite(want)
        assert finite.all() == (h == 2) and finite.any()
        np.testing.assert_array_equal(np.isnan(out[h]), np.isnan(want))
        np.testing.assert_array_equal(np.isposinf(out[h]), np.isposinf(want))
        np.testing.assert_array_equal(np.isneginf(out[h]), np.isneginf(want))
        # sums that may cancel, each rounded a few times: against the magnitudes that go in
        size = np.abs(want[finite])
        assert (np.abs(out[h][finite] - want[finite]) <= 1e-5 * np.maximum(size, np.where(size > 1e6, 3e38, 4.0))).all()


# a block row in so many stretches: the combining kernel asks for four or eight of them at once, and for the others in batches
@pytest.mark.parametrize("stretches", [2, 4, 5, 7, 8, 9, 16, 17, 25])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_combining_the_stretches_of_a_long_row(oracle, stretches, D):
    S, heads, token = 128 * stretches - 64, 2, 70
    i, j = np.arange(S)[:, None], np.arange(S)[None, :]
    mask = (abs(i - j) <= 20) | (i == token)
    rng = np.random.default_rng(stretches + D)
    q, k, v = (rng.standard_normal((heads, S, D)).astype(np.float32) for _ in range(3))
    k *= np.linspace(0.1, 4.0, S, dtype=np.float32)[:, None]  # the stretches' maxima differ
    rp, ci = (dev(x) for x in csr_of(mask))
    bm = H.attention_block_mask(rp, ci, S)
    plain = H.BlockMask(bm.S, bm.block, bm.block_row_ptr, bm.block_col_idx, None, None, bm.nnz)
    plain.block_row_lens = bm.row_lens()
    H.split_long_block_rows(plain, 2, list_unequal_rows=True)
    assert int(plain.split_rows.view(-1, 4)[:, 2].max()) == stretches
    bm.pairing["fp32", heads, D] = (plain.items, plain.split_rows, plain.n_slots)
    out = H.attn_blocksparse_f32(*(dev(x) for x in (q, k, v)), bm, D ** -0.5).cpu().numpy()
    for h in range(heads):
        assert oracle.rel_fro(out[h], oracle.attention_dense_fp64(q[h], k[h], v[h], mask, D ** -0.5)) <= TOL


# rows of two stretches beside one of so many
@pytest.mark.parametrize("stretches", [3, 4, 5, 9, 12])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_combining_a_long_rows_stretches_beside_many_rows_of_two(oracle, stretches, D):
    S, heads, token = 128 * stretches, 2, 70
    i, j = np.arange(S)[:, None], np.arange(S)[None, :]
    mask = (abs(i - j) <= 80) | (i == token)
    rng = np.random.default_rng(stretches + D)
    q, k, v = (rng.standard_normal((heads, S, D)).astype(np.float32) for _ in range(3))
    k *= np.linspace(0.1, 4.0, S, dtype=np.float32)[:, None]  # the stretches' maxima differ
    rp, ci = (dev(x) for x in csr_of(mask))
    bm = H.attention_block_mask(rp, ci, S)
    plain = H.BlockMask(bm.S, bm.block, bm.block_row_ptr, bm.block_col_idx, None, None, bm.nnz)
    plain.block_row_lens = bm.row_lens()
    H.split_long_block_rows(plain, 2, list_unequal_rows=True)
    rows = plain.split_rows.view(-1, 4)
    assert int(rows[:, 2].max()) == stretches and plain.n_slots <= 4 * len(rows)
    bm.pairing["fp32", heads, D] = (plain.items, plain.split_rows, plain.n_slots)
    out = H.attn_blocksparse_f32(*(dev(x) for x in (q, k, v)), bm, D ** -0.5).cpu().numpy()
    for h in range(heads):
        assert oracle.rel_fro(out[h], oracle.attention_dense_fp64(q[h], k[h], v[h], mask, D ** -0.5)) <= TOL
