"""GPU parity of the sampled product, the sparse softmax and the attention block that chains them
with the batched SpMM, through the C ABI, against the CPU oracle and dense torch arithmetic."""
import math

import numpy as np
import pytest
import torch

import sspmm_amd
from sspmm_amd import _lib, synth
from gpu_util import dev, max_rel_err

pytestmark = pytest.mark.gpu


def _pattern(m_rows, K, V, sparsity, seed):
    return synth.vector_sparse(m_rows * V, K, V, sparsity, seed=seed)


@pytest.mark.parametrize("V", [8, 16])
@pytest.mark.parametrize("F", [8, 40, 64, 128, 200, 256])
def test_sddmm_matches_oracle(oracle, built_library, V, F):
    vs = _pattern(20, 300, V, 0.8, seed=100 + F)
    rng = np.random.default_rng(F)
    lhs = rng.standard_normal((vs.m_vec * V, F)).astype(np.float16)
    rhs = rng.standard_normal((300, F)).astype(np.float16)
    print("sddmm V=%d F=%d nvec=%d" % (V, F, vs.col_idx.size), flush=True)
    got = sspmm_amd.sddmm(None, dev(vs.row_offsets), dev(vs.col_idx), dev(lhs), dev(rhs), V)
    torch.cuda.synchronize()
    want = oracle.sddmm(vs.m_vec, V, vs.row_offsets, vs.col_idx, lhs, rhs)
    assert got.shape == (vs.col_idx.size * V,)
    assert max_rel_err(got.cpu().numpy(), want) <= 2e-3
    # exact on small integers (every product and partial sum is representable)
    lhs_i = rng.integers(-3, 4, lhs.shape).astype(np.float16)
    rhs_i = rng.integers(-3, 4, rhs.shape).astype(np.float16)
    got = sspmm_amd.sddmm(None, dev(vs.row_offsets), dev(vs.col_idx), dev(lhs_i), dev(rhs_i), V).cpu().numpy()
    assert np.array_equal(got, oracle.sddmm(vs.m_vec, V, vs.row_offsets, vs.col_idx, lhs_i, rhs_i))


@pytest.mark.parametrize("per_row", [0, 1, 15, 16, 17, 31, 32, 33, 100])
def test_sddmm_row_length_tails_and_permutation(oracle, built_library, per_row):
    V, K, F, m_vec = 8, 128, 64, 6
    rng = np.random.default_rng(per_row)
    cols = np.concatenate([rng.permutation(K)[:per_row] for _ in range(m_vec)] or [[]]).astype(np.int32)
    off = (np.arange(m_vec + 1) * per_row).astype(np.int32)
    lhs = rng.standard_normal((m_vec * V, F)).astype(np.float16)
    rhs = rng.standard_normal((K, F)).astype(np.float16)
    want = oracle.sddmm(m_vec, V, off, cols, lhs, rhs)
    perm = dev(rng.permutation(m_vec).astype(np.int32))
    for ri in (None, perm):
        got = sspmm_amd.sddmm(ri, dev(off), dev(cols) if cols.size else torch.empty(0, dtype=torch.int32, device="cuda"),
                              dev(lhs), dev(rhs), V)
        torch.cuda.synchronize()
        assert got.numel() == cols.size * V
        if cols.size:
            assert max_rel_err(got.cpu().numpy(), want) <= 2e-3


@pytest.mark.parametrize("V", [8, 16])
def test_sddmm_of_many_waves_reads_its_indices_in_blocks(oracle, built_library, V):
    """64 features and more than 8192 waves: indices in blocks of 64, rows that end at and around a block's end."""
    K, F, batch = 200, 64, 431
    lens = [0, 1, 15, 16, 17, 47, 48, 49, 63, 64, 65, 79, 80, 81, 127, 128, 129, 143, 193, 200]
    rng = np.random.default_rng(V)
    cols = np.concatenate([rng.permutation(K)[:n] for n in lens]).astype(np.int32)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    assert (batch - 1) * len(lens) > 8192 >= len(lens)
    lhs = rng.integers(-3, 4, (batch, len(lens) * V, F)).astype(np.float16)  # (every product and sum is representable)
    rhs = rng.integers(-3, 4, (batch, K, F)).astype(np.float16)
    got = sspmm_amd.bsddmm(None, dev(off), dev(cols), dev(lhs), dev(rhs), V)
    torch.cuda.synchronize()
    for b in (0, batch // 2, batch - 1):
        want = oracle.sddmm(len(lens), V, off, cols, lhs[b], rhs[b])
        assert np.array_equal(got[b].cpu().numpy(), want)
        assert torch.equal(got[b], sspmm_amd.sddmm(None, dev(off), dev(cols), dev(lhs[b]), dev(rhs[b]), V))


@pytest.mark.parametrize("V", [8, 16])
def test_softmax_matches_oracle_and_rows_sum_to_one(oracle, built_library, V):
    rng = np.random.default_rng(7)
    lens = np.array([0, 1, 5, 64, 65, 200, 0, 1000, 3, 256, 257, 512, 513])  # around what a wave keeps in registers
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    vals = (rng.standard_normal(off[-1] * V) * 4).astype(np.float16)
    scaler = 1.0 / math.sqrt(64)
    got = sspmm_amd.csr_softmax(None, dev(off), dev(vals), scaler, V)
    torch.cuda.synchronize()
    got = got.cpu().numpy()
    want = oracle.softmax(len(lens), V, off, vals, scaler)
    assert np.abs(got.astype(np.float64) - want.astype(np.float64)).max() <= 2e-3
    g = got.astype(np.float64).reshape(-1, V)
    for i, n in enumerate(lens):
        if n:
            assert np.all(np.abs(g[off[i]:off[i + 1]].sum(axis=0) - 1) < 1e-2)
    # a negative scaler turns the row's minimum into the reference point
    neg = sspmm_amd.csr_softmax(None, dev(off), dev(vals), -0.25, V).cpu().numpy()
    assert np.abs(neg.astype(np.float64) - oracle.softmax(len(lens), V, off, vals, -0.25).astype(np.float64)).max() <= 2e-3
    # a large common offset must not overflow: softmax is shift invariant
    big = (vals.astype(np.float32) + 30000).astype(np.float16)
    shifted = sspmm_amd.csr_softmax(None, dev(off), dev(big), 1.0, V).cpu().numpy()
    assert np.isfinite(shifted).all()


def test_batched_ops_match_looped_single_calls(oracle, built_library):
    V, K, F, batch = 8, 160, 64, 5
    vs = _pattern(16, K, V, 0.85, seed=9)
    rng = np.random.default_rng(10)
    q = rng.standard_normal((batch, vs.m_vec * V, F)).astype(np.float16)
    k = rng.standard_normal((batch, K, F)).astype(np.float16)
    off, col = dev(vs.row_offsets), dev(vs.col_idx)
    w = sspmm_amd.bsddmm(None, off, col, dev(q), dev(k), V)
    p = sspmm_amd.bcsr_softmax(None, off, w, 0.125, V, batch)
    torch.cuda.synchronize()
    assert w.shape == (batch, vs.col_idx.size * V) and p.shape == w.shape
    for b in range(batch):
        assert torch.equal(w[b], sspmm_amd.sddmm(None, off, col, dev(q[b]), dev(k[b]), V))
        assert torch.equal(p[b], sspmm_amd.csr_softmax(None, off, w[b].contiguous(), 0.125, V))


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("V", [8, 16])
def test_sparse_attention_matches_dense_masked_attention(built_library, V, fused):
    """The reference's block (sddmm -> softmax -> spmm), as three launches and as one, against torch attention
    with a -inf mask."""
    seq, d, batch = 256, 64, 6
    vs = _pattern(seq // V, seq, V, 0.8, seed=11)
    g = torch.Generator("cuda").manual_seed(12)
    q, k, v = (torch.randn(batch, seq, d, device="cuda", generator=g).half() for _ in range(3))
    out = sspmm_amd.sparse_attention(None, dev(vs.row_offsets), dev(vs.col_idx), q, k, v, 1.0 / math.sqrt(d), V, fused=fused)
    torch.cuda.synchronize()
    mask = torch.full((seq, seq), float("-inf"), device="cuda")
    for i in range(vs.m_vec):
        cols = torch.from_numpy(vs.col_idx[vs.row_offsets[i]:vs.row_offsets[i + 1]].astype(np.int64)).cuda()
        mask[i * V:(i + 1) * V, cols] = 0
    scores = q.float() @ k.float().transpose(1, 2) / math.sqrt(d) + mask
    want = torch.softmax(scores, dim=-1) @ v.float()
    assert out.shape == (batch, seq, d) and out.dtype == torch.float16
    assert max_rel_err(out.float().cpu().numpy(), want.cpu().numpy()) <= 1e-2


def _dense_attention(off, cols, V, q, k, v, scale):
    """float64 numpy: per vector-row, softmax over the stored columns, rows without any give zeros."""
    batch, m, d = q.shape
    out = np.zeros((batch, m, v.shape[-1]))
    q64, k64, v64 = (t.astype(np.float64) for t in (q, k, v))
    for i in range(len(off) - 1):
        c = cols[off[i]:off[i + 1]]
        if c.size == 0:
            continue
        s = np.einsum("bvd,bjd->bvj", q64[:, i * V:(i + 1) * V], k64[:, c]) * scale
        e = np.exp(s - s.max(axis=-1, keepdims=True))
        out[:, i * V:(i + 1) * V] = np.einsum("bvj,bjd->bvd", e / e.sum(axis=-1, keepdims=True), v64[:, c])
    return out


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("V", [8, 16])
def test_one_launch_attention_row_lengths_permutation_and_large_scores(built_library, V, d):
    """Rows of every length around the kernel's step of 32 vectors (none, one, a full step, one more, several steps
    and a tail), visited through a permutation, with scores large enough that the running maximum has to move by
    hundreds between steps; against float64 arithmetic and against the three launches."""
    n_keys, batch = 200, 3
    lens = [0, 1, 2, 31, 32, 33, 63, 64, 65, 96, 100, 200, 0, 7]
    rng = np.random.default_rng(40 + V + d)
    cols = np.concatenate([np.sort(rng.permutation(n_keys)[:n]) for n in lens]).astype(np.int32)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    m = len(lens) * V
    q = (rng.standard_normal((batch, m, d)) * 3 * (64 / d) ** 0.5).astype(np.float16)
    k = (rng.standard_normal((batch, n_keys, d)) * 3).astype(np.float16)
    v = rng.standard_normal((batch, n_keys, d)).astype(np.float16)
    perm = dev(rng.permutation(len(lens)).astype(np.int32))
    for scale in (0.125, 2.0):  # scores up to a few hundred, then a few thousand
        want = _dense_attention(off, cols, V, q, k, v, scale)
        for ri in (None, perm):
            print("attention V=%d d=%d scale=%g permuted=%s" % (V, d, scale, ri is not None), flush=True)
            got = sspmm_amd.fused_sparse_attention(ri, dev(off), dev(cols), dev(q), dev(k), dev(v), scale, V)
            torch.cuda.synchronize()
            got = got.cpu().numpy().astype(np.float64)
            assert np.isfinite(got).all()
            assert np.abs(got - want).max() <= 4e-3 * max(1.0, np.abs(want).max())
            for i, n in enumerate(lens):
                if n == 0:
                    assert not got[:, i * V:(i + 1) * V].any()
    chain = sspmm_amd.sparse_attention(None, dev(off), dev(cols), dev(q), dev(k), dev(v), 0.125, V, fused=False)
    one = sspmm_amd.sparse_attention(None, dev(off), dev(cols), dev(q), dev(k), dev(v), 0.125, V)  # picks the one launch
    assert torch.equal(one, sspmm_amd.fused_sparse_attention(None, dev(off), dev(cols), dev(q), dev(k), dev(v), 0.125, V))
    # (the chain rounds scores of magnitude up to ~100 to fp16, a step of 1/16 in the exponent's argument before the scale)
    assert (one.float() - chain.float()).abs().max().item() <= 3e-2


@pytest.mark.parametrize("gap", [7.0, 9.0, 10.5, 12.0])
def test_one_launch_attentions_with_many_small_probabilities(built_library, gap):
    """One key ahead of all others by gap^2 / 8, 6 to 18 in the exponent, so that the others' probabilities are small, subnormal in
    fp16 or nothing there: together they are a good part of the sum.  A probability's rounding is 2^-25 at most there
    (half a step), one for each key, and 2^-11 of it above; the result's rounding is 2^-11 of values of about one."""
    from sspmm_amd.layers import attention_fm
    keys, d = 4096, 64
    x = np.float16(gap)
    q, k = np.zeros((1, 64, d), np.float16), np.zeros((1, keys, d), np.float16)
    q[..., 0], k[0, 0, 0] = x, x
    v = np.where(np.arange(keys) % 2, 1.0, 0.5)[None, :, None].repeat(d, 2).astype(np.float16)
    v[0, 0] = -1.0
    bound = keys * 2.0 ** -25 + 2.0 ** -10
    for V in (8, 16):
        off = (np.arange(64 // V + 1) * keys).astype(np.int32)
        cols = np.tile(np.arange(keys, dtype=np.int32), 64 // V)
        want = _dense_attention(off, cols, V, q, k, v, 0.125)
        got = sspmm_amd.fused_sparse_attention(None, dev(off), dev(cols), dev(q), dev(k), dev(v), 0.125, V)
        assert np.abs(got.cpu().numpy() - want).max() <= bound
    for seq in (keys, keys - 4):
        qkv = np.concatenate([np.broadcast_to(q[0, :1], (seq, d)).T, k[0, :seq].T, v[0, :seq].T])
        want = _dense_attention(np.array([0, seq], np.int32), np.arange(seq), 1, q[:, :1], k, v, 0.125)[0, 0]
        got = attention_fm(dev(np.ascontiguousarray(qkv)), d, 1, 1, seq)
        assert np.abs(got.cpu().numpy() - want[:, None]).max() <= bound


def _one_key_ahead_of_many(keys, d):
    """q, k, v: key 0 ahead of all others by 25.05 in the base-2 exponent at a scale of 1/8, so that each of their probabilities is just
    under half the smallest that fp16 holds; their values are zero, key 0's is 2047/1024."""
    a, b = np.float16(11.78125), np.float16(11.7890625)
    assert 25.0 < float(a) * float(b) / 8 * np.log2(np.e) < 25.06
    q, k, v = (np.zeros((1, n, d), np.float16) for n in (64, keys, keys))
    q[..., 0], k[0, 0, 0], v[0, 0] = a, b, 2047 / 1024
    return q, k, v


# half a step of fp16 below two, and a few steps of the fp32 sums: without the others' probabilities in the sum the result is 0.95 steps off
_MANY_KEYS_BOUND = 2.0 ** -11 + 2.0 ** -16


@pytest.mark.parametrize("V,d", [(8, 32), (8, 64), (8, 128), (16, 32), (16, 64), (16, 128)])
@pytest.mark.parametrize("pairs", [1, 40, 300])
def test_one_launch_attention_sums_what_fp16_does_not_hold(built_library, V, d, pairs):
    keys = 16384
    q, k, v = _one_key_ahead_of_many(keys, d)
    off = (np.arange(64 // V + 1) * keys).astype(np.int32)
    cols = np.tile(np.arange(keys, dtype=np.int32), 64 // V)
    want = _dense_attention(off, cols, V, q, k, v, 0.125)
    got = sspmm_amd.fused_sparse_attention(None, dev(off), dev(cols), *(dev(t).expand(pairs, -1, -1).contiguous() for t in (q, k, v)), 0.125, V)
    assert np.abs(got.cpu().numpy() - want).max() <= _MANY_KEYS_BOUND


def test_dense_attention_sums_what_fp16_does_not_hold(built_library):
    """(The two waves that share queries keep sums of their own, so half of the keys would count: 0.48 steps of 0.97.)"""
    from sspmm_amd.layers import attention_fm
    seq = 16384
    q, k, v = _one_key_ahead_of_many(seq, 64)
    qkv = np.concatenate([np.broadcast_to(q[0, :1], (seq, 64)).T, k[0].T, v[0].T])
    want = _dense_attention(np.array([0, seq], np.int32), np.arange(seq), 1, q[:, :1], k, v, 0.125)[0, 0]
    got = attention_fm(dev(np.ascontiguousarray(qkv)), 64, 1, 1, seq)
    assert np.abs(got.cpu().numpy() - want[:, None]).max() <= _MANY_KEYS_BOUND


@pytest.mark.parametrize("V,d", [(8, 32), (8, 64), (16, 64), (8, 128), (16, 128)])
def test_one_launch_attention_with_scores_of_any_size(built_library, V, d):
    """Scaled scores from a fraction to 2^32, of either sign: the largest probability is one whatever fp32 makes of its exponent.  A
    score is one exact product, so what is left is the rounding of the probabilities and of the result to fp16, 2^-11 each of values
    up to one, and of the exponents, under 2^-14 while a maximum moves."""
    keys, rows = 133, 64
    rng = np.random.default_rng(V + d)
    q, k = np.zeros((2, rows, d), np.float16), np.zeros((2, keys, d), np.float16)
    q[..., 0] = np.exp2(rng.uniform(-8, 15.9, (2, rows))) * rng.choice([-1.0, 1.0], (2, rows))
    k[..., 0] = np.exp2(rng.uniform(-4, 15.9, (2, keys)))
    k[1] = np.sort(k[1], axis=0)  # (every step moves the maximum)
    v = rng.uniform(-1, 1, (2, keys, d)).astype(np.float16)
    off = (np.arange(rows // V + 1) * keys).astype(np.int32)
    cols = np.tile(np.arange(keys, dtype=np.int32), rows // V)
    want = _dense_attention(off, cols, V, q, k, v, 1.0)
    got = sspmm_amd.fused_sparse_attention(None, dev(off), dev(cols), dev(q), dev(k), dev(v), 1.0, V).cpu().numpy()
    assert np.abs(got - want).max() <= 2.0 ** -10 + 2.0 ** -13


def test_one_launch_attention_at_full_size_by_its_properties(built_library):
    """The benchmark's block (4096 tokens, 90 % of the vectors masked out, 48 heads of 64 features): with every row of
    v the same the probabilities of a row must add up to one, so every query gets that row back; columns stored in
    another order inside the vector-rows change the sums' order only; a permutation of the vector-rows changes nothing."""
    V, seq, heads, d = 8, 4096, 48, 64
    from sspmm_amd.attention import static_random_mask
    cols, off, rows = static_random_mask(seq // V, seq, 0.9, seed=5)
    rng = np.random.default_rng(6)
    shuffled = cols.copy()
    for i in range(len(off) - 1):
        rng.shuffle(shuffled[off[i]:off[i + 1]])
    g = torch.Generator("cuda").manual_seed(7)
    q, k, v = (torch.randn(heads, seq, d, device="cuda", generator=g).half() for _ in range(3))
    const = torch.full((d,), 0.0, device="cuda").half()
    const[::2], const[1::2] = 0.75, -1.5
    v_const = const.expand(heads, seq, d).contiguous()
    d_off, d_cols, d_rows, d_shuf = dev(off), dev(cols), dev(rows), dev(shuffled)
    print("attention at full size: %d vectors per head" % cols.size, flush=True)
    out = sspmm_amd.fused_sparse_attention(None, d_off, d_cols, q, k, v_const, 0.125, V)
    assert (out.float() - const.float()).abs().max().item() <= 2e-3
    a = sspmm_amd.fused_sparse_attention(None, d_off, d_cols, q, k, v, 0.125, V)
    b = sspmm_amd.fused_sparse_attention(d_rows, d_off, d_cols, q, k, v, 0.125, V)
    c = sspmm_amd.fused_sparse_attention(None, d_off, d_shuf, q, k, v, 0.125, V)
    assert torch.equal(a, b)
    assert (a.float() - c.float()).abs().max().item() <= 2e-3
    chain = sspmm_amd.sparse_attention(None, d_off, d_cols, q, k, v, 0.125, V, fused=False)
    assert (a.float() - chain.float()).abs().max().item() <= 4e-3


@pytest.mark.parametrize("d", [40, 256])
def test_heads_of_other_widths_take_the_three_operators(built_library, d):
    """`sparse_attention` with nothing forced: heads that are not 32, 64 or 128 wide run the chain, and `fused=True` says so."""
    V, seq, batch = 8, 128, 2
    vs = _pattern(seq // V, seq, V, 0.75, seed=31)
    off, col = dev(vs.row_offsets), dev(vs.col_idx)
    g = torch.Generator("cuda").manual_seed(32)
    q, k, v = (torch.randn(batch, seq, d, device="cuda", generator=g).half() for _ in range(3))
    out = sspmm_amd.sparse_attention(None, off, col, q, k, v, d ** -0.5, V)
    want = _dense_attention(vs.row_offsets, vs.col_idx, V, *(t.cpu().numpy() for t in (q, k, v)), d ** -0.5)
    assert np.abs(out.float().cpu().numpy() - want).max() <= 1e-2
    with pytest.raises(ValueError):
        sspmm_amd.sparse_attention(None, off, col, q, k, v, d ** -0.5, V, fused=True)


@pytest.mark.parametrize("d", [32, 64, 128])
def test_one_launch_attention_of_a_single_key_returns_its_value_row(built_library, d):
    """A query that attends to one key gets that row of v back exactly (probability one, fp16 in and out)."""
    V, n_keys, m_vec = 8, 50, 5
    rng = np.random.default_rng(3 + d)
    cols = rng.integers(0, n_keys, m_vec).astype(np.int32)
    off = np.arange(m_vec + 1, dtype=np.int32)
    q, k, v = (rng.standard_normal((2, n, d)).astype(np.float16) for n in (m_vec * V, n_keys, n_keys))
    got = sspmm_amd.fused_sparse_attention(None, dev(off), dev(cols), dev(q), dev(k), dev(v), 0.125, V).cpu().numpy()
    for i in range(m_vec):
        assert np.array_equal(got[:, i * V:(i + 1) * V], np.repeat(v[:, cols[i]][:, None], V, axis=1))


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("V", [8, 16])
def test_packed_heads_give_the_bits_of_the_copied_out_heads(built_library, V, d):
    """The launch on a fused projection [seq, batch, 3 * heads * d] against the same launch on q, k and v copied out
    into [batch * heads, seq, d] as the reference's module lays them out (spattention.py:151-157, 181-184)."""
    seq, bsz, heads = 192, 3, 5
    E = heads * d
    vs = _pattern(seq // V, seq, V, 0.7, seed=21)
    off, col = dev(vs.row_offsets), dev(vs.col_idx)
    g = torch.Generator("cuda").manual_seed(22)
    qkv = torch.randn(seq, bsz, 3 * E, device="cuda", generator=g).half()
    got = sspmm_amd.sparse_attention_packed(None, off, col, qkv, heads, 0.125, V)
    torch.cuda.synchronize()
    q, k, v = (t.contiguous().view(seq, bsz * heads, d).transpose(0, 1).contiguous() for t in qkv.chunk(3, dim=-1))
    want = sspmm_amd.fused_sparse_attention(None, off, col, q, k, v, 0.125, V)
    want = want.transpose(0, 1).contiguous().view(seq, bsz, E)
    assert got.shape == (seq, bsz, E)
    assert torch.equal(got, want)
    with pytest.raises(ValueError):
        sspmm_amd.sparse_attention_packed(None, off, col, qkv, heads + 1, 0.125, V)
    from sspmm_amd.attention import packed_attention_fits
    assert packed_attention_fits(8192, 8, 3 * 512) and not packed_attention_fits(16384, 32, 3 * 1024)


def test_argument_errors(built_library):
    off = torch.zeros(3, dtype=torch.int32, device="cuda")
    col = torch.zeros(0, dtype=torch.int32, device="cuda")
    with pytest.raises(ValueError):
        sspmm_amd.sddmm(None, off, col, torch.zeros(16, 64, device="cuda").half(), torch.zeros(8, 64, device="cuda").half(), 4)
    with pytest.raises(ValueError):
        sspmm_amd.sddmm(None, off, col, torch.zeros(16, 64, device="cuda").half(), torch.zeros(8, 32, device="cuda").half(), 8)
    with pytest.raises(TypeError):
        sspmm_amd.csr_softmax(None, off, torch.zeros(0, device="cuda"), 1.0, 8)
    with pytest.raises(ValueError):  # the one-launch block takes heads of 32, 64 or 128 features
        sspmm_amd.fused_sparse_attention(None, off, col, *(torch.zeros(1, 16, 48, device="cuda").half() for _ in range(3)), 1.0, 8)
    with pytest.raises(RuntimeError):  # scale must be positive
        sspmm_amd.fused_sparse_attention(None, off, col, *(torch.zeros(1, 16, 64, device="cuda").half() for _ in range(3)), 0.0, 8)
    with pytest.raises(RuntimeError):  # F must be a multiple of 8
        sspmm_amd.sddmm(None, off, col, torch.zeros(16, 12, device="cuda").half(), torch.zeros(8, 12, device="cuda").half(), 8)


def test_sparse_attention_encoder_matches_dense_masked_attention(built_library):
    """The end-to-end model of the reference (four blocks, each with its own static mask) against the same model
    whose attention is dense fp32 arithmetic with the mask applied as -inf (the recipe of the reference's own checks,
    verify/softmax.py:36-38, verify/spmm.py:36-41)."""
    from sspmm_amd.attention import SparseAttentionEncoder
    torch.manual_seed(3)
    seq, V = 512, 8
    model = SparseAttentionEncoder(vocab_size=257, embed_dim=128, num_heads=2, sparsity=0.9, seq_len=seq, mlp_dim=256,
                                   num_class=16, vec_length=V, layers=4, seed=11).cuda().half().eval()
    tokens = torch.randint(0, 257, (2, seq), device="cuda", generator=torch.Generator("cuda").manual_seed(4))
    masks = []
    for blk in model.blocks:
        off, col = blk.row_offsets.cpu().numpy(), blk.column_indices.cpu().numpy()
        assert off[-1] == col.size == round(0.1 * (seq // V) * seq)
        dense = np.zeros((seq, seq), bool)
        for i in range(seq // V):
            dense[i * V:(i + 1) * V, col[off[i]:off[i + 1]]] = True
        assert np.array_equal(np.sort(np.diff(off)[blk.row_indices.cpu().numpy()]), np.diff(off)[blk.row_indices.cpu().numpy()])
        masks.append(torch.from_numpy(dense).cuda())
    with torch.no_grad():
        got = model(tokens)
        want = model(tokens, dense_masks=masks)
    assert got.shape == (seq, 2, 16) and got.dtype == torch.float16
    assert torch.isfinite(got).all()
    assert max_rel_err(got.float().cpu().numpy(), want.float().cpu().numpy()) <= 1e-2


@pytest.mark.parametrize("E", [64, 128, 256, 512, 1024, 2048])
@pytest.mark.parametrize("outer,inner", [(1, 1), (3, 1), (37, 3), (130, 2)])
def test_row_layernorm_with_residual(built_library, E, outer, inner):
    """Every width, row counts that leave part of a workgroup without a row, x dense and as a batch-major view, with and
    without the residual and the sum.  The sum is exact; statistics in fp32 leave the fp16 rounding of the result."""
    from sspmm_amd.attention import add_layernorm_rows
    g = torch.Generator("cuda").manual_seed(E + outer)
    ln = torch.nn.LayerNorm(E).cuda().half()
    with torch.no_grad():
        ln.weight.copy_(torch.randn(E, device="cuda", generator=g))
        ln.bias.copy_(torch.randn(E, device="cuda", generator=g))
        a = torch.randn(outer, inner, E, device="cuda", generator=g).half()
        for x in ((torch.randn(outer, inner, E, device="cuda", generator=g) * 3 + 1).half(),
                  (torch.randn(inner, outer, E, device="cuda", generator=g) * 3 + 1).half().transpose(0, 1)):
            for res, keep in ((None, False), (a, False), (a, True)):
                total, got = add_layernorm_rows(x, res, ln, keep_sum=keep)
                s = x if res is None else res + x
                want = torch.nn.functional.layer_norm(s.double(), (E,), ln.weight.double(), ln.bias.double(), ln.eps)
                assert got.is_contiguous() and got.shape == (outer, inner, E)
                assert ((got.double() - want).abs() <= 2 ** -10 * want.abs() + 1e-5).all()
                assert (total is None) if not keep else torch.equal(total, s)


def test_encoder_with_fused_norms_matches_the_modules(built_library):
    """The encoder's inference path against its modules called one by one, which a hook on any of them, autograd or
    autocast still get."""
    from sspmm_amd import attention as A
    model = A.SparseAttentionEncoder(50, 128, 4, 0.9, 96, 192, 16, vec_length=8, layers=3, seed=2).cuda().half().eval()
    tokens = torch.randint(0, 50, (3, 96), device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    calls = []
    plain = A.add_layernorm_rows
    A.add_layernorm_rows = lambda *args, **kw: (calls.append(1), plain(*args, **kw))[1]
    try:
        with torch.no_grad():
            fused = model(tokens)
            assert len(calls) == 7
            handle = model.blocks[1].layer_norm2.register_forward_hook(lambda m, i, o: calls.append("hook"))
            modules = model(tokens)
            handle.remove()
        assert calls[7:] == ["hook"]
        with_grad = model(tokens)
        assert with_grad.requires_grad and len(calls) == 8
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16):
            model(tokens)
        assert len(calls) == 8
    finally:
        A.add_layernorm_rows = plain
    # (both round every activation to fp16; a LayerNorm that differs by an ulp moves the sums behind it by as much)
    scale = modules.float().pow(2).mean().sqrt()
    assert (fused.float() - modules.float()).abs().max() <= 1e-2 * scale
    assert torch.equal(with_grad.detach(), modules)


def _block_by_modules(x, attn, blk, norm, tail):
    """float64, with the roundings to fp16 that an activation written to memory has: (x', out)."""
    lin = lambda m, t: t @ m.weight.double().t() + m.bias.double()  # noqa: E731
    ln = lambda m, t: torch.nn.functional.layer_norm(t, m.normalized_shape, m.weight.double(), m.bias.double(), m.eps)  # noqa: E731
    r = x.double()
    if attn is not None:
        n = ln(blk.layer_norm2, lin(blk.out_proj, attn.double()) + r).half().double()
        r = (lin(blk.linear2, lin(blk.linear1, n).half().double()) + r).half().double()
    h = ln(norm, r)
    return r, h if tail is None else lin(tail, h.half().double())


@pytest.mark.parametrize("E,mlp,n_out", [(128, 256, 64), (128, 1024, 384), (256, 256, 320), (256, 1024, 768), (512, 512, 1536)])
@pytest.mark.parametrize("outer,inner", [(1, 1), (33, 1), (127, 3), (4096, 1), (4097, 1), (2731, 3)])
def test_block_dense_in_one_launch(built_library, E, mlp, n_out, outer, inner):
    """Every width and tile of tokens (16, 32, 64) with a last tile that is not full, output widths that leave waves without a
    chunk, x dense and batch-major, with and without attention, tail and x'.  Roundings to fp16 at other places (a
    hidden activation an ulp away, 2^-11) stay below 4 * 2^-11 of the result's size after the sums behind them."""
    from sspmm_amd.attention import SparseAttentionBlock, block_dense
    g = torch.Generator("cuda").manual_seed(E + outer + n_out)
    none = torch.zeros(1, dtype=torch.int32)
    torch.manual_seed(E + n_out)
    blk = SparseAttentionBlock(E, mlp, E // 32, none, none, none).cuda().half()
    norm, tail = torch.nn.LayerNorm(E).cuda().half(), torch.nn.Linear(E, n_out).cuda().half()
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).half()  # noqa: E731
    with torch.no_grad():
        for m in (norm, blk.layer_norm2):
            m.weight.copy_(1 + 0.2 * rnd(E))
            m.bias.copy_(rnd(E))
        attn = rnd(outer, inner, E)
        close = lambda got, want: ((got.double() - want).abs().max() <= 4 * 2 ** -11 * want.abs().max()).item()  # noqa: E731
        for x in (rnd(outer, inner, E) * 2 + 1, (rnd(inner, outer, E) * 2 + 1).transpose(0, 1)):
            for a, last, keep in ((attn, tail, True), (attn, None, False), (None, tail, False), (None, None, True)):
                kept, got = block_dense(x, a, blk, norm, last, keep_x=keep)
                want_x, want = _block_by_modules(x, a, blk, norm, last)
                assert got.is_contiguous() and got.shape == (outer, inner, n_out if last is not None else E)
                if a is None:  # an embedding in the place of x: the same values as torch makes of it
                    pos = rnd(outer, 1, E)
                    embedded = x * 16.0 + pos
                    made, from_table = block_dense(x, a, blk, norm, last, keep_x=True, pos=pos, scale=16.0)
                    assert torch.equal(made, embedded) and torch.equal(from_table, block_dense(embedded, a, blk, norm, last)[1])
                    # (torch rounds the scaled product to fp16 once, the kernel to fp32 first: an ulp of it apart at a tie)
                    other = block_dense(x, a, blk, norm, last, keep_x=True, pos=pos, scale=11.3)[0]
                    assert ((other.float() - (x * 11.3 + pos).float()).abs() <= 2 ** -10 * (x.float() * 11.3).abs() + 2 ** -10 * other.float().abs()).all()
                if last is not None and n_out % E == 0:  # the same split into heads
                    for d in (32, 64, 128):
                        split = block_dense(x, a, blk, norm, last, head_dim=d)[1]
                        assert torch.equal(split, got.view(outer, inner, n_out // E, E // d, d).permute(2, 1, 3, 0, 4))
                assert close(got, want), (a is None, last is None, (got.double() - want).abs().max().item(), want.abs().max().item())
                assert (kept is None) if not keep else (torch.equal(kept, x) if a is None else close(kept, want_x))


@pytest.mark.parametrize("d,heads", [(32, 4), (64, 3), (128, 2)])
@pytest.mark.parametrize("V", [8, 16])
def test_attention_on_split_heads_is_the_packed_one(built_library, V, d, heads):
    """The same launch on other strides: bit for bit, with and without a permutation of the rows."""
    seq, bsz = 208, 3
    vs = _pattern(seq // V, seq, V, 0.8, seed=d)
    qkv = torch.randn(seq, bsz, 3 * heads * d, device="cuda", generator=torch.Generator("cuda").manual_seed(d)).half()
    split = qkv.view(seq, bsz, 3, heads, d).permute(2, 1, 3, 0, 4).contiguous()
    off, col = dev(vs.row_offsets), dev(vs.col_idx)
    want = sspmm_amd.attention.sparse_attention_packed(None, off, col, qkv, heads, 0.2, V)
    for rows in (None, torch.randperm(seq // V, device="cuda").int()):
        assert torch.equal(sspmm_amd.attention.sparse_attention_split(rows, off, col, split, 0.2, V), want)


@pytest.mark.parametrize("embed,heads,classes", [(128, 4, 64), (256, 8, 16), (512, 8, 256)])
def test_encoder_in_two_launches_per_block_matches_the_modules(built_library, embed, heads, classes):
    """A head of a width that the launch does not take stays a module's; a hook on a linear layer gets its module called."""
    from sspmm_amd import attention as A
    model = A.SparseAttentionEncoder(50, embed, heads, 0.9, 96, 256, classes, vec_length=8, layers=3, seed=2).cuda().half().eval()
    tokens = torch.randint(0, 50, (3, 96), device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    calls = []
    plain = A.block_dense
    A.block_dense = lambda *args, **kw: (calls.append(1), plain(*args, **kw))[1]
    try:
        with torch.no_grad():
            fused = model(tokens)
            assert len(calls) == 4
            handle = model.blocks[1].linear1.register_forward_hook(lambda m, i, o: calls.append("hook"))
            norms = model(tokens)
            handle.remove()
        assert calls[4:] == ["hook"]
        modules = model(tokens)
        assert modules.requires_grad and len(calls) == 5
    finally:
        A.block_dense = plain
    scale = modules.float().pow(2).mean().sqrt()  # (as above)
    assert (fused.float() - modules.float()).abs().max() <= 1e-2 * scale
    assert (norms.float() - modules.float()).abs().max() <= 1e-2 * scale


@pytest.mark.parametrize("V", [8, 16])
@pytest.mark.parametrize("scaler", [0.3, -0.7])
def test_softmax_with_masked_entries(built_library, V, scaler):
    """Entries that a mask of the far infinity (or of the type's far end) takes out, in rows around what a wave keeps in registers
    (256 and 512 vectors), some of which keep one entry: against float64, half an fp16 ulp of a result up to 1 and what
    the base-2 exponential adds in fp32 (2^-20 relative)."""
    rng = np.random.default_rng(V)
    lens = np.array([1, 2, 63, 64, 65, 255, 256, 257, 511, 512, 513, 700])
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    x = (rng.standard_normal((off[-1], V)) * 5).astype(np.float16)
    masked = rng.random(x.shape) < 0.5
    masked[off[:-1]] = False
    far = -np.sign(scaler) * np.where(rng.random(x.shape) < 0.5, np.inf, 65504)
    x = np.where(masked, far, x).astype(np.float16)
    got = sspmm_amd.csr_softmax(None, dev(off), dev(x.reshape(-1)), scaler, V).cpu().numpy().reshape(-1, V).astype(np.float64)
    for i in range(len(lens)):
        z = x[off[i]:off[i + 1]].astype(np.float64) * scaler
        e = np.exp(z - z.max(axis=0))
        want = e / e.sum(axis=0)
        assert (np.abs(got[off[i]:off[i + 1]] - want) <= want * (2.0 ** -11 + 2.0 ** -20) + 2.0 ** -24).all()


@pytest.mark.parametrize("mlp,classes", [(256, 2 ** 20 + 64), (2 ** 20 + 256, 64)])
def test_encoder_with_more_features_than_the_dense_launch_takes(built_library, mlp, classes):
    """A head or a hidden layer of more than 2^20 features runs on the modules, as wide ones of any other size do."""
    from sspmm_amd import attention as A
    model = A.SparseAttentionEncoder(10, 128, 4, 0.5, 16, mlp, classes, vec_length=8, layers=1, seed=2).cuda().half().eval()
    tokens = torch.randint(0, 10, (1, 16), device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    with torch.no_grad():
        got = model(tokens)
    want = model(tokens).detach()  # (with gradients: the modules one by one)
    assert got.shape == (16, 1, classes)
    scale = want.float().pow(2).mean().sqrt()
    assert (got.float() - want.float()).abs().max() <= 1e-2 * scale


@pytest.mark.parametrize("embed,mlp,classes,batch,launches,with_head", [(512, 4096, 4096, 1, 3, True), (512, 4352, 64, 1, 0, None), (512, 4352, 64, 43, 3, True),
                                                                        (256, 512, 8192, 1, 3, True), (256, 512, 8256, 1, 3, False),
                                                                        (128, 16384, 64, 1, 3, True), (128, 16640, 64, 1, 0, None)])
def test_wide_hidden_layers_and_heads_go_to_the_library(built_library, embed, mlp, classes, batch, launches, with_head):
    """Either side of the sizes up to which one launch per block beats the products one by one (hidden layers: of up to 4096
    tokens; 43 x 96 are more), with the results of the modules."""
    from sspmm_amd import attention as A
    model = A.SparseAttentionEncoder(50, embed, 4, 0.9, 96, mlp, classes, vec_length=8, layers=2, seed=2).cuda().half().eval()
    tokens = torch.randint(0, 50, (batch, 96), device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    tails = []
    plain = A.block_dense
    A.block_dense = lambda x, attn, block, norm, tail=None, *args, **kw: (tails.append(tail), plain(x, attn, block, norm, tail, *args, **kw))[1]
    try:
        with torch.no_grad():
            got = model(tokens)
    finally:
        A.block_dense = plain
    assert len(tails) == launches and (not tails or (tails[-1] is not None) == with_head)
    want = model(tokens).detach()  # (with gradients: the modules one by one)
    scale = want.float().pow(2).mean().sqrt()
    assert (got.float() - want.float()).abs().max() <= 1e-2 * scale


@pytest.mark.parametrize("V", [8, 16])
@pytest.mark.parametrize("batch,lens", [(3, [1, 63, 64, 65, 0, 128, 129, 191]), (2, [207, 208, 209, 208]), (2, [209, 208, 209, 210]),
                                        (2, [255, 256, 257, 300]), (1, [511, 512, 513, 1100, 0, 3])])
@pytest.mark.parametrize("scaler", [0.3, -0.7, 0.0])
def test_softmax_either_side_of_its_kernels(built_library, V, batch, lens, scaler):
    """Rows up to and beyond what a wave's slots hold, mean lengths either side of 208 (where 16-row vectors change kernels), a scaler
    of either sign and none: against float64, half an fp16 ulp of a result up to 1 and 2^-20 for the exponential.  In place
    and without a stride (the single product) the same bits as that."""
    from sspmm_amd import _lib
    rng = np.random.default_rng(len(lens) + V)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    x = (rng.standard_normal((batch, off[-1], V)) * 4).astype(np.float16)
    got = sspmm_amd.bcsr_softmax(None, dev(off), dev(x.reshape(batch, -1)), scaler, V, batch).cpu().numpy().reshape(batch, -1, V).astype(np.float64)
    for i in range(len(lens)):
        z = x[:, off[i]:off[i + 1]].astype(np.float64) * scaler
        if lens[i] == 0:
            continue
        e = np.exp(z - z.max(axis=1, keepdims=True))
        want = e / e.sum(axis=1, keepdims=True)
        assert (np.abs(got[:, off[i]:off[i + 1]] - want) <= want * (2.0 ** -11 + 2.0 ** -20) + 2.0 ** -24).all()
    one = dev(x[0].reshape(-1))
    assert _lib.lib().sspmm_softmax_f16(len(lens), V, None, dev(off).data_ptr(), one.data_ptr(), scaler, one.data_ptr(),
                                        torch.cuda.current_stream().cuda_stream) == 0
    assert np.abs(one.cpu().numpy().reshape(-1, V).astype(np.float64) - got[0]).max() <= 2.0 ** -11


@pytest.mark.parametrize("count", [1, 48, 49, 100])
def test_packed_weights_hold_every_fragment_where_the_kernel_reads_it(built_library, count):
    """More matrices than one launch of the packing takes, of every group size and of different shapes: groups of rows, in each
    units of 64 columns (32 for groups of 128), in each a 1 KB piece per 32 columns and 16 rows, in it 16 bytes per lane."""
    from sspmm_amd.attention import pack_weights
    g = torch.Generator("cuda").manual_seed(count)
    linears, groups, want = [], [], []
    for i in range(count):
        group = (32, 64, 128)[i % 3]
        rows, cols = group * (1 + i % 4), 64 * (1 + i % 5)
        m = torch.nn.Linear(cols, rows).cuda().half()
        with torch.no_grad():
            m.weight.copy_(torch.randint(-2000, 2000, (rows, cols), device="cuda", generator=g))
        linears.append(m)
        groups.append(group)
        nj, unit = group // 16, 32 if group == 128 else 64
        w = m.weight.detach().cpu().numpy().reshape(rows // group, nj // 2, 4, 2, 4, cols // unit, unit // 32, 4, 8)
        # (group, pair of tiles, lane % 16 / 4, tile of the pair, lane % 4, unit, step, lane / 16, half) -> as the waves load them
        want.append(w.transpose(0, 5, 6, 1, 3, 7, 2, 4, 8).reshape(-1))
    packed = pack_weights(linears, groups)
    for i in range(count):
        assert np.array_equal(packed[i].cpu().numpy(), want[i]), i


def _two_layers(E, mlp, count, g, size=1.0, bias=True):
    from sspmm_amd.attention import SparseAttentionBlock
    none = torch.zeros(1, dtype=torch.int32)
    blocks = []
    for _ in range(count):
        b = SparseAttentionBlock(E, mlp, E // 32, none, none, none).cuda().half()
        with torch.no_grad():
            for m in (b.linear1, b.linear2):
                m.weight.copy_(torch.randn(m.weight.shape, device="cuda", generator=g) * size * m.in_features ** -0.5)
                m.bias.copy_(torch.randn(m.bias.shape, device="cuda", generator=g))
            for m in (b.layer_norm1, b.layer_norm2):
                m.weight.copy_(1 + 0.2 * torch.randn(E, device="cuda", generator=g))
                m.bias.copy_(torch.randn(E, device="cuda", generator=g))
        if not bias:
            b.linear1.bias = b.linear2.bias = b.out_proj.bias = None
        blocks.append(b)
    return blocks


@pytest.mark.parametrize("E,mlp,count,size,bias", [(128, 256, 1, 1.0, True), (128, 1280, 17, 2.0 ** -9, True), (256, 256, 2, 1.0, False),
                                                   (256, 1024, 33, 4.0, True), (512, 512, 3, 1.0, True), (512, 256, 1, 2.0 ** -6, True)])
def test_two_linear_layers_as_one_matrix(built_library, E, mlp, count, size, bias):
    """What one to three launches leave of pairs of linear layers, against their product in float64: an element's rounding to fp16 (2^-11
    of it, or half the smallest step of fp16, 2^-25, next to a largest element of 2^13 or more), and that of the fp32 sums, 2^-24 of their
    terms each.  Weights whose products fp16 would not hold unscaled, a row of zeros, and one with an infinity."""
    from sspmm_amd.attention import fold_blocks, pack_weights
    g = torch.Generator("cuda").manual_seed(E + mlp)
    blocks = _two_layers(E, mlp, count, g, size, bias)
    with torch.no_grad():
        blocks[0].linear2.weight[3] = 0
        blocks[-1].linear2.weight[5, 7] = float("inf")
    packed, folded = fold_blocks(blocks, [b.out_proj for b in blocks], [E // 4] * count)
    group = E // 4
    nj, unit = group // 16, 32 if group == 128 else 64
    for b, (matrix, affine) in zip(blocks, folded):
        got = matrix.cpu().numpy().astype(np.float64).reshape(E // group, E // unit, unit // 32, nj // 2, 2, 4, 4, 4, 8)
        # (the inverse of the order in which the waves load: see test_packed_weights_hold_every_fragment_where_the_kernel_reads_it)
        got = got.transpose(0, 3, 6, 4, 7, 1, 2, 5, 8).reshape(E, E)
        down, shift = affine.cpu().numpy().astype(np.float64).reshape(2, E)
        w1, w2 = (m.weight.detach().cpu().numpy().astype(np.float64) for m in (b.linear1, b.linear2))
        b1, b2 = ((m.bias.detach().cpu().numpy().astype(np.float64) if bias else np.zeros(m.out_features)) for m in (b.linear1, b.linear2))
        with np.errstate(invalid="ignore"):
            want, terms, want_shift = w2 @ w1, np.abs(w2) @ np.abs(w1), w2 @ b1 + b2
            finite = np.isfinite(want).all(1)
            assert finite.sum() == E - (b is blocks[-1]) and not np.isfinite(got[~finite]).any()
            most = np.abs(got).max(1)
            assert (np.log2(down) % 1 == 0).all() and ((most[finite] >= 2 ** 13) & (most[finite] <= 2 ** 14) | (most[finite] == 0)).all()
            bound = 2.0 ** -11 * np.abs(want) + (2.0 ** -25 * down)[:, None] + mlp * 2.0 ** -24 * terms
            assert (np.abs(got * down[:, None] - want)[finite] <= bound[finite]).all()
            assert (np.abs(shift - want_shift)[finite] <= (mlp * 2.0 ** -24 * (np.abs(w2) @ np.abs(b1)) + 2.0 ** -23 * np.abs(b2) + 1e-30)[finite]).all()
    for one, other in zip(packed, pack_weights([b.out_proj for b in blocks], [E // 4] * count)):
        assert torch.equal(one, other)


@pytest.mark.parametrize("E,mlp,n_out,outer,inner", [(128, 256, 128, 1, 1), (128, 512, 64, 70, 61), (256, 1024, 768, 37, 3), (256, 256, 64, 1433, 3),
                                                     (256, 512, 256, 2731, 3), (512, 256, 1536, 19, 1), (512, 512, 64, 1366, 3), (512, 256, 512, 2731, 3)])
def test_block_dense_on_one_matrix_for_two_layers(built_library, E, mlp, n_out, outer, inner):
    """Every width and tile of tokens (16, 32, 64) with a last tile that is not full; with and without a tail, x', biases.  The bound is
    that of test_block_dense_in_one_launch: the hidden features are not rounded, the matrix is to 2^-22 (what that is worth where the first layer
    cancels, test_two_linear_layers_as_one_where_the_first_cancels says; here nothing does)."""
    lin = lambda m, t: t @ m.weight.double().t() + (0 if m.bias is None else m.bias.double())  # noqa: E731
    ln = lambda m, t: torch.nn.functional.layer_norm(t, m.normalized_shape, m.weight.double(), m.bias.double(), m.eps)  # noqa: E731
    from sspmm_amd.attention import block_dense, fold_blocks
    g = torch.Generator("cuda").manual_seed(E + outer)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).half()  # noqa: E731
    for bias in (True, False):
        blk, = _two_layers(E, mlp, 1, g, bias=bias)
        norm, tail = torch.nn.LayerNorm(E).cuda().half(), torch.nn.Linear(E, n_out, bias=bias).cuda().half()
        attn, x = rnd(outer, inner, E), (rnd(inner, outer, E) * 2 + 1).transpose(0, 1)
        for last, keep in ((tail, True), (None, False)):
            with torch.no_grad():
                packed, folded = fold_blocks([blk], [blk.out_proj] + [tail] * (last is not None), [E // 4] + [64] * (last is not None))
                kept, got = block_dense(x, attn, blk, norm, last, keep_x=keep, packed=packed, folded=folded[0])
                n = ln(blk.layer_norm2, lin(blk.out_proj, attn.double()) + x.double()).half().double()
                want_x = (lin(blk.linear2, lin(blk.linear1, n)) + x.double()).half().double()
                h = ln(norm, want_x)
                want = h if last is None else lin(last, h.half().double())
                assert ((got.double() - want).abs().max() <= 4 * 2 ** -11 * want.abs().max()).item()
                assert (kept is None) if not keep else ((kept.double() - want_x).abs().max() <= 4 * 2 ** -11 * want_x.abs().max()).item()
                if last is not None and n_out % E == 0:
                    for d in (32, 64, 128):
                        split = block_dense(x, attn, blk, norm, last, packed=packed, folded=folded[0], head_dim=d)[1]
                        assert torch.equal(split, got.view(outer, inner, n_out // E, E // d, d).permute(2, 1, 3, 0, 4))


def _unpacked(matrix, E):
    """A folded matrix of E x E out of the order in which the waves load it."""
    group = E // 4
    nj, unit = group // 16, 32 if group == 128 else 64
    w = matrix.cpu().numpy().astype(np.float64).reshape(E // group, E // unit, unit // 32, nj // 2, 2, 4, 4, 4, 8)
    return w.transpose(0, 3, 6, 4, 7, 1, 2, 5, 8).reshape(E, E)


@pytest.mark.parametrize("E,mlp,count", [(128, 256, 17), (128, 1280, 1), (256, 512, 3), (512, 256, 2)])
def test_two_linear_layers_as_two_matrices(built_library, E, mlp, count):
    """The matrix and what its rounding leaves hold 22 bits: of integers up to 15 the sums need 19 at most (225 x 1280), so the two are
    the product itself.  Of an element that is not finite nothing is left."""
    from sspmm_amd.attention import fold_blocks
    g = torch.Generator("cuda").manual_seed(E + mlp)
    blocks = _two_layers(E, mlp, count, g)
    with torch.no_grad():
        for b in blocks:
            for m in (b.linear1, b.linear2):
                m.weight.copy_(torch.randint(-15, 16, m.weight.shape, device="cuda", generator=g).half())
        blocks[-1].linear2.weight[5, 7] = float("inf")
        folded = fold_blocks(blocks, [b.out_proj for b in blocks], [E // 4] * count)[1]
    for b, pair in zip(blocks, folded):
        w1, w2 = (m.weight.detach().cpu().numpy().astype(np.float64) for m in (b.linear1, b.linear2))
        down = pair[1][:E].cpu().numpy().astype(np.float64)[:, None]
        matrix, rest = _unpacked(pair[0], E), _unpacked(pair.rest, E)
        rows = np.arange(E) != (5 if b is blocks[-1] else -1)
        assert np.array_equal(((matrix + rest) * down)[rows], (w2 @ w1)[rows]) and np.abs(rest).max() > 0
        assert not np.isfinite(matrix[~rows]).any() and (rest[~rows] == 0).all()


@pytest.mark.parametrize("E,tokens", [(128, 37), (256, 5000), (512, 9000)])
def test_folded_entries_without_what_the_rounding_leaves(built_library, E, tokens):
    """The C entries with the matrix alone: the same matrix, and of weights whose products it holds exactly (halves up to 1.5, 256 hidden features,
    one in 32 not zero: sums of 8 on average) the result with the remainder, which is zero then, to the order of the fp32 sums."""
    import ctypes as C
    from sspmm_amd.attention import block_dense, fold_blocks
    g = torch.Generator("cuda").manual_seed(E)
    blk, = _two_layers(E, 256, 1, g)
    L, stream = _lib.lib(), torch.cuda.current_stream().cuda_stream
    with torch.no_grad():
        for m in (blk.linear1, blk.linear2):
            w = torch.randint(-3, 4, m.weight.shape, device="cuda", generator=g) * 0.5
            m.weight.copy_(w * (torch.rand(m.weight.shape, device="cuda", generator=g) < 1 / 32))
        packed, (pair,) = fold_blocks([blk], [blk.out_proj], [E // 4])
        assert (pair.rest == 0).all()
        x, attn = torch.randn(tokens, 1, E, device="cuda", generator=g).half(), torch.randn(tokens, 1, E, device="cuda", generator=g).half()
        want = block_dense(x, attn, blk, blk.layer_norm1, keep_x=True, packed=packed, folded=pair)
    w21, affine, kept, out = torch.empty_like(pair[0]), torch.empty_like(pair[1]), torch.empty_like(x), torch.empty_like(x)
    one = lambda t: (C.c_void_p * 1)(t.data_ptr())  # noqa: E731
    assert L.sspmm_block_fold_f16(0, None, None, None, None, None, 1, E, (C.c_int32 * 1)(256), one(blk.linear1.weight), one(blk.linear1.bias),
                                  one(blk.linear2.weight), one(blk.linear2.bias), w21.data_ptr(), affine.data_ptr(), stream) == 0
    assert torch.equal(w21, pair[0]) and torch.equal(affine, pair[1])
    ln2, ln1 = blk.layer_norm2, blk.layer_norm1
    assert L.sspmm_block_dense_folded_f16(tokens, 1, E, x.data_ptr(), E, E, attn.data_ptr(), packed[0].data_ptr(), blk.out_proj.bias.data_ptr(),
                                          ln2.weight.data_ptr(), ln2.bias.data_ptr(), ln2.eps, w21.data_ptr(), affine.data_ptr(), ln1.weight.data_ptr(),
                                          ln1.bias.data_ptr(), ln1.eps, 0, 0, None, None, kept.data_ptr(), out.data_ptr(), stream) == 0
    for got, ref in zip((kept, out), want):  # (one step of fp16 where a sum lies next to the middle of two)
        assert (got.double() - ref.double()).abs().max() <= 2.0 ** -10 * ref.double().abs().max()


@pytest.mark.parametrize("E,mlp,tokens", [(128, 256, 333), (256, 1024, 500), (256, 512, 4100), (512, 1024, 40), (512, 512, 4100)])
@pytest.mark.parametrize("kind", ["offset", "shift", "centred"])
def test_two_linear_layers_as_one_where_the_first_cancels(built_library, E, mlp, tokens, kind):
    """Rows of the first layer with a part that a LayerNorm's output of mean zero cancels, a large beta that the first bias takes back, and
    rows without a mean under a beta: the largest and the root mean square of the error against float64 are no larger than those of the
    layers one after the other, where these cancel before anything is rounded.  (Both end in a rounding to fp16; the output
    projection is zero, and every second feature of a token 1 and -1, so that the LayerNorm's output is known exactly.)"""
    from sspmm_amd.attention import block_dense, fold_blocks, pack_weights
    g = torch.Generator("cuda").manual_seed(E + mlp + tokens)
    blk, = _two_layers(E, mlp, 1, g)
    gamma, beta = {"offset": (1.0, 0.0), "shift": (2.0 ** -4, 8.0), "centred": (0.25, 1.0)}[kind]
    with torch.no_grad():
        blk.out_proj.weight.zero_(), blk.out_proj.bias.zero_(), blk.linear2.bias.zero_()
        blk.layer_norm2.weight.fill_(gamma), blk.layer_norm2.bias.fill_(beta)
        w1, b1 = blk.linear1.weight, blk.linear1.bias
        if kind == "offset":
            w1.add_(torch.randn(mlp, 1, device="cuda", generator=g).half())  # (sixteen deviations of the rest at 256 features)
        elif kind == "centred":
            w1.sub_(w1.double().mean(1, keepdim=True).half())
        b1.copy_(-(w1.double().sum(1) * beta).half())
        sign = torch.rand(tokens, E, device="cuda", generator=g).argsort(1) % 2 * 2.0 - 1.0
        x = sign.half().view(tokens, 1, E)
        n = sign.double() * gamma + beta
        want = (n @ w1.double().t() + b1.double()) @ blk.linear2.weight.double().t() + sign.double()
        norm, attn = blk.layer_norm1, torch.zeros_like(x)
        two = block_dense(x, attn, blk, norm, keep_x=True, packed=pack_weights([blk.out_proj, blk.linear1, blk.linear2], [E // 4, 64, E // 4]))[0]
        packed, folded = fold_blocks([blk], [blk.out_proj], [E // 4])
        one = block_dense(x, attn, blk, norm, keep_x=True, packed=packed, folded=folded[0])[0]
    off = [(t.view(tokens, E).double() - want).abs() for t in (one, two)]
    assert off[0].max() <= off[1].max() and off[0].square().mean() <= off[1].square().mean()


@pytest.mark.parametrize("E,outer,inner", [(128, 2000, 1), (256, 1001, 2), (256, 700, 5), (128, 37, 7), (256, 9, 31), (512, 5, 64), (128, 3, 1000), (256, 2, 4097)])
def test_block_dense_finds_a_tokens_place(built_library, E, outer, inner):
    """Token / inner by a product: the bits of one long sequence, whatever it is cut into, x batch-major, out dense and split into
    heads, and an embedding's positions; LayerNorms without weights are those with ones and zeros."""
    from sspmm_amd.attention import block_dense, fold_blocks
    g = torch.Generator("cuda").manual_seed(E + inner)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).half()  # noqa: E731
    blk, = _two_layers(E, 256, 1, g)
    norm, tail = torch.nn.LayerNorm(E).cuda().half(), torch.nn.Linear(E, E).cuda().half()
    plain = torch.nn.LayerNorm(E, elementwise_affine=False)
    x, attn, pos, T = rnd(inner, outer, E).transpose(0, 1), rnd(outer, inner, E), rnd(outer, 1, E), outer * inner
    with torch.no_grad():
        packed, folded = fold_blocks([blk], [blk.out_proj, tail], [E // 4, 64])
        whole = block_dense(x.reshape(T, 1, E), attn.view(T, 1, E), blk, norm, tail, True, packed, 0, folded=folded[0])
        kept, got = block_dense(x, attn, blk, norm, tail, True, packed, 0, folded=folded[0])
        split = block_dense(x, attn, blk, plain, tail, False, packed, 32, folded=folded[0])[1]
        assert torch.equal(kept.view(T, 1, E), whole[0]) and torch.equal(got.view(T, 1, E), whole[1])
        assert torch.equal(split, got.view(outer, inner, 1, E // 32, 32).permute(2, 1, 3, 0, 4))
        want = block_dense(x.reshape(T, 1, E), None, None, norm, tail, True, packed[1:], 0, pos.expand(outer, inner, E).reshape(T, 1, E), 3.0)
        kept, got = block_dense(x, None, None, plain, tail, True, packed[1:], 0, pos, 3.0)
        assert torch.equal(kept.view(T, 1, E), want[0]) and torch.equal(got.view(T, 1, E), want[1])


@pytest.mark.parametrize("E,outer,inner", [(128, 5, 1), (128, 1367, 3), (256, 37, 3), (256, 1400, 3), (512, 2731, 3), (512, 19, 2)])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_block_dense_looks_tokens_up(built_library, E, outer, inner, dtype):
    """The rows of a table in the place of the embedding, for every width and tile of tokens: the same bits, whatever the tokens'
    strides; a token that is no row of the table makes a row of NaN and leaves the others alone."""
    from sspmm_amd.attention import block_dense, pack_weights
    g = torch.Generator("cuda").manual_seed(E + outer)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).half()  # noqa: E731
    norm, tail = torch.nn.LayerNorm(E).cuda().half(), torch.nn.Linear(E, 3 * E).cuda().half()
    table, pos = rnd(50, E), rnd(outer, 1, E)
    wide = torch.randint(0, 50, (2 * inner, 3 * outer), device="cuda", generator=g).to(dtype)
    with torch.no_grad():
        packed = pack_weights([tail], [64])
        for tokens in (wide[:inner, :outer].contiguous(), wide[::2, ::3], wide[:inner, :outer].t().contiguous().t()):
            assert tokens.shape == (inner, outer)
            x = table[tokens.long()].transpose(0, 1)
            for d in (0, 32):
                want = block_dense(x, None, None, norm, tail, True, packed, d, pos, 11.3)
                got = block_dense(tokens, None, None, norm, tail, True, packed, d, pos, 11.3, table=table)
                assert torch.equal(want[0], got[0]) and torch.equal(want[1], got[1])
        tokens = wide[:inner, :outer].contiguous()
        tokens[0, 1], tokens[inner - 1, 0] = 50, -1
        kept, out = block_dense(tokens, None, None, norm, tail, True, packed, 0, pos, 11.3, table=table)
    lost = ((tokens < 0) | (tokens >= 50)).t()
    assert torch.equal(kept.isnan().all(-1), lost) and torch.equal(out.isnan().any(-1), lost)


def test_encoder_looks_tokens_up_in_its_first_launch(built_library):
    """Tokens of either type and any strides give the bits of the embedding called as a module, which a hook on it, a limit on the
    rows' norm and tokens that a kernel does not read get."""
    from sspmm_amd import attention as A
    model = A.SparseAttentionEncoder(50, 128, 4, 0.9, 96, 256, 64, vec_length=8, layers=2, seed=2).cuda().half().eval()
    tokens = torch.randint(0, 50, (3, 96), device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    tables, plain = [], A.block_dense
    A.block_dense = lambda *args, **kw: (tables.append(kw.get("table")), plain(*args, **kw))[1]
    try:
        with torch.no_grad():
            got = [model(t) for t in (tokens, tokens.int(), tokens.t().contiguous().t(), torch.stack([tokens, tokens], -1)[..., 1])]
            assert len(tables) == 12 and all((t is model.encoder.weight) == (i % 3 == 0) for i, t in enumerate(tables))
            del tables[:]
            seen = []
            handle = model.encoder.register_forward_hook(lambda m, i, o: seen.append(1))
            want = model(tokens)
            handle.remove()
            assert seen and all(torch.equal(want, t) for t in got)
            model.encoder.max_norm = 1e4
            assert torch.equal(model(tokens), want)
            model.encoder.max_norm = None
            assert len(tables) == 6 and all(t is None for t in tables)
            with pytest.raises(RuntimeError):
                model(tokens.short())
    finally:
        A.block_dense = plain


@pytest.mark.parametrize("embed,heads,mlp,V", [(128, 4, 512, 8), (256, 8, 1024, 16), (512, 8, 512, 8), (192, 6, 512, 8), (1024, 16, 512, 16)])
def test_encoder_against_float64(built_library, embed, heads, mlp, V):
    """The whole model on each of its routes (two launches a block, fused norms, and for 192 features the modules) against dense
    masked attention in float64.  An activation's rounding to fp16 is 2^-11 / sqrt(3) of it in the mean; the residual stream is
    rounded once per block and each block adds what came from five further roundings at a fraction of its size: four
    times the one rounding in all (measured 5.1 to 6.0e-4)."""
    import copy
    from sspmm_amd.attention import SparseAttentionEncoder
    seq = 160
    model = SparseAttentionEncoder(50, embed, heads, 0.8, seq, mlp, 64, vec_length=V, layers=4, seed=3).cuda().half().eval()
    tokens = torch.randint(0, 50, (3, seq), device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    masks = []
    for b in model.blocks:
        rows = torch.repeat_interleave(torch.arange(seq // V, device="cuda"), b.row_offsets.diff().long())
        mask = torch.zeros(seq // V, V, seq, dtype=torch.bool, device="cuda")
        mask[rows, :, b.column_indices.long()] = True
        masks.append(mask.view(seq, seq))
    with torch.no_grad():
        got = model(tokens).double()
        want = copy.deepcopy(model).double()(tokens, masks)
    error = ((got - want).norm() / want.norm()).item()
    print("embed %d: relative error %.2e" % (embed, error), flush=True)
    assert error <= 4 * 2.0 ** -11 / 3 ** 0.5


@pytest.mark.parametrize("embed,mlps", [(128, (256, 512)), (256, (256, 512, 256)), (512, (512, 256, 768)), (256, (1024, 256, 512, 256))])
def test_encoder_folds_the_layers_that_are_wider_than_the_model(built_library, embed, mlps):
    """Blocks with hidden layers of both kinds behind one another: the bound of test_encoder_against_float64, against the same."""
    import copy
    from sspmm_amd import attention as A
    model = A.SparseAttentionEncoder(50, embed, embed // 32, 0.8, 96, 256, 64, vec_length=8, layers=len(mlps), seed=3)
    for b, n in zip(model.blocks, mlps):
        b.linear1, b.linear2 = torch.nn.Linear(embed, n), torch.nn.Linear(n, embed)
    model = model.cuda().half().eval()
    tokens = torch.randint(0, 50, (3, 96), device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    masks, folds, plain = [], [], A.block_dense
    for b in model.blocks:
        mask = torch.zeros(12, 8, 96, dtype=torch.bool, device="cuda")
        mask[torch.repeat_interleave(torch.arange(12, device="cuda"), b.row_offsets.diff().long()), :, b.column_indices.long()] = True
        masks.append(mask.view(96, 96))
    A.block_dense = lambda *args, **kw: (folds.append(kw.get("folded") is not None), plain(*args, **kw))[1]
    try:
        with torch.no_grad():
            got = model(tokens).double()
    finally:
        A.block_dense = plain
    assert folds == [False] + [n > embed for n in mlps]
    with torch.no_grad():
        want = copy.deepcopy(model).double()(tokens, masks)
    assert (got - want).norm() / want.norm() <= 4 * 2.0 ** -11 / 3 ** 0.5


@pytest.mark.parametrize("mlp", [256, 512])
def test_encoder_refuses_tokens_outside_the_table(built_library, monkeypatch, mlp):
    """As torch's lookup does, by an assertion on the device (looked at here, not made), with and without layers to fold; sequences beside are
    what they are without such a token."""
    from sspmm_amd.attention import SparseAttentionEncoder
    model = SparseAttentionEncoder(50, 256, 8, 0.8, 96, mlp, 64, vec_length=8, layers=2, seed=2).cuda().half().eval()
    tokens = torch.randint(0, 50, (3, 96), device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    seen = []
    monkeypatch.setattr(torch, "_assert_async", lambda ok, *message: seen.append(ok))
    with torch.no_grad():
        want = model(tokens)
        for bad in (50, -1, 1 << 40):
            tokens[1, 17] = bad
            got = model(tokens)
            assert got[:, 1].isnan().any() and torch.equal(got[:, ::2], want[:, ::2])
        tokens[1, 17] = 49
        got = model(tokens)
        assert not got.isnan().any()
    assert [ok.item() for ok in seen] == [1, 0, 0, 0, 1]


@pytest.mark.parametrize("where,name", [("linear1", "weight"), ("linear2", "bias"), ("out_proj", "weight"), ("in_proj", "bias"), ("layer_norm1", "weight"),
                                        ("layer_norm2", "bias"), ("encoder", "weight"), ("linear", "weight"), ("layer_norm", "bias"),
                                        ("block", "linear1"), ("block", "layer_norm2"), ("block", "column_indices"), ("model", "encoder")])
def test_encoder_takes_an_instances_own_attribute_first(built_library, where, name):
    """What a program has put into a module's __dict__ comes before the parameter, buffer or module of that name, as everywhere in torch."""
    import copy
    from sspmm_amd.attention import SparseAttentionEncoder
    model = SparseAttentionEncoder(50, 128, 4, 0.8, 96, 256, 64, vec_length=8, layers=2, seed=2).cuda().half().eval()
    tokens = torch.randint(0, 50, (2, 96), device="cuda", generator=torch.Generator("cuda").manual_seed(1))

    def owner(m):
        return {"block": m.blocks[1], "model": m}.get(where) or getattr(m if hasattr(m, where) else m.blocks[1], where)

    with torch.no_grad():
        want, old = copy.deepcopy(model), getattr(owner(model), name)
        if isinstance(old, torch.nn.Module):
            new = copy.deepcopy(old)
            new.weight.copy_(torch.randn_like(new.weight) * 0.1)
        else:
            new = old.flip(0) if name == "column_indices" else torch.randn_like(old) * 0.1
        setattr(owner(want), name, torch.nn.Parameter(new) if isinstance(old, torch.nn.Parameter) else new)
        owner(model).__dict__[name] = new
        assert getattr(owner(model), name) is new
        assert torch.equal(model(tokens), want(tokens))
        del owner(model).__dict__[name]
        assert not torch.equal(model(tokens), want(tokens))
