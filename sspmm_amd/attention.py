"""Python operator surface of the steps either side of `bspmm` in the reference's sparse
attention block, mirroring its torch extensions `sptrans.sddmm` and `sptrans.softmax`
(reference end2end/sspmm_e2e/src/cuda/sddmm.cpp:11-46, softmax.cpp:11-43): same names, same
argument order, same shape inference (sddmm_kernel.cu:1169-1186 and 1236-1258,
softmax_kernel.cu:208-216 and 256-266), and the block that chains them
(end2end/sspmm_e2e/spattention.py:167-179).
"""
import ctypes

import torch

from . import _lib
from .spmm import _check_inputs, _ptr, bspmm


def _check_pattern(row_indices, row_offsets, column_indices, vec_length):
    if vec_length not in (8, 16):
        raise ValueError("vec_length must be 8 or 16, got %r" % (vec_length,))
    for name, t in (("row_offsets", row_offsets), ("column_indices", column_indices), ("row_indices", row_indices)):
        if t is None:
            continue
        if t.dtype != torch.int32 or not t.is_cuda or not t.is_contiguous():
            raise TypeError("%s must be a contiguous int32 GPU tensor" % name)


def _check_half(name, t):
    if t.dtype != torch.float16 or not t.is_cuda or not t.is_contiguous():
        raise TypeError("%s must be a contiguous float16 GPU tensor" % name)


def bsddmm(row_indices, row_offsets, column_indices, lhs_matrix, rhs_matrix, vec_length):
    """out[b, j*V + v] = lhs[b, i*V + v, :] . rhs[b, col_j, :]: lhs [batch, M, F], rhs [batch, n, F] ->
    fp16 [batch, nvec*V] (reference batched_sddmm_cuda)."""
    _check_pattern(row_indices, row_offsets, column_indices, vec_length)
    _check_half("lhs_matrix", lhs_matrix)
    _check_half("rhs_matrix", rhs_matrix)
    m, k, n = lhs_matrix.size(-2), lhs_matrix.size(-1), rhs_matrix.size(-2)
    if rhs_matrix.size(-1) != k:
        raise ValueError("lhs_matrix and rhs_matrix must have the same feature length")
    batch = lhs_matrix.numel() // (m * k) if m * k > 0 else 1
    m_vec = row_offsets.numel() - 1
    if m != m_vec * vec_length:
        raise ValueError("lhs_matrix must have m_vec * vec_length = %d rows, got %d" % (m_vec * vec_length, m))
    nvec = column_indices.numel()
    out = torch.empty((batch, nvec * vec_length), dtype=torch.float16, device=lhs_matrix.device)
    rc = _lib.call(_lib.lib().sspmm_sddmm_batched_f16, lhs_matrix.device, batch, m_vec, vec_length, k, n, _ptr(row_indices),
                   row_offsets.data_ptr(), column_indices.data_ptr(), lhs_matrix.data_ptr(), m * k, rhs_matrix.data_ptr(), n * k,
                   out.data_ptr(), nvec * vec_length)
    _lib.check(rc, "sspmm_sddmm")
    return out


def sddmm(row_indices, row_offsets, column_indices, lhs_matrix, rhs_matrix, vec_length):
    """lhs [M, F], rhs [n, F] -> fp16 [nvec*V] (reference sddmm_cuda)."""
    if lhs_matrix.dim() != 2 or rhs_matrix.dim() != 2:
        raise ValueError("lhs_matrix and rhs_matrix must be 2-D")
    return bsddmm(row_indices, row_offsets, column_indices, lhs_matrix, rhs_matrix, vec_length).view(-1)


def bcsr_softmax(row_indices, row_offsets, values, scaler, vec_length, batch_size):
    """Row softmax over the stored entries, values [batch, nvec*V] -> fp16 of the same shape
    (reference batched_csr_softmax_cuda)."""
    _check_pattern(row_indices, row_offsets, None, vec_length)
    _check_half("values", values)
    m_vec = row_offsets.numel() - 1
    stride = values.numel() // batch_size if batch_size > 0 else 0
    out = torch.empty_like(values)
    rc = _lib.call(_lib.lib().sspmm_softmax_batched_f16, values.device, batch_size, m_vec, vec_length, _ptr(row_indices),
                   row_offsets.data_ptr(), values.data_ptr(), float(scaler), out.data_ptr(), stride)
    _lib.check(rc, "sspmm_softmax")
    return out


def csr_softmax(row_indices, row_offsets, values, scaler, vec_length):
    """values [nvec*V] -> fp16 [nvec*V] (reference csr_softmax_cuda)."""
    return bcsr_softmax(row_indices, row_offsets, values, scaler, vec_length, 1)


FUSED_HEAD_WIDTHS = (32, 64, 128)


def fused_sparse_attention(row_indices, row_offsets, column_indices, q, k, v, scaling, vec_length):
    """The block's three steps in one launch (heads of 32, 64 or 128 features): scores and probabilities never leave the
    chip.  Same arguments and result shape as `sparse_attention`; differs from the three-step chain by fp16 rounding
    of intermediate values only (the chain rounds the scores and the normalised probabilities to fp16, this rounds
    the probabilities before the division by their sum)."""
    _check_pattern(row_indices, row_offsets, column_indices, vec_length)
    for name, t in (("q", q), ("k", k), ("v", v)):
        _check_half(name, t)
    m, d, n = q.size(-2), q.size(-1), k.size(-2)
    if d not in FUSED_HEAD_WIDTHS or k.size(-1) != d or v.size(-1) != d:
        raise ValueError("fused_sparse_attention takes heads of 32, 64 or 128 features, the same for q, k and v")
    if v.size(-2) != n:
        raise ValueError("k and v must have the same number of rows")
    m_vec = row_offsets.numel() - 1
    if m != m_vec * vec_length:
        raise ValueError("q must have m_vec * vec_length = %d rows, got %d" % (m_vec * vec_length, m))
    batch = q.numel() // (m * d) if m > 0 else 1
    if k.numel() != batch * n * d or v.numel() != batch * n * d:
        raise ValueError("q, k and v must have the same batch size")
    out = torch.empty(q.shape, dtype=torch.float16, device=q.device)
    rc = _lib.call(_lib.lib().sspmm_sparse_attention_f16, q.device, batch, m_vec, vec_length, d, n, _ptr(row_indices),
                   row_offsets.data_ptr(), column_indices.data_ptr(), q.data_ptr(), m * d, k.data_ptr(), n * d, v.data_ptr(), n * d,
                   float(scaling), out.data_ptr(), m * d)
    _lib.check(rc, "sspmm_sparse_attention")
    return out


def packed_attention_fits(seq, bsz, three_e):
    """Whether `sparse_attention_packed` takes a projection of this shape: the rows of one (batch element, head) pair,
    which lie `bsz * three_e` elements apart, must span less than 2 GiB (one 32-bit buffer descriptor)."""
    return (seq - 1) * bsz * three_e * 2 < (1 << 31) - 256 and bsz * three_e < (1 << 23) and seq < (1 << 24)


def sparse_attention_packed(row_indices, row_offsets, column_indices, qkv, num_heads, scaling, vec_length):
    """Multi-head attention on a vector-sparse mask straight from a fused projection: qkv [seq, batch, 3 * embed] (q,
    k and v side by side in the last dimension, heads of 32, 64 or 128 features side by side in each) -> [seq, batch, embed],
    in one launch and without the copies into [batch * heads, seq, 64] and back that the reference's module makes
    around its three operators (spattention.py:151-157 and 181-184)."""
    _check_pattern(row_indices, row_offsets, column_indices, vec_length)
    _check_half("qkv", qkv)
    if qkv.dim() != 3 or qkv.size(-1) % (3 * num_heads) or qkv.size(-1) // (3 * num_heads) not in FUSED_HEAD_WIDTHS:
        raise ValueError("qkv must be [seq, batch, 3 * num_heads * d] with d = 32, 64 or 128")
    seq, bsz, three_e = qkv.shape
    e = three_e // 3
    d = e // num_heads
    m_vec = row_offsets.numel() - 1
    if seq != m_vec * vec_length:
        raise ValueError("qkv must have m_vec * vec_length = %d rows, got %d" % (m_vec * vec_length, seq))
    out = torch.empty((seq, bsz, e), dtype=torch.float16, device=qkv.device)
    base, ld = qkv.data_ptr(), bsz * three_e
    rc = _lib.call(_lib.lib().sspmm_sparse_attention_heads_f16, qkv.device, bsz, num_heads, m_vec, vec_length, d, seq,
                   _ptr(row_indices), row_offsets.data_ptr(), column_indices.data_ptr(),
                   base, three_e, d, ld, base + 2 * e, three_e, d, ld, base + 4 * e, three_e, d, ld, float(scaling),
                   out.data_ptr(), e, d, bsz * e)
    _lib.check(rc, "sspmm_sparse_attention_heads")
    return out


def sparse_attention_split(row_indices, row_offsets, column_indices, qkv, scaling, vec_length):
    """The same from a projection split into heads: qkv [3, batch, heads, seq, d] -> [seq, batch, heads * d].  A head's
    rows then lie side by side instead of 3 * batch * embed elements apart: 4096 keys, 32 pairs of element and head, 32 / 64 / 128 features, V = 8
    59.2 -> 54.2, 76.4 -> 75.7, 152 -> 147 us, V = 16 32.7 -> 29.7, 44.1 -> 43.3, 84.4 -> 82.7, 4 pairs 10.3 -> 8.9, 12.3 -> 12.2, 21.5 -> 21.4."""
    _check_pattern(row_indices, row_offsets, column_indices, vec_length)
    _check_half("qkv", qkv)
    if qkv.dim() != 5 or qkv.size(0) != 3 or qkv.size(-1) not in FUSED_HEAD_WIDTHS:
        raise ValueError("qkv must be [3, batch, heads, seq, d] with d = 32, 64 or 128")
    _, bsz, heads, seq, d = qkv.shape
    m_vec = row_offsets.numel() - 1
    if seq != m_vec * vec_length:
        raise ValueError("qkv must have m_vec * vec_length = %d rows, got %d" % (m_vec * vec_length, seq))
    out = torch.empty((seq, bsz, heads * d), dtype=torch.float16, device=qkv.device)
    base, head, elem = qkv.data_ptr(), seq * d, heads * seq * d
    part = 2 * bsz * elem
    rc = _lib.call(_lib.lib().sspmm_sparse_attention_heads_f16, qkv.device, bsz, heads, m_vec, vec_length, d, seq,
                   _ptr(row_indices), row_offsets.data_ptr(), column_indices.data_ptr(),
                   base, elem, head, d, base + part, elem, head, d, base + 2 * part, elem, head, d, float(scaling),
                   out.data_ptr(), heads * d, d, bsz * heads * d)
    _lib.check(rc, "sspmm_sparse_attention_heads")
    return out


def sparse_attention(row_indices, row_offsets, column_indices, q, k, v, scaling, vec_length, fused=None):
    """softmax(mask(q k^T) * scaling) v on a vector-sparse mask shared by the batch:
    q [batch, tgt, d], k [batch, src, d], v [batch, src, d_v] -> fp16 [batch, tgt, d_v]; the three
    steps of the reference's block (spattention.py:167-179).  fused: None = one launch where the shapes allow it
    (d = d_v = 32, 64 or 128), False = always the three operators, True = one launch or an error."""
    if fused is None:
        fused = q.size(-1) in FUSED_HEAD_WIDTHS and v.size(-1) == q.size(-1) and row_offsets.numel() > 1 and q.numel() > 0
    if fused:
        return fused_sparse_attention(row_indices, row_offsets, column_indices, q, k, v, scaling, vec_length)
    w = bsddmm(row_indices, row_offsets, column_indices, q, k, vec_length)
    w = bcsr_softmax(row_indices, row_offsets, w, scaling, vec_length, w.size(0))
    _check_inputs(row_indices, row_offsets, column_indices, w, v, vec_length)
    return bspmm(row_indices, row_offsets, column_indices, w, v, vec_length)


def static_random_mask(m_vec, n, sparsity, seed=0):
    """A vector-sparse attention mask as the reference's end-to-end model draws it (verify/static_mask.py:7-27:
    scipy.sparse.random of m_vec x n with density 1 - sparsity, i.e. round(density * m_vec * n) positions drawn uniformly
    without replacement, CSR with ascending columns; row_indices = vector-rows by ascending length).  Seeded numpy
    in place of scipy's global state.  Returns (column_indices, row_offsets, row_indices) as int32 numpy arrays."""
    import numpy as np
    rng = np.random.default_rng(seed)
    k = int(round((1.0 - sparsity) * m_vec * n))
    flat = np.sort(rng.choice(m_vec * n, size=k, replace=False))
    rows, cols = flat // n, flat % n
    row_offsets = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=m_vec))]).astype(np.int32)
    row_indices = np.argsort(np.diff(row_offsets), kind="stable").astype(np.int32)
    return cols.astype(np.int32), row_offsets, row_indices


ROW_WIDTHS = (64, 128, 256, 512, 1024, 2048)


def add_layernorm_rows(x, a, ln, keep_sum=False):
    """(x + a or None, LayerNorm(x + a)) on token-major activations [seq, batch, embed] fp16 in one launch; a may be
    None.  x may be a view with strides of its own in the first two dimensions, a is dense; the results are dense.  The
    sum is only returned with keep_sum."""
    outer, inner, E = x.shape
    out = torch.empty((outer, inner, E), dtype=torch.float16, device=x.device)
    total = torch.empty_like(out) if keep_sum else None
    stride = x.stride()
    rc = _lib.call(_lib.lib().sspmm_add_layernorm_rows_f16, x.device, outer, inner, E, x.data_ptr(), stride[0], stride[1], _ptr(a),
                   _ptr(ln.weight), _ptr(ln.bias), float(ln.eps), _ptr(total), out.data_ptr())
    _lib.check(rc, "sspmm_add_layernorm_rows_f16")
    return total, out


BLOCK_WIDTHS = (128, 256, 512)


def pack_weights(linears, rows_per_wave):
    """The weights of torch.nn.Linear modules in the order in which block_dense's kernel loads them, each a tensor of its
    own out of one allocation, by one launch; rows_per_wave[i] = embed / 4 for out_proj and linear2, 64 for the others."""
    n = len(linears)
    weights = [_weights(m)[0] for m in linears]
    shapes = [w.shape for w in weights]
    sizes = [r * c for r, c in shapes]
    device = weights[0].device
    packed = torch.empty(sum(sizes), dtype=torch.float16, device=device)
    ints = ctypes.c_int32 * n
    rc = _lib.call(_lib.lib().sspmm_block_pack_f16, device, n, (ctypes.c_void_p * n)(*[w.data_ptr() for w in weights]),
                   ints(*[r for r, _ in shapes]), ints(*[c for _, c in shapes]), ints(*rows_per_wave), packed.data_ptr())
    _lib.check(rc, "sspmm_block_pack_f16")
    return packed.split(sizes)


class FoldedLayers(tuple):
    """(matrix, affine) of two linear layers with nothing between them, and `rest`, what the matrix's rounding to fp16 left."""


def fold_blocks(blocks, linears, rows_per_wave, tokens_ok=None):
    """pack_weights(linears, rows_per_wave), and in the same launch linear1 and linear2 of every block as the one linear map they
    are, there being nothing between them: (packed, [FoldedLayers per block]) for block_dense's `folded`.
    tokens_ok: an int32 that becomes one, for block_dense behind it."""
    n, f, E = len(linears), len(blocks), linears[0].in_features
    weights = [_weights(m)[0] for m in linears]
    shapes = [w.shape for w in weights]
    sizes = [r * c for r, c in shapes]
    device = weights[0].device
    pairs = [_parts(b, "linear1", "linear2") for b in blocks]
    up, down = [_weights(a) for a, _ in pairs], [_weights(b) for _, b in pairs]
    packed = torch.empty(sum(sizes) + 2 * f * E * E, dtype=torch.float16, device=device)
    affine = torch.empty((f, 2 * E), dtype=torch.float32, device=device)
    ints, ptrs, some = ctypes.c_int32 * n, ctypes.c_void_p * n, ctypes.c_void_p * f
    at = packed.data_ptr() + 2 * sum(sizes)
    rc = _lib.call(_lib.lib().sspmm_block_fold_split_f16, device, n, ptrs(*[w.data_ptr() for w in weights]), ints(*[r for r, _ in shapes]),
                   ints(*[c for _, c in shapes]), ints(*rows_per_wave), packed.data_ptr(), f, E, (ctypes.c_int32 * f)(*[a.out_features for a, _ in pairs]),
                   some(*[w.data_ptr() for w, _ in up]), some(*[_ptr(b) for _, b in up]), some(*[w.data_ptr() for w, _ in down]),
                   some(*[_ptr(b) for _, b in down]), at, at + 2 * f * E * E, affine.data_ptr(), _ptr(tokens_ok))
    _lib.check(rc, "sspmm_block_fold_split_f16")
    parts = packed.split(sizes + 2 * f * [E * E])
    folded = [FoldedLayers(pair) for pair in zip(parts[n:], affine)]
    for pair, rest in zip(folded, parts[n + f:]):
        pair.rest = rest
    return parts[:n], folded


def block_dense(x, attn, block, norm, tail=None, keep_x=False, packed=None, head_dim=0, pos=None, scale=1.0, folded=None, table=None, tokens_ok=None):
    """(x', out): everything between the attention of `block` and the next one's in one launch, on token-major activations
    [seq, batch, embed] fp16:
        s = out_proj(attn) + x, x' = linear2(linear1(layer_norm2(s))) + x, h = norm(x'), out = tail(h) or h itself.
    attn None: x' = x and `block` is not looked at.  x may be a view with strides of its own in the first two dimensions,
    attn is dense, and so are the results.  x' is only returned with keep_x.  packed: pack_weights of out_proj, linear1 and
    linear2 (where there is attn) and tail (where there is one), in this order.  head_dim: out as
    [tail.out_features / embed, batch, embed / head_dim, seq, head_dim], for sparse_attention_split.  pos
    [seq, embed]: x is an embedding, and (x * scale) + pos stands in its place, each rounded to fp16.  folded: linear1 and linear2 as
    fold_blocks leaves them (with attn, without pos), packed then that of out_proj and tail.  table (without attn, with pos): x are
    tokens [batch, seq], and the embedding is read from the table's rows; a token that is none of them makes a row of NaN, and 0 of tokens_ok."""
    outer, inner, E = x.shape if table is None else (x.size(1), x.size(0), table.size(1))
    n_out = 0 if tail is None else tail.out_features
    shape = (n_out // E, inner, E // head_dim, outer, head_dim) if head_dim else (outer, inner, n_out or E)
    out = torch.empty(shape, dtype=torch.float16, device=x.device)
    kept = torch.empty((outer, inner, E), dtype=torch.float16, device=x.device) if keep_x else None
    stride = x.stride()
    if table is not None:
        gamma_n, beta_n = _weights(norm)
        rc = _lib.call(_lib.lib().sspmm_block_embed_checked_f16, x.device, outer, inner, E, x.data_ptr(), x.element_size(), stride[1], stride[0], table.data_ptr(),
                       table.size(0), pos.data_ptr(), float(scale), _ptr(gamma_n), _ptr(beta_n), float(norm.eps), n_out, head_dim, packed[-1].data_ptr(),
                       _ptr(_weights(tail)[1]), _ptr(kept), out.data_ptr(), _ptr(tokens_ok))
        _lib.check(rc, "sspmm_block_embed_checked_f16")
        return kept, out
    if packed is None:
        own = [] if attn is None else [block.out_proj, block.linear1, block.linear2]
        if own or tail is not None:
            packed = pack_weights(own + ([] if tail is None else [tail]), [E // 4, 64, E // 4][:len(own)] + [64] * (tail is not None))
    last = (None, None) if tail is None else (packed[-1].data_ptr(), _ptr(_weights(tail)[1]))
    gamma_n, beta_n = _weights(norm)
    if folded is not None:
        proj, ln = _parts(block, "out_proj", "layer_norm2")
        gamma, beta = _weights(ln)
        rc = _lib.call(_lib.lib().sspmm_block_dense_split_f16, x.device, outer, inner, E, x.data_ptr(), stride[0], stride[1], _ptr(attn), packed[0].data_ptr(),
                       _ptr(_weights(proj)[1]), _ptr(gamma), _ptr(beta), float(ln.eps), folded[0].data_ptr(), folded.rest.data_ptr(), folded[1].data_ptr(),
                       _ptr(gamma_n), _ptr(beta_n), float(norm.eps), n_out, head_dim, *last, _ptr(kept), out.data_ptr())
        _lib.check(rc, "sspmm_block_dense_split_f16")
        return kept, out
    if attn is None:
        own = (None, None, None, None, 0.0, 0, None, None, None, None)
    else:
        proj, up, down, ln = _parts(block, "out_proj", "linear1", "linear2", "layer_norm2")
        gamma, beta = _weights(ln)
        own = (packed[0].data_ptr(), _ptr(_weights(proj)[1]), _ptr(gamma), _ptr(beta), float(ln.eps), up.out_features,
               packed[1].data_ptr(), _ptr(_weights(up)[1]), packed[2].data_ptr(), _ptr(_weights(down)[1]))
    rc = _lib.call(_lib.lib().sspmm_block_dense_f16, x.device, outer, inner, E, x.data_ptr(), stride[0], stride[1], _ptr(pos), float(scale),
                   _ptr(attn), *own, _ptr(gamma_n), _ptr(beta_n), float(norm.eps), n_out, head_dim, *last, _ptr(kept), out.data_ptr())
    _lib.check(rc, "sspmm_block_dense_f16")
    return kept, out


def _rows_operand(t):
    return (type(t) is torch.Tensor and t.is_cuda and t.dtype == torch.float16 and t.dim() == 3 and t.numel() > 0 and t.stride(2) == 1 and
            t.stride(0) % 8 == 0 and t.stride(1) % 8 == 0 and t.data_ptr() % 16 == 0)


def _plain_module(m, kind):
    """Whether calling m does nothing but kind's own forward: no hooks, no subclass (a parametrization is one), no
    forward of the instance's own."""
    return (type(m) is kind and not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks) and
            "forward" not in m.__dict__)


# A module's parameters, buffers and modules by way of its __getattr__ are 0.3 us each, and a forward pass of four blocks asks for some
# two hundred of them: 260 us of the host a pass, where the device takes 230 for two sequences of 4096 tokens.  These look where it
# would, after the instance's own attributes, which it is not asked for: 192 us, and the pass 238 -> 219.
def _weights(m):
    """(m.weight, m.bias)"""
    own = m.__dict__
    if "weight" in own or "bias" in own:
        return m.weight, m.bias
    own = own["_parameters"]
    try:
        return own["weight"], own["bias"]
    except KeyError:
        return m.weight, m.bias


def _parts(m, *names):
    """m's modules of these names"""
    own = m.__dict__
    modules = own["_modules"]
    try:
        return [own[n] if n in own else modules[n] for n in names]
    except KeyError:
        return [getattr(m, n) for n in names]


def _pattern(block):
    own = block.__dict__
    if "row_offsets" in own or "column_indices" in own:
        return block.row_offsets, block.column_indices
    own = own["_buffers"]
    try:
        return own["row_offsets"], own["column_indices"]
    except KeyError:
        return block.row_offsets, block.column_indices


_TENSORS = (torch.Tensor, torch.nn.Parameter)


def _operand(t, device, shape):
    """Whether a kernel on GPU `device` may read t, of this shape, as it lies."""
    return (type(t) in _TENSORS and t.dtype is torch.float16 and t.get_device() == device and t.shape == shape and t.is_contiguous() and
            t.data_ptr() % 16 == 0)


def _rows_norm_applies(ln, x):
    """Whether add_layernorm_rows may stand in for ln on activations like x."""
    if not _plain_module(ln, torch.nn.LayerNorm):
        return False
    E, device, (w, b) = x.size(-1), x.get_device(), _weights(ln)
    return (E in ROW_WIDTHS and ln.normalized_shape == (E,) and _operand(w, device, (E,)) and (b is None or _operand(b, device, (E,))))


BLOCK_FEATURES = 1 << 20  # hidden or output features that block_dense takes at most
# However few tokens there are, a wide hidden layer costs the launch that multiplies the two linear layers its W1, which a CU streams
# whole at 64 bytes a cycle for every sixteen rows (256 features: 8192 hidden ones 33 us more than 4096, whatever the number of
# blocks), where library products spread the weights over the chip.  Up to this many weights in a matrix the two launches a block are ahead all
# the same, by what the modules cost the host.  Forward pass, 64 / 512 / 4096 tokens, in these launches called one after the
# other - as modules with the norms fused called / replayed from a graph, us: one block 256 x 4096 79 / 80 / 81 - 220 / 230 / 229, 45 / 52 / 96,
# 256 x 8192 87 / 88 / 104 - 223 / 230 / 230, 47 / 58 / 124, four blocks of the latter 181 / 185 / 197 - 626 / 653 / 654, 164 / 186 / 454.  Twice as
# many, 256 x 16384: 152 / 153 / 168 - 229 / 230 / 231, 58 / 70 / 176, and 512 x 8192 172 / 171 / 191 - 229 / 229 / 232, 54 / 72 / 174: called they are
# ahead there too, replayed they would be 2.5 times as slow, so the line stays.  Beyond 4096 tokens these launches are ahead whatever the
# sizes: 6144 tokens 512 x 16384 341 - 392, 390, 512 x 32768 590 - 668, 664, 256 x 65536 584 - 748, 750.  A head is level with the library's
# product at best when it is
# that large and behind beyond, with many tokens too: outputs in the launch / as a module, us of the device, 512 x 4096, 64 and
# 32768 tokens 90 / 54 and 351 / 374, 512 x 8192 134 / 54 and 573 / 559, 256 x 65536 413 / 35 at 64 tokens and 814 / 487 at 8192.
BLOCK_WEIGHTS = 1 << 21


def _plain_linear(m, x, in_features, out_features, multiple):
    """Whether m is a torch.nn.Linear of these sizes (out_features None: any multiple of `multiple` up to BLOCK_FEATURES)
    whose weights a kernel may read as they lie, for activations like x."""
    if not _plain_module(m, torch.nn.Linear):
        return False
    outs, device, (w, b) = m.out_features, x.get_device(), _weights(m)
    return (m.in_features == in_features and outs % multiple == 0 and outs <= BLOCK_FEATURES and (out_features is None or outs == out_features) and
            _operand(w, device, (outs, in_features)) and (b is None or _operand(b, device, (outs,))))


# (bound once: _eager is asked by calls of a few microseconds)
_nn_module, _forward_ad = torch.nn.modules.module, torch.autograd.forward_ad
_tracing, _compiling, _autocast = torch.jit.is_tracing, torch.compiler.is_compiling, torch.is_autocast_enabled
_dispatch_modes, _function_modes = torch._C._len_torch_dispatch_stack, torch._C._len_torch_function_stack
_transforms = torch._C._functorch.maybe_current_level


def _eager():
    """Nothing watches the operators: no forward-mode gradients, no tracing or compiling, no autocast, no modes or module hooks
    that want to see every one of them."""
    return not (_tracing() or _compiling() or _autocast("cuda") or _forward_ad._current_level >= 0 or
                _dispatch_modes() or _function_modes() or _transforms() is not None or
                _nn_module._global_forward_hooks or _nn_module._global_forward_pre_hooks or
                _nn_module._global_backward_hooks or _nn_module._global_backward_pre_hooks)


def _eager_inference():
    """Nothing but the values is wanted: as _eager, and no gradients."""
    return not torch.is_grad_enabled() and _eager()


class SparseAttentionBlock(torch.nn.Module):
    """One block of the reference's end-to-end model (SparseTransformerBlock, end2end/sspmm_e2e/end_to_end.py:45-78):
    LayerNorm -> multi-head attention on a static vector-sparse mask (bsddmm -> bcsr_softmax -> bspmm,
    spattention.py:151-186) -> + x -> LayerNorm -> linear1 -> linear2 -> + x, on [seq, batch, embed] activations.
    The block's arithmetic follows the reference as written, including the second residual adding the block's input
    and the two linear layers without an activation between them."""

    def __init__(self, embed_dim, mlp_dim, num_heads, column_indices, row_offsets, row_indices, vec_length=8):
        super().__init__()
        if embed_dim % num_heads:
            raise ValueError("embed_dim must be a multiple of num_heads")
        self.embed_dim, self.num_heads, self.vec_length = embed_dim, num_heads, vec_length
        self.in_proj = torch.nn.Linear(embed_dim, 3 * embed_dim)
        self.out_proj = torch.nn.Linear(embed_dim, embed_dim)
        self.layer_norm1 = torch.nn.LayerNorm(embed_dim)
        self.layer_norm2 = torch.nn.LayerNorm(embed_dim)
        self.linear1 = torch.nn.Linear(embed_dim, mlp_dim)
        self.linear2 = torch.nn.Linear(mlp_dim, embed_dim)
        self.register_buffer("column_indices", column_indices)
        self.register_buffer("row_offsets", row_offsets)
        self.register_buffer("row_indices", row_indices)

    def attention(self, x, dense_mask=None):
        """x [seq, batch, embed] -> [seq, batch, embed].  With dense_mask (bool [seq, seq]) the three sparse steps
        are replaced by dense masked attention in fp32 (for checks)."""
        seq, bsz, E = x.shape
        h, d = self.num_heads, E // self.num_heads
        scaling = float(d) ** -0.5
        qkv = self.in_proj(x)
        if dense_mask is None and d in FUSED_HEAD_WIDTHS and qkv.dtype == torch.float16 and packed_attention_fits(seq, bsz, 3 * E):
            # the heads are read where the projection left them and written where the output projection wants them
            return self.out_proj(sparse_attention_packed(self.row_indices, self.row_offsets, self.column_indices,
                                                         qkv.contiguous(), h, scaling, self.vec_length))
        q, k, v = qkv.chunk(3, dim=-1)
        # [seq, batch * heads, d] -> [batch * heads, seq, d] (spattention.py:151-157)
        q, k, v = (t.contiguous().view(seq, bsz * h, d).transpose(0, 1).contiguous() for t in (q, k, v))
        if dense_mask is None:
            out = sparse_attention(self.row_indices, self.row_offsets, self.column_indices, q, k, v, scaling, self.vec_length)
        else:
            s = (q.float() @ k.float().transpose(1, 2)) * scaling
            s = s.masked_fill(~dense_mask, float("-inf"))
            out = (torch.softmax(s, dim=-1) @ v.float()).to(x.dtype)
        out = out.transpose(0, 1).contiguous().view(seq, bsz, E)
        return self.out_proj(out)

    def forward(self, x, dense_mask=None):
        out = self.attention(self.layer_norm1(x), dense_mask) + x
        out = self.linear2(self.linear1(self.layer_norm2(out)))
        return out + x


class SparseAttentionEncoder(torch.nn.Module):
    """The reference's end-to-end model (SparseTransformerEncoder, end_to_end.py:123-153): embedding * sqrt(embed),
    sinusoidal positions, four SparseAttentionBlocks each with a mask of its own, LayerNorm, linear head."""

    def __init__(self, vocab_size, embed_dim, num_heads, sparsity, seq_len, mlp_dim, num_class, vec_length=8, layers=4, seed=0):
        super().__init__()
        import math
        self.embed_dim = embed_dim
        self.encoder = torch.nn.Embedding(vocab_size, embed_dim)
        pe = torch.zeros(seq_len, embed_dim)
        pos = torch.arange(0, seq_len, dtype=torch.float).unsqueeze(1)
        div = torch.exp(torch.arange(0, embed_dim, 2).float() * (-math.log(10000.0) / embed_dim))
        pe[:, 0::2] = torch.sin(pos * div)
        pe[:, 1::2] = torch.cos(pos * div)
        self.register_buffer("pe", pe.unsqueeze(1))
        blocks = []
        for i in range(layers):
            cols, offs, rows = static_random_mask(seq_len // vec_length, seq_len, sparsity, seed=seed + i)
            blocks.append(SparseAttentionBlock(embed_dim, mlp_dim, num_heads, torch.from_numpy(cols), torch.from_numpy(offs),
                                               torch.from_numpy(rows), vec_length))
        self.blocks = torch.nn.ModuleList(blocks)
        self.layer_norm = torch.nn.LayerNorm(embed_dim)
        self.linear = torch.nn.Linear(embed_dim, num_class)

    def forward(self, tokens, dense_masks=None):
        """tokens: int [batch, seq] -> [seq, batch, num_class].  A token that is no row of the embedding's table is an error of the
        device, as in torch.nn.Embedding."""
        scale = self.embed_dim ** 0.5
        if dense_masks is None and _eager_inference():
            table = self._table(tokens)
            if table is not None and self._norms_apply(table) and self._blocks_apply(table, tokens.size(1), tokens.size(0)):
                pe = self._positions(tokens.size(1), table)
                if pe is not None:
                    return self._fused_blocks(tokens, pe, scale, table)
        out = self.encoder(tokens)
        if dense_masks is None and out.dim() == 3:
            x = out.transpose(0, 1)
            pe = self._positions(tokens.size(1), x)
            if pe is not None and self._fused_norms_apply(x) and self._blocks_apply(x, x.size(0), x.size(1)):
                return self._fused_blocks(x, pe, scale)
        out = out * scale
        out = out.transpose(0, 1) + self.pe[:tokens.size(1)].to(out.dtype)
        if dense_masks is None and self._fused_norms_apply(out):
            return self.linear(self._blocks_with_fused_norms(out))
        for i, blk in enumerate(self.blocks):
            out = blk(out, None if dense_masks is None else dense_masks[i])
        return self.linear(self.layer_norm(out))

    def _table(self, tokens):
        """The embedding's weight, where a kernel may look the tokens' rows up in it; None otherwise."""
        encoder, = _parts(self, "encoder")
        if not (type(tokens) is torch.Tensor and tokens.is_cuda and tokens.dim() == 2 and tokens.numel() > 0 and
                tokens.dtype in (torch.int64, torch.int32) and _plain_module(encoder, torch.nn.Embedding) and encoder.max_norm is None):
            return None
        weight = None if "weight" in encoder.__dict__ else encoder._parameters.get("weight")
        shape = (encoder.num_embeddings, self.embed_dim)
        return weight if weight is not None and shape[0] > 0 and _operand(weight, tokens.get_device(), shape) else None

    def _positions(self, seq, like):
        """The first rows of pe as a kernel reads them next to `like`, or None."""
        pe = self.pe[:seq].to(like.dtype)
        return pe if pe.shape == (seq, 1, like.size(-1)) and _rows_operand(pe) and pe.is_contiguous() and pe.device == like.device else None

    def _norms_apply(self, x):
        return (len(self.blocks) > 0 and _rows_norm_applies(_parts(self, "layer_norm")[0], x) and
                all(_plain_module(b, SparseAttentionBlock) and "attention" not in b.__dict__ and
                    all([_rows_norm_applies(n, x) for n in _parts(b, "layer_norm1", "layer_norm2")]) for b in self.blocks))

    def _fused_norms_apply(self, x):
        return _rows_operand(x) and _eager_inference() and self._norms_apply(x)

    def _blocks_with_fused_norms(self, x):
        """The blocks and the final LayerNorm with every residual sum in the launch of the LayerNorm behind it, also
        across blocks: a sum that only a LayerNorm reads is never written."""
        def add_norm(x, a, ln, keep_sum=False):
            if _rows_operand(x) and _rows_operand(a) and a.is_contiguous() and a.shape == x.shape and a.device == x.device:
                return add_layernorm_rows(x, a, ln, keep_sum)
            s = a + x  # (a projection that has been replaced by one of another type)
            return s, ln(s)

        _, h = add_layernorm_rows(x, None, self.blocks[0].layer_norm1)
        for i, blk in enumerate(self.blocks):
            last = i + 1 == len(self.blocks)
            _, h = add_norm(x, blk.attention(h), blk.layer_norm2)
            y = blk.linear2(blk.linear1(h))
            x, h = add_norm(x, y, self.layer_norm if last else self.blocks[i + 1].layer_norm1, keep_sum=not last)
        return h

    def _blocks_apply(self, x, seq, bsz):
        """(where the fused norms do) heads that one launch of attention takes, and products that block_dense does and is
        ahead with (see BLOCK_WEIGHTS).  x: an operand on the device, of the blocks' width."""
        E = x.size(-1)
        if not (E in BLOCK_WIDTHS and packed_attention_fits(seq, bsz, 3 * E)):
            return False
        for b in self.blocks:
            into, out, up, down = _parts(b, "in_proj", "out_proj", "linear1", "linear2")
            if not (b.embed_dim == E and E % b.num_heads == 0 and E // b.num_heads in FUSED_HEAD_WIDTHS and
                    _plain_linear(into, x, E, 3 * E, 64) and _plain_linear(out, x, E, E, 64) and
                    _plain_linear(up, x, E, None, 256) and _plain_linear(down, x, up.out_features, E, 64) and
                    (E * up.out_features <= BLOCK_WEIGHTS or seq * bsz > 4096)):
                return False
        return True

    def _fused_blocks(self, x, pe, scale, table=None):
        """(x * scale) + pe through the blocks and the head (x: an embedding, or with table the tokens to look up in it).  Two launches per
        block: its attention, and all that follows up to the next block's projection (or the head)."""
        like = x if table is None else table
        E, blocks = like.size(-1), list(self.blocks)
        final, linear = _parts(self, "layer_norm", "linear")
        head = _plain_linear(linear, like, E, None, 64) and E * linear.out_features <= BLOCK_WEIGHTS
        into, norms = [_parts(b, "in_proj")[0] for b in blocks], [_parts(b, "layer_norm1")[0] for b in blocks]
        # (the two linear layers as one, in two matrices of E x E, where those are fewer weights than the two layers'.  Four blocks replayed, folded /
        # two layers, us: 512 features, 256 hidden ones 169 / 148 at 512 tokens, 567 / 539 at 16384, 512 hidden 172 / 166, 569 / 570, 768 hidden
        # 176 / 185, 572 / 600; 256 features, 256 hidden 74 / 72, 336 / 337, 512 hidden 76 / 83, 337 / 350)
        fold = [_parts(b, "linear1")[0].out_features > E for b in blocks]
        linears, rows, ends = [into[0]], [64], [1]
        for i, blk in enumerate(blocks):
            tail = [into[i + 1]] if i + 1 < len(blocks) else [linear] * head
            linears += (_parts(blk, "out_proj") if fold[i] else _parts(blk, "out_proj", "linear1", "linear2")) + tail
            rows += ([E // 4] if fold[i] else [E // 4, 64, E // 4]) + [64] * len(tail)
            ends.append(len(linears))
        ok = None if table is None else torch.empty(1, dtype=torch.int32, device=table.device)
        packed, pairs = fold_blocks([b for b, f in zip(blocks, fold) if f], linears, rows, ok)
        pairs = iter(pairs)
        folded = [next(pairs) if f else None for f in fold]

        def attention(blk, qkv):
            # (in the pattern's own order: the longest rows last, which row_indices asks for, cost 1 to 4 %)
            offsets, columns = _pattern(blk)
            return sparse_attention_split(None, offsets, columns, qkv, float(qkv.size(-1)) ** -0.5, blk.vec_length)

        x, qkv = block_dense(x, None, None, norms[0], into[0], True, packed[:1], E // blocks[0].num_heads, pe, scale,
                             table=table, tokens_ok=ok)
        if ok is not None:
            # (as torch's own lookup does; 1.7 us of the device and some 6 of the host, where the lookup as a launch of its own is 14 and more)
            torch._assert_async(ok, "a token is no row of the embedding's table")
        for i, blk in enumerate(blocks[:-1]):
            x, qkv = block_dense(x, attention(blk, qkv), blk, norms[i + 1], into[i + 1], True, packed[ends[i]:ends[i + 1]],
                                 E // blocks[i + 1].num_heads, folded=folded[i])
        out = block_dense(x, attention(blocks[-1], qkv), blocks[-1], final, linear if head else None,
                          packed=packed[ends[-2]:], folded=folded[-1])[1]
        return out if head else linear(out)
