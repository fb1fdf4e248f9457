"""The C ABI library loads without a GPU, exports every symbol include/sspmm.h declares, and
rejects bad arguments before touching the device."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "sspmm.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b((?:sspmm|svc)_[a-z0-9_]+)\s*\(", text)))


def test_every_declared_symbol_is_exported_and_bound(built_library):
    from sspmm_amd import _lib
    L = ctypes.CDLL(built_library)
    names = _declared_symbols()
    assert len(names) >= 10
    for n in names:
        assert hasattr(L, n), "library does not export %s" % n
        assert n in _lib.SIGNATURES, "ctypes binding misses %s" % n
    assert sorted(_lib.SIGNATURES) == names


def test_argument_errors_without_device_work(built_library):
    from sspmm_amd import _lib
    L = _lib.lib()
    assert L.sspmm_version() >= 1
    one = 1  # any non-null pointer value; rejected calls never dereference it
    # unsupported vector length (the reference prints and carries on: sspmm.cu:582-583)
    assert L.sspmm_f16_f32(4, 4, 64, 64, None, one, one, one, one, one, None) == 1
    assert L.sspmm_f16_f16(4, 2, 64, 64, None, one, one, one, one, one, None) == 1
    # negative sizes, null outputs
    assert L.sspmm_f16_f32(-1, 8, 64, 64, None, one, one, one, one, one, None) == 1
    assert L.sspmm_f16_f32(4, 8, 64, 64, None, None, one, one, one, one, None) == 1
    assert L.sspmm_f16_f32(4, 8, 64, 64, None, one, one, one, one, None, None) == 1
    assert L.sspmm_f16_f32(4, 8, 1 << 20, 1 << 12, None, one, one, one, one, one, None) == 1  # K*N >= 2^31
    # nothing to do is success
    assert L.sspmm_f16_f32(0, 8, 64, 64, None, None, None, None, None, None, None) == 0
    assert L.sspmm_f16_f16(4, 16, 0, 64, None, one, one, one, one, one, None) == 0
    assert L.sspmm_batched_f16_f16(0, 4, 8, 64, 64, None, one, one, one, 0, one, 0, one, 0, None) == 0
    assert L.sspmm_batched_f16_f16(2, 4, 8, 64, 64, None, one, one, one, 0, one, 0, one, 5, None) == 1  # C overlaps
    assert L.sspmm_sorted_row_swizzle(-3, one, one, None) == 1
    assert L.sspmm_sorted_row_swizzle(0, None, None, None) == 0
    assert L.svc_count(8, 8, 8, one, one, 4, 7, one, one, None) == 1  # unknown order
    assert L.svc_count(8, 8, 0, one, one, 4, 0, one, one, None) == 1  # V < 1
    assert L.svc_count(8, 8, 8, one, one, 4, 0, one, None, None) == 1  # no workspace
    assert L.svc_fill(8, 8, 8, one, one, one, 4, 0, one, one, one, None, None) == 1  # values in, no values out
    # plans: unsupported V, no place to put the handle, no pattern
    import ctypes as C
    handle = C.c_void_p()
    assert L.sspmm_plan_create(4, 4, 64, one, 64, 1, 0, None, C.byref(handle)) == 1
    assert L.sspmm_plan_create(4, 8, 64, one, 64, 1, 0, None, None) == 1
    assert L.sspmm_plan_create(4, 8, 64, None, 64, 1, 0, None, C.byref(handle)) == 1
    assert L.sspmm_plan_destroy(None) == 0
    assert L.sspmm_plan_info(None, None) == 1
    assert L.sspmm_plan_batched_f16_f32(None, 1, 64, one, one, one, 0, one, 0, one, 0, None) == 1
    # the linear-layer and attention entry points reject what they do not cover before touching the device
    assert L.sspmm_linear_f16(4, 8, 64, 64, one, one, one, one, None, 7, one, None) == 1       # unknown activation
    assert L.sspmm_linear_f16(4, 4, 64, 64, one, one, one, one, None, 0, one, None) == 1       # unsupported V
    assert L.sspmm_linear_f16(0, 8, 64, 64, None, None, None, None, None, 1, None, None) == 0  # nothing to do
    assert L.sspmm_attention_fm_f16(1, 1, 64, 32, 16, 16, 16, 64, 16, 64, 0.125, None) == 1    # head size
    assert L.sspmm_attention_fm_f16(1, 1, 96, 64, 16, 16, 16, 96, 16, 96, 0.125, None) == 1    # sequence not a multiple of 64
    assert L.sspmm_attention_fm_f16(0, 1, 64, 64, None, None, None, 0, None, 0, 0.125, None) == 0
    for bad_scale in (0.0, -0.125, float("nan"), float("inf")):
        assert L.sspmm_attention_fm_f16(1, 1, 64, 64, 16, 16, 16, 64, 16, 64, bad_scale, None) == 1
    # the one-launch sparse attention block: heads of 32, 64 or 128 features, V of 8 or 16, a positive finite scale, aligned operands
    sa = lambda V=8, F=64, q=16, stride=512, scale=0.125: L.sspmm_sparse_attention_f16(  # noqa: E731
        1, 1, V, F, 8, None, 16, 16, q, stride, 16, 512, 16, 512, scale, 16, 512, None)
    assert sa(V=4) == 1 and sa(F=48) == 1 and sa(F=256) == 1 and sa(q=8) == 1 and sa(stride=4) == 1
    for bad_scale in (0.0, -0.125, float("nan"), float("inf")):
        assert sa(scale=bad_scale) == 1
    assert L.sspmm_sparse_attention_f16(0, 4, 8, 64, 8, None, None, None, None, 0, None, 0, None, 0, 0.125, None, 0, None) == 0
    # ... and its form for heads that lie side by side: no heads, a row pitch below the head's width, a pitch that is not a
    # multiple of 8, a negative stride
    sh = lambda heads=2, ld=384, head=64, stride=128: L.sspmm_sparse_attention_heads_f16(  # noqa: E731
        1, heads, 1, 8, 64, 8, None, 16, 16, 16, stride, head, ld, 16, stride, head, ld, 16, stride, head, ld, 0.125, 16, stride, head, ld, None)
    assert sh(heads=0) == 1 and sh(ld=32) == 1 and sh(ld=388) == 1 and sh(stride=-128) == 1 and sh(ld=1 << 23) == 1
    assert L.svc_workspace_bytes(16, 100, 8) >= 100 * 8
    assert b"invalid" in L.sspmm_error_string(1)
    assert L.sspmm_error_string(0) == b"success"


def test_argument_errors_of_the_dense_block_entries(built_library):
    """Widths, alignments, missing operands and sizes beyond what the kernels address, all rejected on the host."""
    import ctypes as C
    from sspmm_amd import _lib
    L = _lib.lib()
    p = 4096  # a 16-byte aligned pointer value; rejected calls never dereference it

    def rows(outer=2, inner=3, E=64, x=p, x_outer=192, x_inner=64, a=p, gamma=p, beta=p, total=p, out=p):
        return L.sspmm_add_layernorm_rows_f16(outer, inner, E, x, x_outer, x_inner, a, gamma, beta, 1e-5, total, out, None)

    for bad in (dict(outer=-1), dict(inner=-1), dict(E=96), dict(E=0), dict(x=None), dict(out=None), dict(x_outer=-8), dict(x_outer=4),
                dict(x_inner=12), dict(x=p + 2), dict(a=p + 8), dict(gamma=p + 4), dict(beta=p + 2), dict(total=p + 8), dict(out=p + 8)):
        assert rows(**bad) == 1, bad
    assert rows(outer=0) == 0 and rows(inner=0, x=None) == 0

    def dense(outer=2, inner=3, E=128, x=p, x_outer=384, x_inner=128, pos=None, attn=p, wo=p, mlp=256, w1=p, w2=p, n_out=128, head_dim=0, wt=p,
              bt=p, x_out=p, out=p):
        return L.sspmm_block_dense_f16(outer, inner, E, x, x_outer, x_inner, pos, 1.0, attn, wo, p, p, p, 1e-5, mlp, w1, p, w2, p, p, p, 1e-5,
                                       n_out, head_dim, wt, bt, x_out, out, None)

    for bad in (dict(outer=-1), dict(inner=-1), dict(E=64), dict(E=192), dict(E=1024), dict(mlp=0), dict(mlp=128), dict(mlp=-256),
                dict(mlp=(1 << 20) + 256), dict(n_out=96), dict(n_out=-64), dict(n_out=(1 << 20) + 64), dict(n_out=0), dict(wt=None), dict(x=None),
                dict(out=None), dict(wo=None), dict(w1=None), dict(w2=None), dict(x_outer=4), dict(x_inner=-8), dict(head_dim=16),
                dict(head_dim=64, n_out=192), dict(x=p + 2), dict(pos=p + 8), dict(attn=p + 2), dict(bt=p + 8), dict(x_out=p + 4), dict(out=p + 2)):
        assert dense(**bad) == 1, bad
    assert dense(outer=0) == 0 and dense(inner=0, x=None) == 0

    def pack(src=p, rows=256, cols=128, group=32, dst=p, count=1):
        return L.sspmm_block_pack_f16(count, (C.c_void_p * 1)(src), (C.c_int32 * 1)(rows), (C.c_int32 * 1)(cols), (C.c_int32 * 1)(group), dst, None)

    for bad in (dict(count=-1), dict(src=None), dict(src=p + 2), dict(dst=None), dict(dst=p + 8), dict(group=16), dict(group=48), dict(rows=240),
                dict(rows=0), dict(cols=96), dict(cols=0), dict(rows=1 << 20, cols=1 << 10)):
        assert pack(**bad) == 1, bad
    assert L.sspmm_block_pack_f16(1, None, None, None, None, p, None) == 1
    assert L.sspmm_block_pack_f16(0, None, None, None, None, None, None) == 0

    def folded(outer=2, inner=3, E=128, x=p, attn=p, wo=p, w21=p, affine=p, n_out=128, head_dim=0, wt=p, x_out=p, out=p):
        return L.sspmm_block_dense_folded_f16(outer, inner, E, x, 384, 128, attn, wo, p, p, p, 1e-5, w21, affine, p, p, 1e-5, n_out, head_dim, wt, p,
                                              x_out, out, None)

    for bad in (dict(outer=-1), dict(E=64), dict(E=192), dict(n_out=96), dict(n_out=0), dict(wt=None), dict(x=None), dict(attn=None), dict(wo=None),
                dict(w21=None), dict(affine=None), dict(affine=p + 8), dict(w21=p + 2), dict(out=None), dict(head_dim=16)):
        assert folded(**bad) == 1, bad
    assert folded(outer=0) == 0 and folded(inner=0, attn=None) == 0

    def embed(outer=2, inner=3, E=128, tokens=p, size=8, t_outer=1, t_inner=2, table=p, vocab=7, pos=p, n_out=128, head_dim=0, wt=p, bt=p, x_out=p, out=p):
        return L.sspmm_block_embed_f16(outer, inner, E, tokens, size, t_outer, t_inner, table, vocab, pos, 1.0, p, p, 1e-5, n_out, head_dim, wt, bt,
                                       x_out, out, None)

    for bad in (dict(outer=-1), dict(inner=-1), dict(E=64), dict(tokens=None), dict(tokens=p + 4), dict(tokens=p + 2, size=4), dict(size=2),
                dict(t_outer=-1), dict(t_inner=-2), dict(table=None), dict(table=p + 8), dict(vocab=0), dict(pos=None), dict(pos=p + 2), dict(n_out=96),
                dict(n_out=0), dict(wt=None), dict(head_dim=48), dict(bt=p + 8), dict(x_out=p + 4), dict(out=None)):
        assert embed(**bad) == 1, bad
    assert embed(outer=0) == 0 and embed(inner=0, tokens=None) == 0

    def fold(count=1, src=p, folds=1, E=128, mlp=256, w1=p, b1=p, w2=p, b2=p, w21=p, affine=p):
        one = lambda v: (C.c_void_p * 1)(v)  # noqa: E731
        return L.sspmm_block_fold_f16(count, one(src), (C.c_int32 * 1)(256), (C.c_int32 * 1)(128), (C.c_int32 * 1)(32), p, folds, E, (C.c_int32 * 1)(mlp),
                                      one(w1), one(b1), one(w2), one(b2), w21, affine, None)

    for bad in (dict(count=-1), dict(src=None), dict(folds=-1), dict(E=64), dict(E=0), dict(mlp=0), dict(mlp=128), dict(mlp=-256),
                dict(mlp=(1 << 20) + 256), dict(w1=None), dict(w2=None), dict(w1=p + 2), dict(b1=p + 8), dict(w2=p + 4), dict(w21=None), dict(w21=p + 8),
                dict(affine=None), dict(affine=p + 4)):
        assert fold(**bad) == 1, bad
    assert L.sspmm_block_fold_f16(0, None, None, None, None, None, 0, 256, None, None, None, None, None, None, None, None) == 0

    # (with what the matrix's rounding leaves: the entries above are these without it)
    split = lambda outer=2, rest=p, w21=p, affine=p, attn=p: L.sspmm_block_dense_split_f16(  # noqa: E731
        outer, 3, 128, p, 384, 128, attn, p, p, p, p, 1e-5, w21, rest, affine, p, p, 1e-5, 128, 0, p, p, p, p, None)
    assert all(split(**bad) == 1 for bad in (dict(rest=p + 8), dict(w21=None), dict(affine=None), dict(attn=None), dict(outer=-1)))
    assert split(outer=0) == 0 and split(outer=0, rest=None) == 0
    one = lambda v: (C.c_void_p * 1)(v)  # noqa: E731
    assert L.sspmm_block_fold_split_f16(0, None, None, None, None, None, 1, 128, (C.c_int32 * 1)(256), one(p), one(p), one(p), one(p), p, p + 8, p, p, None) == 1
    assert L.sspmm_block_fold_split_f16(0, None, None, None, None, None, 0, 128, None, None, None, None, None, None, None, None, p + 2, None) == 1
    assert L.sspmm_block_fold_split_f16(0, None, None, None, None, None, 0, 256, None, None, None, None, None, None, None, None, p, None) == 0
    checked = lambda outer, ok: L.sspmm_block_embed_checked_f16(outer, 3, 128, p, 8, 1, 2, p, 7, p, 1.0, p, p, 1e-5, 128, 0, p, p, p, p, ok, None)  # noqa: E731
    assert checked(2, p + 2) == 1 and checked(-1, p) == 1 and checked(0, p) == 0

    assert L.svc_split_row_ptr(-1, 4, p, p, p, p, None) == 1 and L.svc_split_row_ptr(1, 4, p, None, p, p, None) == 1
    assert L.svc_split_row_ptr(0, 0, None, None, None, None, None) == 0


def test_argument_errors_of_the_encoder_tail(built_library):
    """Sizes that a workgroup's LDS does not hold, token counts, alignments and missing operands, rejected on the host; the
    sizes that Python takes for the launch are those that the entry takes."""
    from sspmm_amd import _lib
    from sspmm_amd.layers import encoder_tail_fits
    L = _lib.lib()
    p = 4096

    def tail(hidden=768, ffn=3072, tokens=64, V=16, x=p, context=p, offsets=p, cols=p, values=p, bias=p, gamma=p, beta=p, out=p):
        w = (offsets, cols, values, bias)
        return L.sspmm_encoder_tail_f16(hidden, ffn, tokens, V, x, context, *w, gamma, beta, 1e-5, *w, *w, gamma, beta, 1e-5, out, None)

    for bad in (dict(hidden=-16), dict(ffn=-1), dict(tokens=-4), dict(V=4), dict(V=32), dict(hidden=776), dict(ffn=3080),
                dict(hidden=1040), dict(hidden=1024, ffn=4096), dict(hidden=0), dict(ffn=0), dict(x=None), dict(context=None), dict(out=None),
                dict(offsets=None), dict(gamma=None), dict(x=p + 1), dict(context=p + 3), dict(out=p + 1), dict(values=p + 8), dict(cols=p + 2)):
        assert tail(**bad) == 1, bad
    assert tail(tokens=0) == 0
    for V in (8, 16):
        for hidden in range(V, 1100, 3 * V):
            for ffn in range(V, 5000, 7 * V):
                assert encoder_tail_fits(hidden, ffn, 64, V) == (L.sspmm_encoder_tail_fits(hidden, ffn, 64, V) == 1), (hidden, ffn, V)


def test_norm_weights_of_another_length_do_not_reach_a_kernel():
    """A LayerNorm whose weight or bias has been replaced by one of another length is left to the module, which refuses it: the
    kernels read as many elements as there are features."""
    import torch
    from sspmm_amd.attention import _rows_norm_applies
    from sspmm_amd.layers import _tail_norm
    E, x = 128, torch.zeros(2, 128, dtype=torch.float16)
    made = lambda: torch.nn.LayerNorm(E).half()  # noqa: E731
    assert _tail_norm(made(), E, -1) is not None and _rows_norm_applies(made(), x)
    for name in ("weight", "bias"):
        for shape in ((E - 16,), (E + 16,), (2, E // 2), (0,)):
            ln = made()
            setattr(ln, name, torch.nn.Parameter(torch.ones(shape, dtype=torch.float16)))
            assert _tail_norm(ln, E, -1) is None and not _rows_norm_applies(ln, x), (name, shape)


def test_python_operator_rejects_bad_arguments(built_library):
    import torch
    import sspmm_amd
    t = torch.zeros(4, dtype=torch.int32)
    h = torch.zeros(4, dtype=torch.float16)
    with pytest.raises(ValueError):
        sspmm_amd.spmm(None, t, t, h, h.reshape(2, 2), 4)
    with pytest.raises(TypeError):
        sspmm_amd.spmm(None, t.long(), t, h, h.reshape(2, 2), 8)
    with pytest.raises(ValueError):  # CPU tensors: there is no CPU path
        sspmm_amd.spmm(None, t, t, h, h.reshape(2, 2), 8)
