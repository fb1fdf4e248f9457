"""The model-side callers (sspmm_amd.layers) against dense torch arithmetic on the same weights."""
import numpy as np
import pytest
import torch

import sspmm_amd
from sspmm_amd import synth
from sspmm_amd.layers import SparseEncoderLayer, SparseLinear
from gpu_util import dev, max_rel_err

pytestmark = pytest.mark.gpu


def _vector_sparse_linear(out_f, in_f, V, sparsity, seed, **kw):
    vs = synth.vector_sparse(out_f, in_f, V, sparsity, seed=seed, std=0.05)
    return SparseLinear.from_cvse(in_f, V, dev(vs.row_offsets), dev(vs.col_idx), dev(vs.values), **kw)


@pytest.mark.parametrize("V", [8, 16])
def test_sparse_linear_from_cvse_matches_dense_matmul(built_library, V):
    lin = _vector_sparse_linear(256, 192, V, 0.8, seed=70, out_dtype=torch.float32)
    x = torch.randn(192, 136, device="cuda", generator=torch.Generator("cuda").manual_seed(1)).half()
    want = lin.dense_weight().float() @ x.float()
    got = lin(x)
    assert got.dtype == torch.float32 and got.shape == (256, 136)
    assert max_rel_err(got.cpu().numpy(), want.cpu().numpy()) <= 2e-5


def test_sparse_linear_from_unstructured_dense_weight(built_library):
    """A scalar-sparse weight goes through the SVC on the GPU; the layer still computes W @ x (+ bias)."""
    g = torch.Generator("cuda").manual_seed(2)
    W = torch.randn(128, 300, device="cuda", generator=g).half()
    W[torch.rand(128, 300, device="cuda", generator=g) < 0.9] = 0
    bias = torch.randn(128, device="cuda", generator=g).half()
    for order in ("sorted", "cpython"):
        lin = SparseLinear.from_dense(W, 8, bias=bias, order=order, out_dtype=torch.float32)
        assert torch.equal(lin.dense_weight(), W)
        x = torch.randn(300, 64, device="cuda", generator=g).half()
        want = W.float() @ x.float() + bias.float()[:, None]
        assert max_rel_err(lin(x).cpu().numpy(), want.cpu().numpy()) <= 2e-5
    with pytest.raises(ValueError):
        lin(torch.zeros(64, 300, device="cuda", dtype=torch.float16))


def test_encoder_layer_matches_the_same_layer_with_dense_products(built_library):
    hidden, heads, ffn, V, batch, seq = 256, 4, 1024, 16, 2, 64
    mk = lambda o, i, s: _vector_sparse_linear(o, i, V, 0.9, seed=s)
    layer = SparseEncoderLayer(hidden, heads, ffn, mk(hidden, hidden, 1), mk(hidden, hidden, 2), mk(hidden, hidden, 3),
                               mk(hidden, hidden, 4), mk(ffn, hidden, 5), mk(hidden, ffn, 6)).cuda().half()
    x = torch.randn(hidden, batch * seq, device="cuda", generator=torch.Generator("cuda").manual_seed(3)).half()
    dense = {n: getattr(layer, n).dense_weight() for n in ("qkv", "o", "ffn1", "ffn2")}
    assert torch.equal(dense["qkv"], torch.cat([layer.q.dense_weight(), layer.k.dense_weight(), layer.v.dense_weight()]))
    with torch.no_grad():
        got = layer(x, batch, seq)
        gelu = torch.nn.functional.gelu
        want = layer(x, batch, seq, linear=lambda name, lin, t: (
            gelu(dense["ffn1"].float() @ t.float()) if name == "ffn1_gelu" else dense[name].float() @ t.float()).half())
    assert got.shape == (hidden, batch * seq)
    assert max_rel_err(got.float().cpu().numpy(), want.float().cpu().numpy()) <= 1e-2


@pytest.mark.parametrize("H,T", [(768, 4096), (256, 128), (100, 36), (1024, 68), (1, 4), (3072, 520), (4096, 16)])
@pytest.mark.parametrize("residual", [True, False])
def test_feature_major_add_layernorm_matches_torch(built_library, H, T, residual):
    """The fused kernel against torch's LayerNorm on the transposed sum: same fp16 sum, statistics in fp32."""
    from sspmm_amd.layers import add_layernorm
    g = torch.Generator("cuda").manual_seed(H + T)
    x = (torch.randn(H, T, device="cuda", generator=g) * 2 + 0.5).half()
    a = torch.randn(H, T, device="cuda", generator=g).half() if residual else None
    ln = torch.nn.LayerNorm(H).cuda().half()
    with torch.no_grad():
        ln.weight.copy_(torch.randn(H, device="cuda", generator=g))
        ln.bias.copy_(torch.randn(H, device="cuda", generator=g))
        got = add_layernorm(x, a, ln)
        s = x if a is None else x + a
        want = torch.nn.functional.layer_norm(s.t().float(), (H,), ln.weight.float(), ln.bias.float(), ln.eps).t()
    assert got.shape == (H, T) and got.dtype == torch.float16
    assert (got.float() - want).abs().max().item() <= 4e-3 * max(1.0, want.abs().max().item())
    # shapes outside the kernel's limits take torch and agree too
    if T % 4 == 0 and H > 1:
        odd = add_layernorm(x[:, :T - 1].contiguous(), None if a is None else a[:, :T - 1].contiguous(), ln)
        assert (odd.float() - want[:, :T - 1]).abs().max().item() <= 4e-3 * max(1.0, want.abs().max().item())


@pytest.mark.parametrize("H", [127, 128, 129, 512, 513, 640, 769, 1023, 1025])
@pytest.mark.parametrize("T", [4, 76])
def test_feature_major_add_layernorm_at_the_edges_of_its_kernels(built_library, H, T):
    test_feature_major_add_layernorm_matches_torch(built_library, H, T, True)


def _attention_reference(q, k, v, batch, heads, seq, scale):
    """fp32 attention of feature-major [heads * d, batch * seq] operands, written out with plain matmuls."""
    d = q.shape[0] // heads
    f = lambda t: t.float().view(heads, d, batch, seq).permute(2, 0, 3, 1)  # noqa: E731  [batch, heads, seq, d]
    p = torch.softmax(f(q) @ f(k).transpose(-1, -2) * scale, dim=-1)
    return (p @ f(v)).permute(1, 3, 0, 2).reshape(heads * d, batch * seq)


@pytest.mark.parametrize("T", [64, 61])
def test_feature_major_add_layernorm_reads_only_operands_of_its_sizes(built_library, T):
    """Weights of another length or type and a residual that is elsewhere go to the module, which refuses them."""
    from sspmm_amd.layers import add_layernorm
    H = 128
    x = torch.ones(H, T, dtype=torch.float16, device="cuda")
    with torch.no_grad():
        for name in ("weight", "bias"):
            for t in (torch.ones(H - 16), torch.ones(2, H // 2)):
                ln = torch.nn.LayerNorm(H).cuda().half()
                setattr(ln, name, torch.nn.Parameter(t.cuda().half()))
                with pytest.raises(RuntimeError):
                    add_layernorm(x, None, ln)
        ln = torch.nn.LayerNorm(H).cuda().half()
        with pytest.raises(RuntimeError):
            add_layernorm(x, x.cpu(), ln)
        want = add_layernorm(x, x, ln)
        for t in (torch.zeros(2 * H).cuda().half()[::2], torch.zeros(H).cuda().half()):
            ln.bias = torch.nn.Parameter(t)
            assert torch.equal(add_layernorm(x, x, ln), want)


@pytest.mark.parametrize("batch,heads,seq", [(1, 1, 64), (2, 3, 128), (3, 2, 192), (8, 12, 512), (1, 2, 320), (1, 1, 1024)])
def test_feature_major_attention_matches_fp32_attention(built_library, batch, heads, seq):
    """sspmm_attention_fm_f16 through the C ABI, operands as three row ranges of one fused projection."""
    from sspmm_amd import _lib
    from sspmm_amd.layers import attention_fm
    hidden, T = heads * 64, batch * seq
    g = torch.Generator("cuda").manual_seed(seq + heads)
    qkv = torch.randn(3 * hidden, T, device="cuda", generator=g).half()
    qkv[:hidden] *= 2.0  # scores spread over several units, so the softmax is far from uniform
    scale = 0.125
    got = attention_fm(qkv, hidden, heads, batch, seq)
    assert got is not None and got.shape == (hidden, T) and got.dtype == torch.float16
    want = _attention_reference(qkv[:hidden], qkv[hidden:2 * hidden], qkv[2 * hidden:], batch, heads, seq, scale)
    assert (got.float() - want).abs().max().item() <= 2e-3 * max(1.0, want.abs().max().item())
    # separate operands with their own leading dimension, output into a wider array: the columns beyond stay untouched
    ld, ld_out = T + 24, T + 8
    q, k, v = (torch.randn(hidden, ld, device="cuda", generator=g).half() for _ in range(3))
    out = torch.full((hidden, ld_out), 7.0, dtype=torch.float16, device="cuda")
    rc = _lib.lib().sspmm_attention_fm_f16(batch, heads, seq, 64, q.data_ptr(), k.data_ptr(), v.data_ptr(), ld, out.data_ptr(),
                                           ld_out, scale, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    want = _attention_reference(q[:, :T], k[:, :T], v[:, :T], batch, heads, seq, scale)
    assert (out[:, :T].float() - want).abs().max().item() <= 2e-3 * max(1.0, want.abs().max().item())
    assert torch.all(out[:, T:] == 7.0)


@pytest.mark.parametrize("batch,heads,seq", [(1, 1, 1), (1, 2, 7), (3, 1, 24), (2, 2, 32), (2, 3, 33), (1, 1, 63), (5, 2, 65), (1, 4, 100), (3, 2, 127),
                                             (2, 1, 160), (1, 1, 191), (8, 12, 500), (1, 2, 1000), (3, 1, 64)])
def test_feature_major_attention_on_ragged_sequences(built_library, batch, heads, seq):
    """Lengths either side of the 32 keys of a wave, the 64 of a block and the eight tokens of a piece, rows at odd elements: the
    context against fp32 attention (same bound as for whole blocks), nothing written beside it, and what surrounds the
    operands (NaN) not let in."""
    from sspmm_amd import _lib
    from sspmm_amd.layers import attention_fm
    hidden, T = heads * 64, batch * seq
    g = torch.Generator("cuda").manual_seed(seq + heads)
    qkv = torch.randn(3 * hidden, T, device="cuda", generator=g).half()
    got = attention_fm(qkv, hidden, heads, batch, seq)
    want = _attention_reference(qkv[:hidden], qkv[hidden:2 * hidden], qkv[2 * hidden:], batch, heads, seq, 0.125)
    assert got.shape == want.shape and (got.float() - want).abs().max().item() <= 2e-3 * max(1.0, want.abs().max().item())
    for scale, lead in ((0.125, 3), (2.0, 1)):
        ld, ld_out = T + 5, T + 3
        q, k, v = (torch.full((hidden * ld + 16,), float("nan"), dtype=torch.float16, device="cuda") for _ in range(3))
        views = [t[lead:lead + hidden * ld].view(hidden, ld) for t in (q, k, v)]
        for t in views:
            t[:, :T] = (torch.randn(hidden, T, device="cuda", generator=g) * (0.25 if scale > 1 else 1)).half()
        out = torch.full((hidden * ld_out + 16,), 7.0, dtype=torch.float16, device="cuda")
        o = out[lead:lead + hidden * ld_out].view(hidden, ld_out)
        rc = _lib.lib().sspmm_attention_fm_ragged_f16(batch, heads, seq, 64, *(t.data_ptr() for t in views), ld, o.data_ptr(), ld_out, scale,
                                                      torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        want = _attention_reference(*(t[:, :T] for t in views), batch, heads, seq, scale)
        assert (o[:, :T].float() - want).abs().max().item() <= 2e-3 * max(1.0, want.abs().max().item())
        assert torch.all(o[:, T:] == 7.0) and torch.all(out[:lead] == 7.0) and torch.all(out[lead + hidden * ld_out:] == 7.0)


@pytest.mark.parametrize("seq", [1, 37, 63, 64, 100, 333])
def test_feature_major_attention_keeps_infinite_values(built_library, seq):
    """One infinite or NaN value: its feature is infinite or NaN for every query, whole blocks or not (scores within a few units of each
    other, so that no probability vanishes in fp16), and the features beside it are what they are without it."""
    from sspmm_amd.layers import attention_fm
    qkv = (torch.randn(3 * 64, seq, device="cuda", generator=torch.Generator("cuda").manual_seed(seq)) * 0.5).half()
    plain = attention_fm(qkv, 64, 1, 1, seq)
    for feature, value in ((5, float("inf")), (21, -float("inf")), (40, float("nan"))):
        qkv[128 + feature, seq // 2] = value
    got = attention_fm(qkv, 64, 1, 1, seq)
    assert torch.all(got[5] == float("inf")) and torch.all(got[21] == -float("inf")) and torch.all(got[40].isnan())
    rest = [f for f in range(64) if f not in (5, 21, 40)]
    assert torch.equal(got[rest], plain[rest])


def test_ragged_attention_is_left_to_torch_where_more_than_the_values_is_wanted(built_library, monkeypatch):
    """A layer on 333 tokens with differentiable products in the place of the sparse ones: gradients of the input and of the
    projections are those through torch's attention (here written out in fp32; the same operations twice, so what differs is the
    order of library sums), which tensor subclasses, dispatch modes, vmap and forward-mode gradients get as well.  Values
    alone come from the kernel, in gradient mode too."""
    import torch.utils._python_dispatch as dispatch
    import sspmm_amd.layers as layers_mod
    hidden, heads, ffn, V, seq = 128, 2, 256, 8, 333
    mk = lambda o, i, s: _vector_sparse_linear(o, i, V, 0.8, seed=s)
    layer = SparseEncoderLayer(hidden, heads, ffn, mk(hidden, hidden, 1), mk(hidden, hidden, 2), mk(hidden, hidden, 3),
                               mk(hidden, hidden, 4), mk(ffn, hidden, 5), mk(hidden, ffn, 6)).cuda().half()
    dense = {n: getattr(layer, n).dense_weight() for n in ("qkv", "o", "ffn1_gelu", "ffn2")}
    g = torch.Generator("cuda").manual_seed(8)
    x0, direction = (torch.randn(hidden, seq, device="cuda", generator=g).half() for _ in range(2))

    def attention(q, k, v, scale):
        p = torch.softmax(q.float() @ k.float().transpose(-1, -2).contiguous() * scale, dim=-1)
        return (p @ v.float()).half()

    monkeypatch.setattr(torch.nn.functional, "scaled_dot_product_attention", attention)

    def gradients():
        x, w = x0.clone().requires_grad_(), {n: d.clone().requires_grad_() for n, d in dense.items()}
        layer(x, 1, seq, linear=lambda name, lin, t: torch.nn.functional.gelu(w[name] @ t) if name == "ffn1_gelu" else w[name] @ t).backward(direction)
        return [x.grad] + [w[n].grad for n in dense]

    got, kernel = gradients(), layers_mod.attention_fm
    with monkeypatch.context() as m:
        m.setattr(layers_mod, "attention_fm", lambda *a, **kw: None)
        want = gradients()
    for a, b in zip(got, want):
        assert a is not None and b.abs().max() > 0 and max_rel_err(a.float().cpu().numpy(), b.float().cpu().numpy()) <= 1e-2

    qkv = torch.randn(3 * hidden, seq, device="cuda", generator=g).half()
    call = lambda t: kernel(t, hidden, heads, 1, seq)  # noqa: E731

    class Watcher(dispatch.TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        pass

    assert call(qkv) is not None and call(qkv.clone().requires_grad_()) is None
    assert call(qkv.as_subclass(Sub)) is None
    with torch.no_grad():
        assert call(qkv.clone().requires_grad_()) is not None
        with Watcher():
            assert call(qkv) is None
        with torch.autograd.forward_ad.dual_level():
            assert call(torch.autograd.forward_ad.make_dual(qkv, qkv)) is None
        with torch.autocast("cuda"):
            assert call(qkv) is None
    assert torch.vmap(lambda t: torch.zeros(()) if call(t) is None else torch.ones(()))(qkv[None]).item() == 0


def test_feature_major_attention_with_maxima_that_keep_growing(built_library):
    """Keys whose norm grows along the sequence: the running maximum of a query's scores rises by many units from one
    block of keys to the next, so the kernel moves the reference point of its exponentials again and again (it
    skips that step while the maximum grows by little)."""
    from sspmm_amd.layers import attention_fm
    batch, heads, seq = 2, 2, 512
    hidden, T = heads * 64, batch * seq
    g = torch.Generator("cuda").manual_seed(11)
    qkv = torch.randn(3 * hidden, T, device="cuda", generator=g)
    growth = 1.0 + 7.0 * (torch.arange(T, device="cuda") % seq).float() / seq
    qkv[hidden:2 * hidden] *= growth
    qkv[:hidden] = qkv[:hidden].abs() * 2.0   # same-sign queries and keys of growing size: scores rise with the position
    qkv[hidden:2 * hidden] = qkv[hidden:2 * hidden].abs()
    qkv = qkv.half()
    got = attention_fm(qkv, hidden, heads, batch, seq)
    want = _attention_reference(qkv[:hidden], qkv[hidden:2 * hidden], qkv[2 * hidden:], batch, heads, seq, 0.125)
    assert (got.float() - want).abs().max().item() <= 2e-3 * max(1.0, want.abs().max().item())


def test_feature_major_attention_rejects_what_it_does_not_cover(built_library):
    from sspmm_amd import _lib
    L = _lib.lib()
    t = torch.zeros(64, 1024, dtype=torch.float16, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    args = lambda **kw: [kw.get("batch", 1), kw.get("heads", 1), kw.get("seq", 64), kw.get("d", 64), t.data_ptr() + kw.get("off", 0),  # noqa: E731
                         t.data_ptr(), t.data_ptr(), kw.get("ld", 1024), t.data_ptr(), 1024, 0.125, s]
    assert L.sspmm_attention_fm_f16(*args()) == 0
    for bad in (dict(d=32), dict(seq=96), dict(seq=16448, ld=16448), dict(ld=1020), dict(off=2), dict(seq=512, batch=4, ld=1024), dict(batch=-1)):
        assert L.sspmm_attention_fm_f16(*args(**bad)) == 1, bad
    assert L.sspmm_attention_fm_f16(*args(batch=0)) == 0
    torch.cuda.synchronize()


def test_attention_fm_takes_and_refuses_what_it_did(built_library):
    """Scales that the kernel does not take are an error for whole blocks and somebody else's for other lengths, where empty
    batches are as well; whole blocks of an empty batch are an empty context; projections that begin at any element are no
    whole blocks."""
    from sspmm_amd.layers import attention_fm
    z = lambda *shape: torch.zeros(*shape, dtype=torch.float16, device="cuda")  # noqa: E731
    for scale in (0.0, -0.125, float("nan"), float("inf")):
        assert attention_fm(z(192, 63), 64, 1, 1, 63, scale) is None
        with pytest.raises(RuntimeError):
            attention_fm(z(192, 64), 64, 1, 1, 64, scale)
    assert attention_fm(z(192, 0), 64, 1, 0, 63) is None and attention_fm(z(192, 0), 64, 1, 1, 0) is None
    assert attention_fm(z(192, 0), 64, 1, 0, 64).shape == (64, 0)
    with pytest.raises(RuntimeError):
        attention_fm(z(192 * 64 + 1)[1:].view(192, 64), 64, 1, 1, 64)
    assert attention_fm(z(192 * 63 + 1)[1:].view(192, 63), 64, 1, 1, 63) is not None


def test_encoder_layer_at_the_benchmark_shape_takes_the_attention_kernel(built_library):
    """hidden 768, 12 heads, 8 x 512 tokens: the layer with the feature-major attention kernel against the same layer
    with torch's attention between relayout copies."""
    hidden, heads, ffn, V, batch, seq = 768, 12, 3072, 16, 8, 512
    mk = lambda o, i, s: _vector_sparse_linear(o, i, V, 0.9, seed=s)
    layer = SparseEncoderLayer(hidden, heads, ffn, mk(hidden, hidden, 1), mk(hidden, hidden, 2), mk(hidden, hidden, 3),
                               mk(hidden, hidden, 4), mk(ffn, hidden, 5), mk(hidden, ffn, 6)).cuda().half()
    x = torch.randn(hidden, batch * seq, device="cuda", generator=torch.Generator("cuda").manual_seed(5)).half()
    import sspmm_amd.layers as layers_mod
    with torch.no_grad():
        got = layer(x, batch, seq)
        kernel = layers_mod.attention_fm
        layers_mod.attention_fm = lambda *a, **kw: None
        try:
            want = layer(x, batch, seq)
        finally:
            layers_mod.attention_fm = kernel
    assert max_rel_err(got.float().cpu().numpy(), want.float().cpu().numpy()) <= 1e-2


def test_encoder_layer_at_the_benchmark_shape_matches_dense_products(built_library):
    """hidden 768, 12 heads, FFN 3072, 8 x 512 tokens, six weights V = 16 at 90 %: the layer against the same layer whose
    four products are dense fp32 matmuls on the densified weights (an independent check of the sparse products at the
    full shape: nothing of this library computes the comparison's products)."""
    hidden, heads, ffn, V, batch, seq = 768, 12, 3072, 16, 8, 512
    mk = lambda o, i, s: _vector_sparse_linear(o, i, V, 0.9, seed=s)
    layer = SparseEncoderLayer(hidden, heads, ffn, mk(hidden, hidden, 1), mk(hidden, hidden, 2), mk(hidden, hidden, 3),
                               mk(hidden, hidden, 4), mk(ffn, hidden, 5), mk(hidden, ffn, 6)).cuda().half()
    x = torch.randn(hidden, batch * seq, device="cuda", generator=torch.Generator("cuda").manual_seed(6)).half()
    dense = {n: getattr(layer, n).dense_weight().float() for n in ("qkv", "o", "ffn1", "ffn2")}
    assert torch.equal(dense["qkv"], torch.cat([layer.q.dense_weight(), layer.k.dense_weight(), layer.v.dense_weight()]).float())
    # the weights are held once: q, k and v are views of the fused layer's arrays, and state_dict names them once
    assert layer.q.values.data_ptr() == layer.qkv.values.data_ptr()
    assert not any(key.startswith(("q.", "k.", "v.", "ffn1_gelu.")) for key in layer.state_dict())
    gelu = torch.nn.functional.gelu
    with torch.no_grad():
        got = layer(x, batch, seq)
        want = layer(x, batch, seq, linear=lambda name, lin, t: (
            gelu(dense["ffn1"] @ t.float()) if name == "ffn1_gelu" else dense[name] @ t.float()).half())
    assert got.shape == (hidden, batch * seq)
    assert max_rel_err(got.float().cpu().numpy(), want.float().cpu().numpy()) <= 1e-2


def test_sparse_linear_drops_its_plan_when_the_buffers_move(built_library):
    lin = _vector_sparse_linear(256, 192, 16, 0.8, seed=72)
    lin.make_plan(64)
    assert lin.plan is not None
    lin = lin.half()   # any conversion or move goes through _apply
    assert lin.plan is None
    x = torch.randn(192, 64, device="cuda", generator=torch.Generator("cuda").manual_seed(7)).half()
    want = lin.dense_weight().float() @ x.float()
    assert max_rel_err(lin(x).float().cpu().numpy(), want.cpu().numpy()) <= 2e-3


@pytest.mark.parametrize("V,out_f,in_f,N", [(16, 3072, 768, 4096), (8, 64, 100, 72), (16, 128, 5000, 64), (8, 256, 96, 33)])
@pytest.mark.parametrize("activation", [None, "gelu"])
@pytest.mark.parametrize("with_bias", [False, True])
def test_linear_epilogue_matches_separate_bias_and_gelu(built_library, V, out_f, in_f, N, activation, with_bias):
    """sspmm_linear_f16 against the fp32 product with bias and erf-GELU applied in fp32: the gather kernel (wide N),
    the staged gather kernel (few waves, N <= 64, K above the split-row kernel's threshold) and the scalar kernel
    (N not a multiple of 8)."""
    from sspmm_amd.spmm import linear
    vs = synth.vector_sparse(out_f, in_f, V, 0.9, seed=out_f + N, std=0.05)
    g = torch.Generator("cuda").manual_seed(N)
    x = torch.randn(in_f, N, device="cuda", generator=g).half()
    bias = torch.randn(out_f, device="cuda", generator=g).half() if with_bias else None
    ro, ci, va = dev(vs.row_offsets), dev(vs.col_idx), dev(vs.values)
    got = linear(ro, ci, va, x, V, bias=bias, activation=activation)
    want = sspmm_amd.spmm(None, ro, ci, va, x, V, out_dtype=torch.float32)
    if bias is not None:
        want = want + bias.float()[:, None]
    if activation == "gelu":
        want = torch.nn.functional.gelu(want)
    assert got.dtype == torch.float16 and got.shape == (out_f, N)
    assert max_rel_err(got.float().cpu().numpy(), want.cpu().numpy()) <= 2e-3
    if bias is None and activation is None:
        assert torch.equal(got, sspmm_amd.spmm(None, ro, ci, va, x, V))


def test_sparse_linear_fuses_bias_and_activation(built_library):
    lin = _vector_sparse_linear(256, 192, 16, 0.8, seed=71, activation="gelu")
    lin.bias = torch.randn(256, device="cuda", generator=torch.Generator("cuda").manual_seed(4)).half()
    x = torch.randn(192, 200, device="cuda", generator=torch.Generator("cuda").manual_seed(5)).half()
    want = torch.nn.functional.gelu(lin.dense_weight().float() @ x.float() + lin.bias.float()[:, None])
    assert max_rel_err(lin(x).float().cpu().numpy(), want.cpu().numpy()) <= 2e-3
    from sspmm_amd import _lib
    L = _lib.lib()
    assert L.sspmm_linear_f16(1, 16, 8, 8, 0, 0, 0, 0, 0, 2, 0, 0) == 1  # unknown activation


@pytest.mark.parametrize("H,T,residual", [(255, 27416, True), (256, 27304, True), (256, 27308, True), (512, 20476, False), (512, 20480, False),
                                         (513, 20440, False), (1024, 10236, False), (1024, 10240, False), (1024, 10240, True)])
def test_feature_major_add_layernorm_of_more_than_the_caches_hold(built_library, H, T, residual):
    """Either side of 40 MiB of operands, from where most widths go through LDS."""
    test_feature_major_add_layernorm_matches_torch(built_library, H, T, residual)


@pytest.mark.parametrize("V", [8, 16])
@pytest.mark.parametrize("hidden,ffn,batch,seq", [(64, 64, 1, 4), (64, 256, 1, 20), (128, 64, 3, 64), (320, 1280, 1, 132), (512, 2048, 2, 68),
                                                  (768, 3072, 3, 100), (768, 3072, 8, 512), (1024, 1024, 1, 1100),
                                                  (64, 128, 1, 1), (128, 128, 1, 15), (256, 64, 1, 18), (512, 2048, 3, 37), (768, 3072, 5, 333)])
def test_encoder_layers_tail_in_one_launch_matches_the_separate_launches(built_library, V, hidden, ffn, batch, seq):
    """Output projection, norms and feed-forward products in one launch against the same layer step by step: token counts
    around the 16 and 64 of a workgroup and its lines and no multiple of the 4 of a thread, rows of 0 to a few hundred vectors, with and without biases.
    The steps round the same values to fp16 at the same places; their sums run in another order, so an activation may
    land on the fp16 next to it (2^-11 relative), which the two norms and products behind it carry on: 2^-8 of the largest."""
    import sspmm_amd.layers as layers_mod
    heads = hidden // 64
    g = torch.Generator("cuda").manual_seed(hidden + seq)
    calls, kernel, pays, least = [], layers_mod.encoder_tail, layers_mod.encoder_tail_pays, layers_mod.TAIL_TOKENS

    def sparse(o, i, seed, bias):
        keep = torch.rand(o // V, i, device="cuda", generator=g) < 0.1
        keep[0] = False                            # a vector-row without vectors
        keep[-1] = torch.arange(i, device="cuda") < 40
        offsets = torch.zeros(o // V + 1, dtype=torch.int32, device="cuda")
        offsets[1:] = keep.sum(1).cumsum(0).int()
        cols = keep.nonzero()[:, 1].int().contiguous()
        values = (torch.randn(cols.numel() * V, device="cuda", generator=g) * 0.1).half()
        return SparseLinear.from_cvse(i, V, offsets, cols, values, torch.randn(o, device="cuda", generator=g).half() if bias else None)

    for bias in (True, False):
        layer = SparseEncoderLayer(hidden, heads, ffn, *(sparse(hidden, hidden, s, True) for s in range(3)), sparse(hidden, hidden, 4, bias),
                                   sparse(ffn, hidden, 5, bias), sparse(hidden, ffn, 6, bias)).cuda().half().eval()
        with torch.no_grad():
            for ln in (layer.ln1, layer.ln2):
                ln.weight.copy_(1 + 0.1 * torch.randn(hidden, device="cuda", generator=g))
                ln.bias.copy_(0.1 * torch.randn(hidden, device="cuda", generator=g))
            x = torch.randn(hidden, batch * seq, device="cuda", generator=g).half()
            want = layer(x, batch, seq, linear=lambda name, lin, t: lin(t))
            layers_mod.encoder_tail = lambda *a: (calls.append(1), kernel(*a))[1]
            layers_mod.encoder_tail_pays, layers_mod.TAIL_TOKENS = lambda *a: True, 1
            try:
                got = layer(x, batch, seq)
                hook = layer.o.register_forward_hook(lambda *a: None)  # (whoever watches a layer gets it called)
                hooked = layer(x, batch, seq)
                hook.remove()
            finally:
                layers_mod.encoder_tail, layers_mod.encoder_tail_pays, layers_mod.TAIL_TOKENS = kernel, pays, least
        assert max_rel_err(got.float().cpu().numpy(), want.float().cpu().numpy()) <= 2.0 ** -8
        assert torch.equal(hooked, want)
    assert len(calls) == 2


@pytest.mark.parametrize("V", [8, 16])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("hidden,ffn,tokens", [(64, 128, 1), (128, 64, 15), (320, 1280, 37), (768, 3072, 333), (512, 2048, 1100), (1024, 1024, 64)])
def test_encoder_layers_tail_matches_dense_fp32_products(built_library, V, bias, hidden, ffn, tokens):
    """The one launch against products with the densified weights in fp32, GELU and norms by torch in fp32, rounded to fp16 where the
    kernel rounds (projections, sums, norms, hidden features): nothing of this library computes the comparison.  An
    activation may land on the fp16 next to it (2^-11 relative), which the norms and products behind it carry on: 2^-8 of the largest."""
    import sspmm_amd.layers as layers_mod
    g = torch.Generator("cuda").manual_seed(hidden + tokens + V)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    o, f1, f2 = (_vector_sparse_linear(a, b, V, 0.9, seed=a + b + i) for i, (a, b) in enumerate(((hidden, hidden), (ffn, hidden), (hidden, ffn))))
    n1, n2 = torch.nn.LayerNorm(hidden).cuda().half(), torch.nn.LayerNorm(hidden).cuda().half()
    with torch.no_grad():
        for t in (n1, n2):
            t.weight.copy_(1 + 0.1 * rand(hidden))
            t.bias.copy_(0.1 * rand(hidden))
        for lin in (o, f1, f2):
            lin.bias = rand(lin.out_features).half() if bias else None
        x, context = rand(hidden, tokens).half(), rand(hidden, tokens).half()
        dev = x.get_device()
        got = layers_mod.encoder_tail(x, context, ffn, V, layers_mod._tail_weight(o, hidden, hidden, V, dev), layers_mod._tail_norm(n1, hidden, dev),
                                      layers_mod._tail_weight(f1, hidden, ffn, V, dev), layers_mod._tail_weight(f2, ffn, hidden, V, dev),
                                      layers_mod._tail_norm(n2, hidden, dev))

        def product(lin, t):
            y = lin.dense_weight().float() @ t.float()
            return y if lin.bias is None else y + lin.bias.float()[:, None]

        def norm(ln, s):
            return torch.nn.functional.layer_norm(s.t().float(), (hidden,), ln.weight.float(), ln.bias.float(), ln.eps).t().half()

        n = norm(n1, x + product(o, context).half())
        want = norm(n2, n + product(f2, torch.nn.functional.gelu(product(f1, n)).half()).half())
    assert max_rel_err(got.float().cpu().numpy(), want.float().cpu().numpy()) <= 2.0 ** -8


@pytest.mark.parametrize("V,hidden,ffn,tokens", [(16, 16, 4112, 20), (8, 64, 4096, 33), (8, 72, 64, 16), (16, 256, 96, 65), (16, 1024, 2048, 18)])
def test_encoder_layers_tail_of_few_and_of_most_rows(built_library, V, hidden, ffn, tokens):
    """Fewer vector-rows than a workgroup has waves, and as many hidden features as fit: the bound of the test above."""
    from sspmm_amd.layers import encoder_tail_fits
    assert encoder_tail_fits(hidden, ffn, tokens, V)
    for bias in (True, False):
        test_encoder_layers_tail_matches_dense_fp32_products(built_library, V, bias, hidden, ffn, tokens)


@pytest.mark.parametrize("where,name", [("o", "values"), ("ffn1", "bias"), ("ln1", "weight"), ("layer", "ffn2")])
def test_encoder_layers_tail_takes_an_instances_own_attribute_first(built_library, monkeypatch, where, name):
    """What a program has put into a module's __dict__ comes before the parameter, buffer or module of that name."""
    import copy
    import sspmm_amd.layers as layers_mod
    monkeypatch.setattr(layers_mod, "encoder_tail_pays", lambda *a: True)
    monkeypatch.setattr(layers_mod, "TAIL_TOKENS", 1)
    sp = [_vector_sparse_linear(o, i, 8, 0.8, seed=k, bias=torch.zeros(o, device="cuda").half())
          for k, (o, i) in enumerate([(128, 128)] * 4 + [(256, 128), (128, 256)])]
    layer = SparseEncoderLayer(128, 2, 256, *sp).cuda().half().eval()
    x = torch.randn(128, 64, device="cuda", generator=torch.Generator("cuda").manual_seed(1)).half()
    owner = layer if where == "layer" else getattr(layer, where)
    old = getattr(owner, name)
    new = copy.deepcopy(old)
    with torch.no_grad():
        (new.values if name == "ffn2" else new).mul_(0.5).add_(0.25)
        owner.__dict__[name] = new
        want = layer(x, 1, 64, linear=lambda n, lin, t: lin(t))
        assert max_rel_err(layer(x, 1, 64).float().cpu().numpy(), want.float().cpu().numpy()) <= 2.0 ** -8
        del owner.__dict__[name]
        assert max_rel_err(layer(x, 1, 64).float().cpu().numpy(), want.float().cpu().numpy()) > 2.0 ** -8


def test_encoder_layers_tail_runs_on_the_weights_of_that_moment(built_library, monkeypatch):
    """A hook behind the projections that gives the layer other weights: the launch behind the attention has their addresses,
    not those of the arrays that went away (looked at without launching), and its result is the one with them."""
    import sspmm_amd.layers as layers_mod
    hidden, ffn, V, seq = 128, 256, 8, 64
    mk = lambda o, i, s: _vector_sparse_linear(o, i, V, 0.8, seed=s)
    layer = SparseEncoderLayer(hidden, 2, ffn, mk(hidden, hidden, 1), mk(hidden, hidden, 2), mk(hidden, hidden, 3),
                               mk(hidden, hidden, 4), mk(ffn, hidden, 5), mk(hidden, ffn, 6)).cuda().half().eval()
    x = torch.randn(hidden, seq, device="cuda", generator=torch.Generator("cuda").manual_seed(9)).half()
    monkeypatch.setattr(layers_mod, "encoder_tail_pays", lambda *a: True)
    monkeypatch.setattr(layers_mod, "TAIL_TOKENS", 1)
    new = [-lin.values for lin in (layer.o, layer.ffn1, layer.ffn2)]

    def replace(*_):
        layer.o.values, layer.ffn1.values, layer.ffn2.values = (t.clone() for t in new)

    layer.qkv.register_forward_hook(replace)
    seen = []
    with torch.no_grad():
        with monkeypatch.context() as m:
            m.setattr(layers_mod, "encoder_tail", lambda x, context, F, V, o, n1, f1, f2, n2: seen.extend(w[2] for w in (o, f1, f2)))
            layer(x, 1, seq)
        assert seen == [lin.values.data_ptr() for lin in (layer.o, layer.ffn1, layer.ffn2)]
        want = layer(x, 1, seq, linear=lambda name, lin, t: lin(t))
        assert max_rel_err(layer(x, 1, seq).float().cpu().numpy(), want.float().cpu().numpy()) <= 2.0 ** -8


@pytest.mark.parametrize("H", [40, 200, 512, 768, 1000, 1100])
@pytest.mark.parametrize("T", [1, 2, 3, 5, 15, 18, 63, 65, 130, 1021])
def test_feature_major_add_layernorm_on_any_number_of_tokens(built_library, H, T):
    """The kernels on rows at odd elements against the same kernels on the same tokens padded to a multiple of four (the same
    operations on every token: the same bits), with what surrounds the operands (NaN) not let in and nothing written beside
    the result; and the module once more for whoever wants gradients."""
    from sspmm_amd import _lib
    from sspmm_amd.layers import add_layernorm
    g = torch.Generator("cuda").manual_seed(H + T)
    wide = (T + 3) // 4 * 4
    ln = torch.nn.LayerNorm(H).cuda().half()
    xs, rs = (torch.randn(H, wide, device="cuda", generator=g).half() for _ in range(2))
    with torch.no_grad():
        ln.weight.copy_(1 + 0.1 * torch.randn(H, device="cuda", generator=g))
        ln.bias.copy_(0.1 * torch.randn(H, device="cuda", generator=g))
        want = add_layernorm(xs, rs, ln)[:, :T]
        x, r = xs[:, :T].contiguous(), rs[:, :T].contiguous()
        assert torch.equal(add_layernorm(x, r, ln), want)
        assert torch.equal(add_layernorm(x, None, ln), add_layernorm(xs, None, ln)[:, :T])
        x_in, r_in = (torch.full((H * T + 8,), float("nan"), dtype=torch.float16, device="cuda") for _ in range(2))
        out = torch.full((H * T + 8,), 7.0, dtype=torch.float16, device="cuda")
        x_in[3:3 + H * T], r_in[1:1 + H * T] = x.flatten(), r.flatten()
        rc = _lib.lib().sspmm_add_layernorm_ragged_f16(H, T, x_in[3:].data_ptr(), r_in[1:].data_ptr(), ln.weight.data_ptr(), ln.bias.data_ptr(),
                                                       ln.eps, out[1:].data_ptr(), torch.cuda.current_stream().cuda_stream)
        assert rc == 0 and torch.equal(out[1:1 + H * T].view(H, T), want)
        assert out[0] == 7.0 and torch.all(out[1 + H * T:] == 7.0)
    assert add_layernorm(x, r, ln).requires_grad == (T % 4 != 0)
