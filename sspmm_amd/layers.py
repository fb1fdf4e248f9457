"""Model-side callers of the SpMM: a linear layer whose weight is vector-sparse, and the
transformer encoder layer of the BERT-base shaped benchmark configuration built from six of
them.

The reference reaches its kernels from torch modules the same way (the sparse attention block
calls `bspmm(row_indices, row_offsets, column_indices, values, v, vec_length)`, reference
end2end/sspmm_e2e/spattention.py:179; the weight-sparse layers of its evaluation are the SpMM
harness shapes, reference SSpMM/sspmm_test.cpp:141,189).  Activations are kept feature-major
([features, tokens]) so that every weight-sparse product is C[out, tokens] = W[out, in] @
X[in, tokens], the SpMM's native orientation, and no transposes sit between the layers.

Inference only: the operators have no backward pass.  Everything that is not an SpMM (attention
scores, softmax, LayerNorm, GELU, bias) runs in torch-ROCm; the products with the sparse
weights run in the HIP kernels behind the C ABI.
"""
import math

import numpy as np
import torch

from . import _lib
from .attention import _eager, _eager_inference, _plain_module
from .spmm import linear as linear_op, spmm
from .svc import svc


class SparseLinear(torch.nn.Module):
    """y[out, tokens] = W @ x[in, tokens] (+ bias[:, None]) with W in the vector-sparse format.

    Build one with `from_dense` (a dense weight whose zero pattern is already vector-structured
    or not: RowMerge on the GPU packs whatever is there) or `from_cvse` (arrays as the SpMM
    takes them)."""

    plan = None  # (until make_plan; here, so that a call without one does not go through the module's lookup of what it lacks: 1 us)

    def __init__(self, in_features, out_features, vec_length, row_offsets, column_indices, values, bias=None,
                 out_dtype=torch.float16, activation=None):
        super().__init__()
        self.activation = activation  # None or "gelu": applied to W @ x + bias
        if out_features % vec_length:
            raise ValueError("out_features must be a multiple of vec_length")
        self.in_features, self.out_features, self.vec_length = in_features, out_features, vec_length
        self.out_dtype = out_dtype
        self.register_buffer("row_offsets", row_offsets)
        self.register_buffer("column_indices", column_indices)
        self.register_buffer("values", values)
        self.register_buffer("bias", bias)

    @classmethod
    def from_cvse(cls, in_features, vec_length, row_offsets, column_indices, values, bias=None, **kw):
        m_vec = row_offsets.numel() - 1
        return cls(in_features, m_vec * vec_length, vec_length, row_offsets, column_indices, values, bias, **kw)

    @classmethod
    def concat(cls, layers):
        """One layer whose output is the outputs of `layers` stacked along the feature axis: their patterns
        concatenated along M.  Three projections of the same input (query, key, value) become one SpMM that reads
        the input once."""
        first = layers[0]
        if any(l.in_features != first.in_features or l.vec_length != first.vec_length or l.out_dtype != first.out_dtype
               for l in layers):
            raise ValueError("the layers must share in_features, vec_length and output type")
        offsets, base = [first.row_offsets[:1]], 0
        for l in layers:
            offsets.append(l.row_offsets[1:] + base)
            base += int(l.column_indices.numel())
        biases = [l.bias for l in layers]
        bias = None
        if any(b is not None for b in biases):
            bias = torch.cat([b if b is not None else torch.zeros(l.out_features, dtype=torch.float16, device=first.values.device)
                              for b, l in zip(biases, layers)])
        return cls(first.in_features, sum(l.out_features for l in layers), first.vec_length,
                   torch.cat(offsets).to(torch.int32).contiguous(), torch.cat([l.column_indices for l in layers]).contiguous(),
                   torch.cat([l.values for l in layers]).contiguous(), bias, out_dtype=first.out_dtype)

    @classmethod
    def from_dense(cls, weight, vec_length, bias=None, order="sorted", **kw):
        """weight: [out, in] fp16 GPU tensor; its non-zeros are merged V rows at a time (SVC on the GPU)."""
        if weight.dtype != torch.float16 or not weight.is_cuda:
            raise TypeError("weight must be a float16 GPU tensor")
        out_features, in_features = weight.shape
        mask = weight != 0
        row_ptr = torch.zeros(out_features + 1, dtype=torch.int32, device=weight.device)
        row_ptr[1:] = mask.sum(dim=1).cumsum(0).to(torch.int32)
        col_ind = mask.nonzero()[:, 1].to(torch.int32).contiguous()
        r = svc(row_ptr, col_ind, weight[mask].contiguous(), out_features, in_features, vec_length, order=order)
        return cls(in_features, out_features, vec_length, r.vec_row_ptr, r.vec_col, r.vec_val, bias, **kw)

    def rows(self, first, last):
        """The layer of output features first .. last-1 (multiples of vec_length) as a layer of its own whose arrays
        are views of this one's: nothing is copied, and the view is not registered anywhere."""
        V = self.vec_length
        if first % V or last % V or not 0 <= first <= last <= self.out_features:
            raise ValueError("row range must be multiples of vec_length inside [0, out_features]")
        off = self.row_offsets[first // V:last // V + 1]
        lo, hi = int(off[0]), int(off[-1])
        return SparseLinear(self.in_features, last - first, V, (off - lo).to(torch.int32), self.column_indices[lo:hi],
                            self.values[lo * V:hi * V], None if self.bias is None else self.bias[first:last],
                            out_dtype=self.out_dtype, activation=self.activation)

    def _apply(self, fn, *args, **kw):
        # a plan lives on the device it was built on and describes the row offsets it was built from: when the
        # buffers are moved or converted it is dropped, and make_plan has to be called again
        self.plan = None
        return super()._apply(fn, *args, **kw)

    def make_plan(self, max_tokens):
        """Builds the pattern's plan (sspmm_amd.Plan) for inputs of up to max_tokens columns; later calls of the
        layer use it.  Worth it for weights whose merged rows are uneven (unstructured pruning through RowMerge)."""
        from .plan import Plan
        self.plan = Plan(self.row_offsets, self.vec_length, self.in_features, max_N=max_tokens)
        return self.plan

    def forward(self, x, activation="layer"):
        """activation: "layer" applies the layer's own (self.activation); None or "gelu" override it for this call."""
        act = self.activation if activation == "layer" else activation
        if x.dim() != 2 or x.size(0) != self.in_features:
            raise ValueError("x must be [in_features, tokens] = [%d, *], got %s" % (self.in_features, tuple(x.shape)))
        plan = self.plan
        if plan is not None and x.size(1) > plan.max_N:
            plan = None
        fuse = plan is None and self.out_dtype == torch.float16 and (self.bias is None or self.bias.dtype == torch.float16)
        if fuse and (self.bias is not None or act is not None):
            # bias and activation in the product's epilogue: one launch, the output written once
            return linear_op(self.row_offsets, self.column_indices, self.values, x.contiguous(), self.vec_length,
                             bias=self.bias, activation=act)
        y = spmm(None, self.row_offsets, self.column_indices, self.values, x.contiguous(), self.vec_length,
                 out_dtype=self.out_dtype, plan=plan)
        if self.bias is not None:
            y = y + self.bias[:, None].to(y.dtype)
        if act == "gelu":
            y = torch.nn.functional.gelu(y)
        return y

    def dense_weight(self):
        """The weight as a dense [out, in] fp16 tensor (for checks)."""
        V = self.vec_length
        off = self.row_offsets.cpu().numpy()
        cols = self.column_indices.cpu().numpy()
        vals = self.values.cpu().numpy().reshape(-1, V)
        W = np.zeros((self.out_features, self.in_features), np.float16)
        for i in range(off.size - 1):
            W[i * V:(i + 1) * V, cols[off[i]:off[i + 1]]] = vals[off[i]:off[i + 1]].T
        return torch.from_numpy(W).to(self.values.device)


_PLAIN = (torch.Tensor, torch.nn.Parameter)


def _of_features(t, features, dev):
    """Whether t is one contiguous fp16 value per feature on GPU dev."""
    return t.dtype == torch.float16 and t.get_device() == dev and t.dim() == 1 and t.numel() == features and t.is_contiguous()


def add_layernorm(x, a, ln):
    """LayerNorm over the features of the feature-major sum x + a ([features, tokens] fp16; a may be None) with the
    weights of `ln` (a torch.nn.LayerNorm over `features`).  One HIP kernel (sspmm_add_layernorm_f16 of the C ABI)
    where its shape limits hold, torch on transposed copies otherwise."""
    shape, dev = x.shape, x.get_device()
    (H, T), w, b = shape, ln.weight, ln.bias
    whole = T % 4 == 0
    ok = (x.dtype == torch.float16 and x.is_cuda and x.is_contiguous() and H <= 4096 and
          (a is None or (a.dtype == torch.float16 and a.is_contiguous() and a.shape == shape and a.get_device() == dev)) and
          w is not None and tuple(ln.normalized_shape) == (H,) and _of_features(w, H, dev) and (b is None or _of_features(b, H, dev)))
    if ok and not whole:
        # (tokens that are no multiple of 4 had torch's module, which whoever wants gradients or watches it still gets)
        ok = (0 < T <= 1 << 30 and _plain_module(ln, torch.nn.LayerNorm) and _eager_inference() and type(x) is torch.Tensor and
              (a is None or type(a) is torch.Tensor) and type(w) in _PLAIN and (b is None or type(b) in _PLAIN))
    if not ok:
        s = x if a is None else x + a
        return ln(s.t()).t().contiguous()
    out = torch.empty_like(x)
    L = _lib.lib()
    rc = _lib.call(L.sspmm_add_layernorm_f16 if whole else L.sspmm_add_layernorm_ragged_f16, x.device, H, T, x.data_ptr(),
                   0 if a is None else a.data_ptr(), w.data_ptr(), 0 if b is None else b.data_ptr(), float(ln.eps), out.data_ptr())
    _lib.check(rc, "sspmm_add_layernorm_f16")
    return out


# Longest sequence that is no multiple of 64 for which the kernel is ahead of torch's attention between two relayout copies whatever the
# batch: 12 heads, 8 x 500 tokens 25 us against 69, 4 x 2000 136 against 215, 2 x 4001 267 against 463; 5000 tokens are ahead with few
# heads and behind with many (2 x 12 heads 410 / 472 us, 8 x 16 1990 / 2000), 6001 behind from 24 heads on (565 / 561), 12001 well behind
# (2170 / 1666): torch's kernel has larger tiles, and the copies, which are linear, stop counting.
ATTENTION_FM_RAGGED = 4096


def attention_fm(qkv, hidden, heads, batch, seq, scale=None):
    """softmax(Q^T K * scale) V per (batch element, head) on the fused feature-major projections qkv
    [3 * hidden, batch * seq] fp16 (rows 0 .. hidden-1 the queries, then keys, then values; token b * seq + s in
    column b * seq + s); returns the context [hidden, batch * seq], or None where the kernel's shape limits do not
    hold or, with sequences that are no multiple of 64, more than the values is wanted (the caller then takes another route)."""
    d = hidden // heads
    T = batch * seq
    whole = seq % 64 == 0
    if not (qkv.dtype == torch.float16 and qkv.is_cuda and qkv.is_contiguous() and tuple(qkv.shape) == (3 * hidden, T) and
            d == 64 and hidden == heads * d and 1 <= seq <= (16384 if whole else ATTENTION_FM_RAGGED)):
        return None
    scale = float(1.0 / math.sqrt(d) if scale is None else scale)
    # (ragged lengths had torch's attention, which takes any scale, and which whoever wants gradients or watches it still gets)
    if not whole and not (batch >= 1 and 0 < scale <= 3.0e38 and type(qkv) is torch.Tensor and _eager() and
                          not (torch.is_grad_enabled() and qkv.requires_grad)):
        return None
    out = torch.empty(hidden, T, dtype=torch.float16, device=qkv.device)
    esz = qkv.element_size()
    L = _lib.lib()
    rc = _lib.call(L.sspmm_attention_fm_f16 if whole else L.sspmm_attention_fm_ragged_f16, qkv.device, batch, heads, seq, d, qkv.data_ptr(),
                   qkv.data_ptr() + hidden * T * esz, qkv.data_ptr() + 2 * hidden * T * esz, T, out.data_ptr(), T, scale)
    _lib.check(rc, "sspmm_attention_fm_f16")
    return out


# LDS of a workgroup of the launch below, which holds 16 tokens' activations of both widths, value tiles, row tables and biases
_TAIL_LDS = 160 * 1024


def encoder_tail_fits(hidden, ffn, tokens, V):
    """Whether sspmm_encoder_tail_f16 takes these sizes."""
    lds = 32 * (hidden + 1 + max(hidden, ffn) + 1) + 16 * (528 if V == 8 else 1024) + 16 * ((2 * hidden + ffn) // V + 6) + 2048 + 2 * (2 * hidden + ffn)
    return V in (8, 16) and 0 < hidden <= 1024 and 0 < ffn <= 8192 and hidden % V == 0 and ffn % V == 0 and 0 < tokens <= 1 << 24 and \
        lds <= _TAIL_LDS


TAIL_TOKENS = 1024


def encoder_tail_pays(hidden, tokens, vectors, cus):
    """Whether the one launch is ahead of the five it replaces; `vectors`: stored vectors of its three weights.  A workgroup of
    16 tokens, one per CU, takes as long however few of them there are: a layer with it some 35 us and 0.45 us per thousand
    vectors, where the separate launches' time follows the tokens.  Layer with 768 features (replayed, so that the host plays
    no part), separate / one launch, us: V = 16 at 90 % (33 000 vectors) 512 tokens 41 / 45, 1024 52 / 47, 2048 63 / 53, 4096 83 / 59; V = 8 at 90 %
    (66 000) 1024 56 / 65, 2048 72 / 71, 3072 89 / 77, 4096 100 / 79; at 85 % (99 000) 2048 79 / 83, 3072 99 / 89, 4096 111 / 92; at 80 %
    (133 000) 2048 83 / 95, 4096 122 / 105, 8192 212 / 200; V = 16 at 50 % (166 000) 4096 139 / 123, 8192 235 / 232; V = 8 at 70 %
    (199 000) 2048 99 / 126, 4096 151 / 140, 8192 265 / 267.  Called one by one the separate launches keep the host
    busy for 65 to 70 us and these 35 to 45, so where the device's times are level or a little apart the one launch is ahead: 512 features, V = 8 at
    90 %, 1024 tokens 42 / 45 replayed, 65 / 45 called, at 80 % 2048 tokens 58 / 58, 65 / 59.  Beyond one workgroup per CU a nearly empty last round
    costs a whole one: 8192 tokens 135 / 105 (V = 16 at 90 %) and 192 / 174 (99 000 vectors), 6144 143 / 138 (66 000) and 160 / 163 (99 000); 512 features,
    7168 tokens 108 / 94 (29 000) and 128 / 119 (59 000).  The lines were drawn for a launch 3 us slower and are on its safe side now: between them
    and where the two are level the separate launches run although the one is ahead (33 000 vectors 1024 and 6144 tokens 52 / 47 and 116 / 99, 99 000
    3072 tokens 99 / 89, 133 000 to 199 000 4096 tokens; 256 features, V = 8 at 90 %, 6144 and 8192 tokens 58 / 54 and 64 / 56)."""
    if vectors > 100000 or tokens < max(TAIL_TOKENS, vectors // 30):
        return False
    per_round = 16 * cus
    rounds = -(-tokens // per_round)
    return rounds == 1 or (hidden >= 512 and 20 * tokens >= 17 * rounds * per_round)


_CUS = {}


def _cus(device):
    n = _CUS.get(device)
    if n is None:
        n = _CUS[device] = torch.cuda.get_device_properties(device).multi_processor_count
    return n


def _tail_weight(m, in_features, out_features, V, dev):
    """(row offsets, columns, values, bias) of a SparseLinear of these sizes that does nothing but its product, without a plan,
    on the current GPU, as the launch takes them; None otherwise."""
    if not (_plain_module(m, SparseLinear) and m.in_features == in_features and m.out_features == out_features and m.vec_length == V and
            m.out_dtype == torch.float16 and m.__dict__.get("plan") is None):
        return None
    own = m._buffers
    if not own.keys().isdisjoint(m.__dict__):  # (an attribute of the instance comes before a buffer; here and below)
        return None
    off, col, val, bias = own.get("row_offsets"), own.get("column_indices"), own.get("values"), own.get("bias")
    if not (_plain_tensor(off, torch.int32, dev) and _plain_tensor(col, torch.int32, dev) and _plain_tensor(val, torch.float16, dev) and
            off.numel() == out_features // V + 1 and val.numel() >= col.numel() * V and
            (bias is None or (_plain_tensor(bias, torch.float16, dev) and bias.numel() == out_features))):
        return None
    at = val.data_ptr()
    return None if at % 16 else (off.data_ptr(), col.data_ptr(), at, None if bias is None else bias.data_ptr())


def _plain_tensor(t, dtype, dev):
    return type(t) in _PLAIN and t.dtype == dtype and t.get_device() == dev and t.is_contiguous()


def _tail_norm(ln, features, dev):
    """(weight, bias, eps) of a plain LayerNorm over `features`, or None."""
    if not (_plain_module(ln, torch.nn.LayerNorm) and ln.normalized_shape == (features,)):
        return None
    own = ln._parameters
    if not own.keys().isdisjoint(ln.__dict__):
        return None
    w, b = own.get("weight"), own.get("bias")
    if not (type(w) in _PLAIN and _of_features(w, features, dev) and (b is None or (type(b) in _PLAIN and _of_features(b, features, dev)))):
        return None
    return w.data_ptr(), None if b is None else b.data_ptr(), float(ln.eps)


def encoder_tail(x, context, ffn, V, o, norm1, ffn1, ffn2, norm2):
    """LayerNorm2(n + ffn2(gelu(ffn1(n)))) with n = LayerNorm1(x + o(context)) on feature-major activations
    [hidden, tokens] fp16 in one launch; the weights and norms as _tail_weight and _tail_norm give them."""
    out = torch.empty_like(x)
    rc = _lib.call(_lib.lib().sspmm_encoder_tail_f16, x.device, x.size(0), ffn, x.size(1), V, x.data_ptr(),
                   context.data_ptr(), *o, *norm1, *ffn1, *ffn2, *norm2, out.data_ptr())
    _lib.check(rc, "sspmm_encoder_tail_f16")
    return out


class _WithGelu:
    """A SparseLinear called with the GELU behind it."""

    def __init__(self, layer):
        self.layer = layer

    in_features = property(lambda self: self.layer.in_features)
    out_features = property(lambda self: self.layer.out_features)

    def dense_weight(self):
        return self.layer.dense_weight()

    def __call__(self, x):
        return self.layer(x, activation="gelu")


class SparseEncoderLayer(torch.nn.Module):
    """Post-LayerNorm transformer encoder layer with vector-sparse Q, K, V, output and FFN weights
    and dense attention, on feature-major activations x[hidden, batch * seq]."""

    def __init__(self, hidden, heads, ffn, q, k, v, o, ffn1, ffn2):
        super().__init__()
        self.hidden, self.heads, self.ffn = hidden, heads, ffn
        self.o, self.ffn1, self.ffn2 = o, ffn1, ffn2
        # query, key and value projections as one SpMM over the three patterns stacked along M.  The fused layer is
        # the only copy the module keeps (q, k and v below are views of its arrays), so the weights are held once and
        # state_dict names them once.
        self.qkv = SparseLinear.concat([q, k, v])
        self._qkv_rows = (0, q.out_features, q.out_features + k.out_features,
                          q.out_features + k.out_features + v.out_features)
        self.ln1 = torch.nn.LayerNorm(hidden)
        self.ln2 = torch.nn.LayerNorm(hidden)

    q = property(lambda self: self.qkv.rows(self._qkv_rows[0], self._qkv_rows[1]))
    k = property(lambda self: self.qkv.rows(self._qkv_rows[1], self._qkv_rows[2]))
    v = property(lambda self: self.qkv.rows(self._qkv_rows[2], self._qkv_rows[3]))

    @property
    def ffn1_gelu(self):
        """The first feed-forward product with its GELU in the product's epilogue: ffn1 itself, called with the
        activation (no second module, no second copy of the arrays)."""
        return _WithGelu(self.ffn1)

    def _attention(self, qkv, batch, seq):
        """qkv: [3 * hidden, batch*seq] feature-major; returns the context [hidden, batch*seq].  One HIP kernel that
        reads and writes the feature-major layout (sspmm_attention_fm_f16 of the C ABI and its ragged form) where its shape limits hold
        (head size 64).  Otherwise torch's attention between two relayout copies:
        one brings the three projections into the [batch, heads, seq, head size] layout it wants contiguous (on
        strided views of the feature-major activations it runs ten times slower), one brings the context back."""
        h, d = self.heads, self.hidden // self.heads
        ctx = attention_fm(qkv, self.hidden, h, batch, seq)
        if ctx is not None:
            return ctx
        c = qkv.view(3, h, d, batch, seq).permute(0, 3, 1, 4, 2).contiguous()
        ctx = torch.nn.functional.scaled_dot_product_attention(c[0], c[1], c[2], scale=1.0 / math.sqrt(d))
        return ctx.permute(1, 3, 0, 2).reshape(self.hidden, batch * seq)

    def _one_launch_tail(self, x, context):
        """What encoder_tail takes besides the activations, where everything behind the attention may run in that one launch
        and is ahead so: nothing but the values is wanted, plain layers and norms, sizes that a workgroup's LDS holds."""
        if type(x) is not torch.Tensor or x.dim() != 2 or x.size(1) < TAIL_TOKENS:  # (small calls are not kept waiting by the rest)
            return None
        H, dev = self.hidden, x.get_device()
        if not (type(self) is SparseEncoderLayer and x.is_cuda and x.dtype == torch.float16 and x.is_contiguous() and x.size(0) == H and
                type(context) is torch.Tensor and context.shape == x.shape and context.dtype == x.dtype and context.get_device() == dev and
                context.is_contiguous()):
            return None
        own = self._modules
        if not own.keys().isdisjoint(self.__dict__):
            return None
        o, ffn1, ffn2 = own.get("o"), own.get("ffn1"), own.get("ffn2")
        if not (type(o) is SparseLinear and type(ffn1) is SparseLinear and type(ffn2) is SparseLinear and o.activation is None and
                ffn2.activation is None):
            return None
        V, F, T = o.vec_length, ffn1.out_features, x.size(1)
        vectors = sum(m._buffers["column_indices"].numel() for m in (o, ffn1, ffn2))
        if not (encoder_tail_fits(H, F, T, V) and encoder_tail_pays(H, T, vectors, _cus(x.device)) and _eager_inference()):
            return None
        parts = (_tail_weight(o, H, H, V, dev), _tail_norm(own.get("ln1"), H, dev), _tail_weight(ffn1, H, F, V, dev),
                 _tail_weight(ffn2, F, H, V, dev), _tail_norm(own.get("ln2"), H, dev))
        return None if None in parts else (F, V) + parts

    def forward(self, x, batch, seq, linear=None):
        """x: [hidden, batch*seq] fp16.  `linear(name, layer, x)` may replace how a projection ("qkv", "o",
        "ffn1_gelu", "ffn2"; "ffn1_gelu" is the first feed-forward product with the GELU behind it) is evaluated
        (the benchmark passes a dense matmul there to time the same layer without sparsity)."""
        f = linear or (lambda name, layer, t: layer(t))
        context = self._attention(f("qkv", self.qkv, x), batch, seq)
        # (the weights are looked up when the launch is next: what has run until here may have replaced them)
        tail = self._one_launch_tail(x, context) if linear is None else None
        return self._tail(f, x, context) if tail is None else encoder_tail(x, context, *tail)

    def _tail(self, f, x, context):
        a = f("o", self.o, context)
        x = add_layernorm(x, a, self.ln1)
        y = f("ffn2", self.ffn2, f("ffn1_gelu", self.ffn1_gelu, x))
        return add_layernorm(x, y, self.ln2)
