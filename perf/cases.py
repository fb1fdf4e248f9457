"""The work that users have this library do, as timing cases through its public entry points.

    listed()            the named cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what a program holds before the call: pattern, weights, activations, plan, model
    run(state)          one pass
    work(case)          bytes and operations the pass cannot do without
    tolerance(case)     what two correct implementations of the same precision may differ by

Seven kinds of work, each over its range of sizes:

    spmm       one product with a vector-sparse weight: pruned linear layers and convolutions as a product
    bspmm      a batch of products that share a pattern
    plan       the product with a merged unstructured matrix, whose vector-rows are very uneven, with a plan
    svc        one CSR matrix to the vector-sparse format, with values; or its rows reordered ahead of that
    svc_stack  a dataset's matrices to the format in one stack, each taken out as device arrays
    attention  sparse attention on a mask shared by the heads: the three operators, or the one call
    model      forward pass of the sparse attention encoder
    layer      forward pass of an encoder layer with vector-sparse weights
"""
import math

import torch

import sspmm_amd
from sspmm_amd.attention import SparseAttentionEncoder, sparse_attention
from sspmm_amd.layers import SparseEncoderLayer, SparseLinear

SPARSITIES = (0.7, 0.8, 0.9, 0.95, 0.98)

# matrices of a pruned-weight dataset: shapes and sparsities of the converter's benchmark
STACK_SHAPES = ((512, 512), (2048, 512), (512, 2048))
STACK_SPARSITIES = (0.5, 0.7, 0.8, 0.9, 0.95, 0.98)


def listed():
    return [
        # the smallest call: one 512 x 512 product, launch and host latency
        {"name": "spmm_small", "kind": "spmm", "M": 512, "K": 512, "N": 256, "V": 8, "sparsity": 0.9, "even": True,
         "out": "f16"},
        # a convolution as a product on a 35 x 35 image: uneven rows and a width that is a multiple of nothing
        {"name": "spmm_ragged", "kind": "spmm", "M": 1024, "K": 1152, "N": 1225, "V": 8, "sparsity": 0.9, "even": False,
         "out": "f32"},
        # a convolution as a product on a 56 x 56 image, the widest of the benchmark's single products
        {"name": "spmm_conv", "kind": "spmm", "M": 1024, "K": 2304, "N": 3136, "V": 16, "sparsity": 0.8, "even": True,
         "out": "f32"},
        # a feed-forward weight on 128 independent inputs in one launch
        {"name": "bspmm_ffn", "kind": "bspmm", "M": 2048, "K": 512, "N": 256, "V": 8, "sparsity": 0.9, "even": True,
         "batch": 128, "out": "f32"},
        # a square weight at the dataset's larger width, less sparse, fp16 results
        {"name": "bspmm_square", "kind": "bspmm", "M": 2048, "K": 2048, "N": 512, "V": 8, "sparsity": 0.8, "even": True,
         "batch": 16, "out": "f16"},
        # the product that follows the merge of an unstructured matrix
        {"name": "spmm_skewed", "kind": "plan", "M": 16384, "K": 16384, "N": 256, "V": 8, "mean": 16, "out": "f32"},
        # the merge of that matrix
        {"name": "svc_skewed", "kind": "svc", "M": 16384, "K": 16384, "V": 8, "mean": 16, "order": "cpython",
         "reorder": False},
        # the merge of a dataset's matrices
        {"name": "svc_stack", "kind": "svc_stack", "count": 20, "V": 8, "order": "cpython"},
        # the three operators of the sparse attention block one after the other, a sequence that is no power of two
        {"name": "attention_ops", "kind": "attention", "one_call": False, "heads": 16, "seq": 2000, "dim": 64, "V": 8,
         "sparsity": 0.9},
        # the encoder at its smallest published configuration: many short launches
        {"name": "model_b2", "kind": "model", "batch": 2, "seq": 4096, "heads": 4, "embed": 256, "mlp": 1024, "V": 8,
         "sparsity": 0.9},
        # and at the batch size of the published throughput runs
        {"name": "model_b8", "kind": "model", "batch": 8, "seq": 4096, "heads": 4, "embed": 256, "mlp": 1024, "V": 8,
         "sparsity": 0.9},
        # an encoder layer on 8 x 512 tokens
        {"name": "encoder_layer", "kind": "layer", "batch": 8, "seq": 512, "hidden": 768, "heads": 12, "ffn": 3072, "V": 16,
         "sparsity": 0.9},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A right-hand side's width: a multiple of 64 as often as any number."""
    n = _log(rng, lo, hi)
    return n if rng.random() < 0.5 else max(64, n // 64 * 64)


def draw(rng):
    kind = rng.choice(("spmm", "spmm", "spmm", "bspmm", "bspmm", "plan", "svc", "svc_stack", "attention", "attention",
                       "model", "layer", "layer"))
    V = rng.choice((8, 16))
    if kind in ("spmm", "bspmm"):
        case = {"kind": kind, "M": V * _log(rng, 16, 384), "K": _log(rng, 64, 4608), "N": _width(rng, 8, 4096), "V": V,
                "sparsity": rng.choice(SPARSITIES), "even": rng.random() < 0.5, "out": rng.choice(("f16", "f32"))}
        if kind == "bspmm":
            case["N"] = min(case["N"], 512)
            case["K"] = min(case["K"], 2304)
            most = 64 * 1024 * 1024 // (case["N"] * max(case["M"], 2 * case["K"]))
            case["batch"] = max(2, min(_log(rng, 2, 128), most))
        return case
    if kind == "plan":
        return {"kind": kind, "M": _log(rng, 2048, 16384) // V * V, "K": _log(rng, 2048, 16384), "N": _width(rng, 16, 512),
                "V": V, "mean": rng.choice((8, 16, 24)), "out": rng.choice(("f16", "f32"))}
    if kind == "svc":
        return {"kind": kind, "M": _log(rng, 512, 16384), "K": _log(rng, 512, 16384), "V": V, "mean": rng.choice((8, 16, 32)),
                "order": rng.choice(("cpython", "cpython", "sorted")), "reorder": rng.random() < 0.3}
    if kind == "svc_stack":
        return {"kind": kind, "count": _log(rng, 4, 20), "V": V, "order": rng.choice(("cpython", "cpython", "sorted"))}
    if kind == "attention":
        return {"kind": kind, "one_call": rng.random() < 0.5, "heads": _log(rng, 4, 48), "seq": V * _log(rng, 16, 2048 // V),
                "dim": rng.choice((32, 64, 80, 128)), "V": V, "sparsity": rng.choice((0.9, 0.95))}
    if kind == "model":
        heads, dim = rng.choice((4, 8)), rng.choice((32, 64))
        return {"kind": kind, "batch": _log(rng, 1, 8 if heads * dim <= 256 else 3), "seq": 16 * _log(rng, 32, 256), "heads": heads,
                "embed": heads * dim, "mlp": 1024, "V": V, "sparsity": rng.choice((0.9, 0.95))}
    hidden = rng.choice((512, 768))
    return {"kind": kind, "batch": _log(rng, 1, 8), "seq": _log(rng, 24, 512) if rng.random() < 0.5 else 64 * rng.randint(1, 8),
            "hidden": hidden, "heads": hidden // 64, "ffn": 4 * hidden, "V": V, "sparsity": rng.choice((0.8, 0.9, 0.95))}


# ---- inputs ----------------------------------------------------------------------------------------------------------

def _shuffled(gen, rows, cols, groups, K):
    """A sparse pattern with its groups of V rows and its columns renumbered at random, in row order with the columns
    ascending: the structure of a matrix stays (entries per row, vectors per group), and with it the sizes of what comes
    out, whatever the seed.  groups: (V, number of whole groups).  Returns (rows, cols)."""
    V, G = groups
    to = torch.randperm(G, generator=gen, device="cuda")
    name = torch.randperm(K, generator=gen, device="cuda")
    inside = rows < G * V                              # a last short group stays where it is
    rows = torch.where(inside, to[(rows // V).clamp_max(G - 1)] * V + rows % V, rows) if G else rows
    keys = (rows * K + name[cols]).sort().values
    return keys // K, keys % K


def _offsets(rows, count):
    out = torch.zeros(count + 1, dtype=torch.int64, device="cuda")
    out[1:] = torch.bincount(rows, minlength=count).cumsum(0)
    return out.int()


def _structure():
    """Generator of what a case's matrices have in common whatever the seed."""
    return torch.Generator(device="cuda").manual_seed(1)


def _vector_pattern(gen, m_vec, K, sparsity, even, V=1):
    """Column positions uniform without replacement, ascending: the same count in every row, or drawn over the whole
    matrix (rows then move in groups of V between seeds).  Returns (row_offsets, col_idx)."""
    if even:
        per = max(1, int(round((1.0 - sparsity) * K)))
        cols = torch.rand(m_vec, K, generator=gen, device="cuda").topk(per, dim=1).indices.sort(dim=1).values.reshape(-1)
        return (torch.arange(m_vec + 1, device="cuda") * per).int(), cols.int().contiguous()
    at = (torch.rand(m_vec, K, generator=_structure(), device="cuda") >= sparsity).nonzero()
    rows, cols = _shuffled(gen, at[:, 0], at[:, 1], (V, m_vec // V), K)
    return _offsets(rows, m_vec), cols.int().contiguous()


def _half(gen, shape, std=1.0):
    return (torch.randn(shape, generator=gen, device="cuda") * std).half()


def _values(gen, shape, std):
    """Stored values: normally distributed, none of them zero."""
    v = _half(gen, shape, std)
    return torch.where(v == 0, torch.full_like(v, std), v)


def _zipf_csr(gen, M, K, V, mean):
    """CSR with power-law row lengths (exponent 1.5, at most min(K, 2048)) averaging about `mean`, columns uniform and
    ascending."""
    longest, base = min(K, 2048), _structure()
    u = torch.rand(M, generator=base, device="cuda", dtype=torch.float64).clamp_min(1e-12)
    raw = u.pow(-2.0).floor().clamp_max(1e12)          # P(raw >= x) ~ x^-0.5
    lo, hi = 0.0, float(longest)
    for _ in range(40):
        f = 0.5 * (lo + hi)
        if (raw * f).round().clamp_max(longest).mean().item() < mean:
            lo = f
        else:
            hi = f
    lens = (raw * hi).round().clamp_max(longest).long()
    rows = torch.repeat_interleave(torch.arange(M, device="cuda"), lens)
    cols = torch.randint(0, K, (rows.numel(),), generator=base, device="cuda")
    keys = torch.unique(rows * K + cols)               # a column drawn twice for a row counts once
    rows, cols = _shuffled(gen, keys // K, keys % K, (V, M // V), K)
    return _offsets(rows, M), cols.int().contiguous(), _values(gen, (cols.numel(),), 1.0)


def _sparse_linear(gen, out_features, in_features, V, sparsity):
    offsets, cols = _vector_pattern(gen, out_features // V, in_features, sparsity, True)
    return SparseLinear.from_cvse(in_features, V, offsets, cols, _values(gen, (cols.numel() * V,), 0.02),
                                  _half(gen, (out_features,), 0.02))


def prepare(case, seed):
    kind, V = case["kind"], case["V"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    s = {"case": case, "out": {"f16": torch.float16, "f32": torch.float32}.get(case.get("out"))}
    if kind in ("spmm", "bspmm"):
        M, K, N = case["M"], case["K"], case["N"]
        s["offsets"], s["cols"] = _vector_pattern(gen, M // V, K, case["sparsity"], case["even"])
        # the processing order a caller with uneven rows passes along
        s["rows"] = None if case["even"] else sspmm_amd.sorted_row_swizzle(s["offsets"])
        lead = () if kind == "spmm" else (case["batch"],)
        s["values"] = _values(gen, lead + (s["cols"].numel() * V,), 0.02)
        s["B"] = _half(gen, lead + (K, N))
    elif kind == "plan":
        M, K, N = case["M"], case["K"], case["N"]
        ptr, col, val = _zipf_csr(gen, M, K, V, case["mean"])
        r = sspmm_amd.svc(ptr, col, val, M, K, V)
        s["offsets"], s["cols"], s["values"] = r.vec_row_ptr, r.vec_col, r.vec_val
        s["B"] = _half(gen, (K, N))
        s["plan"] = sspmm_amd.Plan(r.vec_row_ptr, V, K, max_N=N)
    elif kind == "svc":
        s["csr"] = _zipf_csr(gen, case["M"], case["K"], V, case["mean"])
    elif kind == "svc_stack":
        s["rows"], ptrs, cols, base = [0], [torch.zeros(1, dtype=torch.int64, device="cuda")], [], 0
        for i in range(case["count"]):
            M, K = STACK_SHAPES[i % 3]
            offsets, col = _vector_pattern(gen, M, K, STACK_SPARSITIES[(i // 3) % 6], False, V)
            s["rows"].append(s["rows"][-1] + M)
            ptrs.append(offsets[1:].long() + base)
            cols.append(col)
            base += col.numel()
        s["ptr"], s["col"] = torch.cat(ptrs).int(), torch.cat(cols)
        s["val"] = _values(gen, (base,), 0.02)
    elif kind == "attention":
        heads, seq, dim = case["heads"], case["seq"], case["dim"]
        s["offsets"], s["cols"] = _vector_pattern(gen, seq // V, seq, case["sparsity"], False)
        s["rows"] = torch.argsort(s["offsets"].diff(), stable=True).int()
        s["q"], s["k"], s["v"] = (_half(gen, (heads, seq, dim)) for _ in range(3))
    elif kind == "model":
        torch.manual_seed(seed)
        s["model"] = SparseAttentionEncoder(257, case["embed"], case["heads"], case["sparsity"], case["seq"], case["mlp"],
                                            case["mlp"], vec_length=V, layers=4, seed=seed).cuda().half().eval()
        s["tokens"] = torch.randint(0, 257, (case["batch"], case["seq"]), generator=gen, device="cuda")
    else:
        hid, ffn, sp = case["hidden"], case["ffn"], case["sparsity"]
        q, k, v, o = (_sparse_linear(gen, hid, hid, V, sp) for _ in range(4))
        s["layer"] = SparseEncoderLayer(hid, case["heads"], ffn, q, k, v, o, _sparse_linear(gen, ffn, hid, V, sp),
                                        _sparse_linear(gen, hid, ffn, V, sp)).cuda().half().eval()
        s["x"] = _half(gen, (hid, case["batch"] * case["seq"]))
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    V = case["V"]
    if kind == "spmm":
        return sspmm_amd.spmm(s["rows"], s["offsets"], s["cols"], s["values"], s["B"], V, out_dtype=s["out"])
    if kind == "bspmm":
        return sspmm_amd.bspmm(s["rows"], s["offsets"], s["cols"], s["values"], s["B"], V, out_dtype=s["out"])
    if kind == "plan":
        return sspmm_amd.spmm(None, s["offsets"], s["cols"], s["values"], s["B"], V, out_dtype=s["out"], plan=s["plan"])
    if kind == "svc":
        ptr, col, val = s["csr"]
        if case["reorder"]:
            perm = sspmm_amd.minhash_order(ptr, col, case["M"])
            return [perm] + list(sspmm_amd.permute_csr(ptr, col, val, perm))
        r = sspmm_amd.svc(ptr, col, val, case["M"], case["K"], V, order=case["order"])
        return [r.vec_row_ptr, r.vec_col, r.vec_val]
    if kind == "svc_stack":
        b = sspmm_amd.svc_batched(s["rows"], max(k for _, k in STACK_SHAPES), s["ptr"], s["col"], s["val"], V,
                                  order=case["order"])
        return [[r.vec_row_ptr, r.vec_col, r.vec_val] for r in (b.matrix(i) for i in range(len(b)))]
    if kind == "attention":
        scale = case["dim"] ** -0.5
        if case["one_call"]:
            return sparse_attention(s["rows"], s["offsets"], s["cols"], s["q"], s["k"], s["v"], scale, V)
        w = sspmm_amd.bsddmm(s["rows"], s["offsets"], s["cols"], s["q"], s["k"], V)
        p = sspmm_amd.bcsr_softmax(s["rows"], s["offsets"], w, scale, V, case["heads"])
        return [w, p, sspmm_amd.bspmm(s["rows"], s["offsets"], s["cols"], p, s["v"], V)]
    with torch.no_grad():
        if kind == "model":
            return s["model"](s["tokens"])
        return s["layer"](s["x"], case["batch"], case["seq"])


# ---- what a pass cannot do without -----------------------------------------------------------------------------------

def _pattern_work(m_vec, K, V, sparsity):
    """(stored vectors, bytes of the pattern without values)"""
    nvec = m_vec * max(1, int(round((1.0 - sparsity) * K)))
    return nvec, 4 * nvec + 4 * (m_vec + 1)


def _stack_matrices(count):
    for i in range(count):
        M, K = STACK_SHAPES[i % 3]
        yield M, K, 1.0 - STACK_SPARSITIES[(i // 3) % 6]


def work(case):
    kind, V = case["kind"], case["V"]
    ob = 4 if case.get("out") == "f32" else 2
    if kind in ("spmm", "bspmm"):
        M, K, N, b = case["M"], case["K"], case["N"], case.get("batch", 1)
        nvec, pattern = _pattern_work(M // V, K, V, case["sparsity"])
        return {"bytes": pattern + b * (2 * nvec * V + 2 * K * N + ob * M * N), "flops": 2 * nvec * V * N * b}
    if kind == "plan":
        M, K, N = case["M"], case["K"], case["N"]
        nnz = M * min(case["mean"], K)
        # merged vectors: few rows of so sparse a matrix share a column
        return {"bytes": 4 * nnz + 4 * (M // V) + 2 * nnz * V + 2 * K * N + ob * M * N, "flops": 2 * nnz * N}
    if kind == "svc":
        nnz = case["M"] * min(case["mean"], case["K"])
        if case["reorder"]:
            return {"bytes": 2 * (6 * nnz + 4 * case["M"]) + 4 * case["M"], "flops": 0}
        return {"bytes": 4 * case["M"] + 6 * nnz + 4 * (case["M"] // V) + (4 + 2 * V) * nnz, "flops": 0}
    if kind == "svc_stack":
        total = 0
        for M, K, density in _stack_matrices(case["count"]):
            nnz = int(M * K * density)
            nvec = int(M // V * K * (1.0 - (1.0 - density) ** V))
            total += 4 * M + 6 * nnz + 4 * (M // V) + (4 + 2 * V) * nvec
        return {"bytes": total, "flops": 0}
    if kind == "attention":
        b, seq, dim = case["heads"], case["seq"], case["dim"]
        nvec, pattern = _pattern_work(seq // V, seq, V, case["sparsity"])
        scores = 0 if case["one_call"] else 4 * 2 * nvec * V    # scores and probabilities, written and read
        return {"bytes": pattern + b * (4 * 2 * seq * dim + scores), "flops": 2 * 2 * nvec * V * dim * b}
    if kind == "model":
        seq, e, mlp, T = case["seq"], case["embed"], case["mlp"], case["batch"] * case["seq"]
        nvec, pattern = _pattern_work(seq // V, seq, V, case["sparsity"])
        weights = 4 * e * e + 2 * e * mlp
        # a block's activations pass through memory once each way, its weights and its mask are read once
        return {"bytes": 4 * (2 * 2 * T * e + 2 * weights + pattern) + 2 * T * (e + mlp) + 2 * e * mlp + 8 * T,
                "flops": 4 * (2 * T * weights + 4 * nvec * V * e * case["batch"]) + 2 * T * e * mlp}
    hid, ffn, T = case["hidden"], case["ffn"], case["batch"] * case["seq"]
    nvec = sum(_pattern_work(o // V, i, V, case["sparsity"])[0] for o, i in 4 * [(hid, hid)] + [(ffn, hid), (hid, ffn)])
    return {"bytes": nvec * (2 * V + 4) + 2 * 2 * T * hid,
            "flops": 2 * nvec * V * T + 4 * case["seq"] * T * hid}


def tolerance(case):
    kind = case["kind"]
    if kind in ("svc", "svc_stack"):
        return "exact"
    # four times what was measured against float64: 4e-7 at most with fp32 results, 2.1e-4 (the rounding alone) with fp16
    # ones; 5.3e-4 for the attention operators and up to 5.8e-4 for model and layer, against float64 and float32
    if kind in ("spmm", "bspmm", "plan"):
        return {"rel": 2e-6} if case["out"] == "f32" else {"rel": 8e-4}
    return {"rel": 2e-3}
