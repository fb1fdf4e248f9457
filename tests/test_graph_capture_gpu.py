"""The entry points enqueue kernels and events only: a caller may record them into a HIP graph.  Every replay is
checked against the eager result, with eager work and synchronisations between the replays."""
import numpy as np
import pytest
import torch

import sspmm_amd
from sspmm_amd import _lib, synth
from gpu_util import dev

pytestmark = pytest.mark.gpu


def _between_replays():
    torch.ones(4096, device="cuda").sum().item()  # eager work and a synchronisation of the program's own


def test_batched_spmm_in_a_graph(built_library):
    L = _lib.lib()
    V, K, N, batch = 8, 512, 256, 16
    vs = synth.vector_sparse(2048, K, V, 0.9, seed=2, std=0.02)
    ro, ci = dev(vs.row_offsets), dev(vs.col_idx)
    g = torch.Generator(device="cuda").manual_seed(5)
    vals = (torch.randn(batch, vs.col_idx.size * V, generator=g, device="cuda") * 0.02).half()
    B = torch.randn(batch, K, N, generator=g, device="cuda").half()
    C = torch.zeros(batch, vs.m_vec * V, N, device="cuda")

    def launch(stream):
        rc = L.sspmm_batched_f16_f32(batch, vs.m_vec, V, N, K, None, ro.data_ptr(), ci.data_ptr(), vals.data_ptr(),
                                     vs.col_idx.size * V, B.data_ptr(), K * N, C.data_ptr(), vs.m_vec * V * N, stream)
        assert rc == 0, rc

    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        launch(s.cuda_stream)
    torch.cuda.synchronize()
    want = C.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        launch(torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        C.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, want)
        _between_replays()


def test_svc_in_a_graph(built_library):
    """svc_count + svc_fill with their fork / join of the helper stream, recorded once and replayed."""
    L = _lib.lib()
    V = 8
    csr = synth.zipf_csr(4096, 4096, seed=4)
    rp, cc, cv = dev(csr.row_ptr), dev(csr.col_ind), dev(csr.values)
    eager = sspmm_amd.svc(rp, cc, cv, csr.M, csr.K, V)
    nnz = csr.col_ind.size
    ws = torch.empty(L.svc_workspace_bytes(csr.M, nnz, V), dtype=torch.uint8, device="cuda")
    vrp = torch.zeros(csr.M // V + 1, dtype=torch.int32, device="cuda")
    vcol = torch.zeros(eager.num_vec, dtype=torch.int32, device="cuda")
    vval = torch.zeros(eager.num_vec * V, dtype=torch.float16, device="cuda")

    def launch(stream):
        rc = L.svc_count(csr.M, csr.K, V, rp.data_ptr(), cc.data_ptr(), nnz, 0, vrp.data_ptr(), ws.data_ptr(), stream)
        assert rc == 0, rc
        rc = L.svc_fill(csr.M, csr.K, V, rp.data_ptr(), cc.data_ptr(), cv.data_ptr(), nnz, 0, vrp.data_ptr(),
                        ws.data_ptr(), vcol.data_ptr(), vval.data_ptr(), stream)
        assert rc == 0, rc

    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        launch(s.cuda_stream)  # creates the helper stream outside the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        launch(torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        vrp.zero_()
        vcol.zero_()
        vval.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(vrp, eager.vec_row_ptr) and torch.equal(vcol, eager.vec_col) and torch.equal(vval, eager.vec_val)
        _between_replays()


@pytest.mark.parametrize("batch,seq,one_launch", [(3, 333, False), (4, 320, True), (3, 347, True)])
def test_encoder_layer_in_a_graph(built_library, monkeypatch, batch, seq, one_launch):
    """The attention on any number of tokens, the norms on any number and all that follows the attention in one launch, recorded
    once and replayed on other activations."""
    from sspmm_amd import layers
    hidden, ffn, V = 128, 256, 8

    def sparse(o, i, seed):
        vs = synth.vector_sparse(o, i, V, 0.9, seed=seed, std=0.05)
        return layers.SparseLinear.from_cvse(i, V, dev(vs.row_offsets), dev(vs.col_idx), dev(vs.values))

    layer = layers.SparseEncoderLayer(hidden, 2, ffn, *(sparse(hidden, hidden, s) for s in range(4)), sparse(ffn, hidden, 5),
                                      sparse(hidden, ffn, 6)).cuda().half().eval()
    launches, tail = [], layers.encoder_tail
    monkeypatch.setattr(layers, "encoder_tail", lambda *a: (launches.append(1), tail(*a))[1])
    monkeypatch.setattr(layers, "TAIL_TOKENS", 1 if one_launch else 1 << 30)
    g = torch.Generator("cuda").manual_seed(seq)
    xs = [torch.randn(hidden, batch * seq, device="cuda", generator=g).half() for _ in range(3)]
    x, s = xs[0].clone(), torch.cuda.Stream()
    with torch.no_grad():
        wants = [layer(t, batch, seq).clone() for t in xs]
        assert len(launches) == (3 if one_launch else 0)
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            layer(x, batch, seq)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            out = layer(x, batch, seq)
    for t, want in zip(xs + xs[:1], wants + wants[:1]):
        x.copy_(t)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        _between_replays()


@pytest.mark.parametrize("mlp", [256, 512])
def test_encoder_in_a_graph(built_library, mlp):
    """The lookup and its assertion, the folded layers (512) and the two layers one after the other (256), recorded once and replayed on other
    tokens and other weights, which every pass packs and multiplies anew."""
    from sspmm_amd.attention import SparseAttentionEncoder
    model = SparseAttentionEncoder(50, 256, 8, 0.8, 96, mlp, 64, vec_length=8, layers=2, seed=2).cuda().half().eval()
    g = torch.Generator("cuda").manual_seed(mlp)
    sets = [(torch.randint(0, 50, (3, 96), device="cuda", generator=g), torch.randn(256, mlp, device="cuda", generator=g).half() * 0.05) for _ in range(3)]
    tokens, s, weight = sets[0][0].clone(), torch.cuda.Stream(), model.blocks[1].linear2.weight
    with torch.no_grad():
        wants = []
        for t, w in sets:
            weight.copy_(w)
            wants.append(model(t).clone())
        assert not torch.equal(wants[0], wants[1])
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            model(tokens)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            out = model(tokens)
        for (t, w), want in zip(sets + sets[:1], wants + wants[:1]):
            tokens.copy_(t)
            weight.copy_(w)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
            _between_replays()
