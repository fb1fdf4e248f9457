"""The SVC of a stack of matrices (svc_count_batched / svc_fill_batched through the C ABI): every matrix of the stack
must come out as it does on its own, bit for bit: against the CPU oracle, the files the reference wrote and the
single-matrix entry points."""
import glob
import os

import numpy as np
import pytest
import torch

import sspmm_amd
from sspmm_amd import formats, synth
from gpu_util import dev

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def _random_csr(rng, M, K, max_len):
    lens = rng.integers(0, min(K, max_len) + 1, M)
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    cols = np.concatenate([np.sort(rng.permutation(K)[:n]) for n in lens] + [np.zeros(0, np.int64)]).astype(np.int32)
    vals = rng.standard_normal(cols.size).astype(np.float16)
    return synth.Csr(M, K, ptr, cols, vals)


def _run(mats, V, order="cpython", with_values=True):
    host = [(c.M, c.K, c.row_ptr, c.col_ind, c.values if with_values else None) for c in mats]
    mat_rows, K_max, rp, ci, cv = sspmm_amd.stack_csr(host)
    print("stack of %d matrices, rows %d, nnz %d, V=%d %s" % (len(mats), mat_rows[-1], ci.size, V, order), flush=True)
    batch = sspmm_amd.svc_batched(mat_rows, K_max, dev(rp), dev(ci), None if cv is None else dev(cv), V, order=order)
    torch.cuda.synchronize()
    return batch


@pytest.mark.parametrize("V", [8, 16])
@pytest.mark.parametrize("order", ["cpython", "sorted"])
def test_stack_equals_every_matrix_on_its_own(oracle, built_library, V, order):
    """Row counts that are and are not multiples of V (a short last group per matrix), an empty matrix, a matrix of
    empty rows, widths from 8 to 5000 columns, groups in every LDS size class."""
    rng = np.random.default_rng(40 + V)
    shapes = [(64, 512, 80), (13, 33, 20), (1, 8, 8), (0, 100, 0), (40, 5000, 900), (17, 700, 0), (128, 2048, 400),
              (5, 4000, 4000), (24, 512, 512)]
    mats = [_random_csr(rng, M, K, mx) for M, K, mx in shapes]
    batch = _run(mats, V, order)
    host = batch.to_host()
    assert len(host) == len(mats)
    for i, (c, (vrp, vcol, vval)) in enumerate(zip(mats, host)):
        wrp, wcol, wval = oracle.svc(c.M, c.K, V, c.row_ptr, c.col_ind, c.values, order=order)
        assert np.array_equal(vrp, wrp), i
        assert np.array_equal(vcol, wcol), i
        assert np.array_equal(vval.view(np.uint16), wval.view(np.uint16)), i
        view = batch.matrix(i)   # the device views agree with the host copies
        assert np.array_equal(view.vec_row_ptr.cpu().numpy(), wrp) and np.array_equal(view.vec_col.cpu().numpy(), wcol)
        assert view.num_vec == wcol.size


@pytest.mark.parametrize("V", [8, 16])
def test_stack_of_the_reference_written_files(built_library, V):
    """All golden `.smtx` inputs in one stack: each comes back as the CVSE file the reference wrote for it."""
    names = sorted(p for p in glob.glob(os.path.join(GOLDEN, "*.smtx")) if ".v" not in os.path.basename(p))
    mats, meta = [], []
    for p in names:
        M, K, nnz, row_ptr, col_ind = formats.read_smtx(p)
        mats.append(synth.Csr(M, K, row_ptr, col_ind, None))
        meta.append((p, K, nnz))
    batch = _run(mats, V, with_values=False)
    for (p, K, nnz), (vrp, vcol, _v) in zip(meta, batch.to_host()):
        with open(p.replace(".smtx", ".v%d.smtx" % V)) as f:
            assert formats.cvse_text(vrp.size - 1, K, nnz, vrp, vcol) == f.read(), p


def test_stack_matches_the_single_matrix_entry_points(built_library):
    """96 matrices of the dataset's shapes in one call against 96 calls of svc()."""
    rng = np.random.default_rng(7)
    mats = []
    for i in range(24):
        M, K = [(512, 512), (2048, 512), (512, 2048)][i % 3]
        s = [0.5, 0.7, 0.9, 0.98][i % 4]
        mask = rng.random((M, K)) >= s
        ptr = np.concatenate([[0], np.cumsum(mask.sum(axis=1))]).astype(np.int32)
        mats.append(synth.Csr(M, K, ptr, np.nonzero(mask)[1].astype(np.int32), None))
    batch = _run(mats, 8, with_values=False)
    for c, (vrp, vcol, _v) in zip(mats, batch.to_host()):
        r = sspmm_amd.svc(dev(c.row_ptr), dev(c.col_ind), None, c.M, c.K, 8)
        assert np.array_equal(vrp, r.vec_row_ptr.cpu().numpy())
        assert np.array_equal(vcol, r.vec_col.cpu().numpy())


def test_group_count_the_device_arrives_at(built_library):
    """mat_groups[count] is the device's own count of the groups; a caller that passes another count gets a wrong
    answer it can detect, not a write outside its arrays."""
    from sspmm_amd import _lib
    L = _lib.lib()
    V = 8
    rng = np.random.default_rng(9)
    mats = [_random_csr(rng, M, 64, 10) for M in (9, 16, 3)]
    mat_rows, K_max, rp, ci, cv = sspmm_amd.stack_csr([(c.M, c.K, c.row_ptr, c.col_ind, None) for c in mats])
    groups = 2 + 2 + 1
    d_rows, d_rp, d_ci = dev(mat_rows), dev(rp), dev(ci)
    ws = torch.empty(L.svc_batched_workspace_bytes(3, int(mat_rows[-1]), ci.size, V), dtype=torch.uint8, device="cuda")
    d_groups = torch.full((4,), -1, dtype=torch.int32, device="cuda")
    vrp = torch.full((groups + 1 + 4,), -7, dtype=torch.int32, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    assert L.svc_count_batched(3, groups, d_rows.data_ptr(), int(mat_rows[-1]), K_max, V, d_rp.data_ptr(), d_ci.data_ptr(),
                               ci.size, 0, d_groups.data_ptr(), vrp.data_ptr(), ws.data_ptr(), s) == 0
    torch.cuda.synchronize()
    assert d_groups.cpu().tolist() == [0, 2, 4, 5]
    assert torch.all(vrp[groups + 1:] == -7)
    # rejected before anything is launched: more groups than the stack can have, no table
    assert L.svc_count_batched(3, 40, d_rows.data_ptr(), int(mat_rows[-1]), K_max, V, d_rp.data_ptr(), d_ci.data_ptr(),
                               ci.size, 0, d_groups.data_ptr(), vrp.data_ptr(), ws.data_ptr(), s) == 1
    assert L.svc_count_batched(3, groups, None, int(mat_rows[-1]), K_max, V, d_rp.data_ptr(), d_ci.data_ptr(),
                               ci.size, 0, d_groups.data_ptr(), vrp.data_ptr(), ws.data_ptr(), s) == 1


def test_converter_takes_the_files_through_one_stack(built_library, tmp_path):
    from sspmm_amd import rowmerge
    names = sorted(os.path.basename(p) for p in glob.glob(os.path.join(GOLDEN, "*.smtx")) if ".v" not in os.path.basename(p))
    stats = rowmerge.convert_files([os.path.join(GOLDEN, n) for n in names], [str(tmp_path / n) for n in names], 8)
    assert len(stats) == len(names)
    for n in names:
        assert (tmp_path / n).read_bytes() == open(os.path.join(GOLDEN, n.replace(".smtx", ".v8.smtx")), "rb").read()


def test_extents_follow_the_row_pointer():
    """The extents that matrix() hands out are those of the row pointer as it is now (host tensors: no launches)."""
    from sspmm_amd.svc import SvcBatch
    ptr = torch.tensor([0, 2, 5, 5, 9], dtype=torch.int32)
    groups = np.array([0, 2, 2, 4])
    b = SvcBatch(8, np.array([16, 0, 16]), None, groups, ptr, torch.arange(9, dtype=torch.int32), None,
                 torch.from_numpy(groups.astype(np.int32)))
    sizes = lambda: [b.matrix(i).num_vec for i in range(3)]  # noqa: E731
    assert sizes() == [5, 0, 4] and b.matrix(2).vec_row_ptr.tolist() == [0, 0, 4]
    ptr[2:4] = 3
    assert sizes() == [3, 0, 6]
    b.vec_row_ptr = torch.tensor([0, 1, 1, 1, 8], dtype=torch.int32)
    assert sizes() == [1, 0, 7] and b.matrix(2).vec_col.tolist() == list(range(1, 8))
    with torch.inference_mode():
        b.vec_row_ptr = torch.tensor([0, 1, 1, 1, 2], dtype=torch.int32)
        assert sizes() == [1, 0, 1]
        b.vec_row_ptr[4] = 6
        assert sizes() == [1, 0, 5]
    for i in (3, -1):
        with pytest.raises(IndexError):
            b.matrix(i)


def test_a_stack_pickled_before_it_had_a_list_of_its_first_groups():
    """The state that a batch had when it kept the array of first groups and the row pointer alone (host tensors: no launches)."""
    import pickle
    from sspmm_amd.svc import SvcBatch
    groups = np.array([0, 2, 2, 4])
    b = SvcBatch(8, np.array([16, 0, 16]), None, groups, torch.tensor([0, 2, 5, 5, 9], dtype=torch.int32), torch.arange(9, dtype=torch.int32),
                 None, torch.from_numpy(groups.astype(np.int32)))
    b.__dict__.pop("_first")
    b._row_ptr.__dict__.pop("ahead", None)
    old = pickle.loads(pickle.dumps(b))
    assert [old.matrix(i).num_vec for i in range(3)] == [5, 0, 4] and [t[0].tolist() for t in old.to_host()] == [[0, 2, 5], [0], [0, 0, 4]]


@pytest.mark.parametrize("rows", [[16], [0, 0], [0, 24, 0, 0, 7, 300, 0], [8] * 70])
def test_row_pointers_of_a_stack_are_each_matrix_s_own(built_library, rows):
    """Empty matrices at either end and in a row, more matrices than a wave has lanes; a second call and one on another
    stream get arrays of their own, and what a caller writes stays with that caller."""
    rng = np.random.default_rng(len(rows))
    mats = []
    for M in rows:
        ptr = np.concatenate([[0], np.cumsum(rng.integers(0, 9, M))]).astype(np.int32)
        mats.append((M, 512, ptr, np.concatenate([np.sort(rng.choice(512, n, replace=False)) for n in np.diff(ptr)] + [np.zeros(0)])
                     .astype(np.int32), None))
    at, K, ptr, col, _ = sspmm_amd.stack_csr(mats)
    batch = sspmm_amd.svc_batched(at, K, torch.from_numpy(ptr).cuda(), torch.from_numpy(col).cuda(), None, 8)
    want = [p for p, _, _ in batch.to_host()]
    first = [batch.matrix(i).vec_row_ptr for i in range(len(rows))]
    for got, w in zip(first, want):
        assert got.cpu().tolist() == w.tolist()
        got.fill_(-1)
    with torch.cuda.stream(torch.cuda.Stream()):
        other = [batch.matrix(i).vec_row_ptr.cpu().tolist() for i in range(len(rows))]
    assert other == [w.tolist() for w in want] == [batch.matrix(i).vec_row_ptr.cpu().tolist() for i in range(len(rows))]


def _stacked(rng, rows, V=8):
    """(batch, its row pointer as a list, first group of every matrix) of random matrices of these row counts."""
    mats = []
    for M in rows:
        ptr = np.concatenate([[0], np.cumsum(rng.integers(1, 9, M))]).astype(np.int32)
        mats.append((M, 512, ptr, np.concatenate([np.sort(rng.choice(512, n, replace=False)) for n in np.diff(ptr)]).astype(np.int32), None))
    at, K, ptr, col, _ = sspmm_amd.stack_csr(mats)
    batch = sspmm_amd.svc_batched(at, K, torch.from_numpy(ptr).cuda(), torch.from_numpy(col).cuda(), None, V)
    want = np.concatenate([[0], np.cumsum(np.concatenate([np.diff(p) for p, _, _ in batch.to_host()]))]).tolist()
    return batch, want, np.concatenate([[0], np.cumsum([(M + V - 1) // V for M in rows])]).tolist()


@pytest.mark.parametrize("how", ["deep copy", "pickle", "other stream first", "dropped"])
def test_extents_on_their_way_to_the_host_stay_with_their_batch(built_library, how):
    """What svc_batched sends ahead for matrix() is not part of a copy, serves its own stream only, and may be dropped unread."""
    import copy
    import io
    batch, ptr, groups = _stacked(np.random.default_rng(9), [40, 3, 8, 100])
    if how == "deep copy":
        _check_matrices(copy.deepcopy(batch), ptr, groups, range(4))
    elif how == "pickle":
        f = io.BytesIO()
        torch.save(batch, f)
        f.seek(0)
        _check_matrices(torch.load(f, weights_only=False), ptr, groups, range(4))
    elif how == "other stream first":
        torch.cuda.synchronize()
        with torch.cuda.stream(torch.cuda.Stream()):
            _check_matrices(batch, ptr, groups, range(4))
    else:
        for seed in range(20):
            _stacked(np.random.default_rng(seed), [8] * (seed + 1))
    _check_matrices(batch, ptr, groups, range(4))


def test_callers_who_take_no_matrix_do_not_pay_for_them(built_library, monkeypatch):
    """The matrices' own row pointers are made for matrix() alone; to_host() has the row pointer that svc_batched sent, as long as
    nobody else can have written it, before and after matrix()."""
    import sys
    svc_mod, made = sys.modules["sspmm_amd.svc"], []
    split = svc_mod._split_row_ptr
    monkeypatch.setattr(svc_mod, "_split_row_ptr", lambda *a: (made.append(1), split(*a))[1])
    batch, ptr, groups = _stacked(np.random.default_rng(11), [40, 3, 8, 100])
    rebased = lambda p: [[x - p[a] for x in p[a:b + 1]] for a, b in zip(groups, groups[1:])]  # noqa: E731
    got = lambda: [t[0].tolist() for t in batch.to_host()]  # noqa: E731
    assert got() == rebased(ptr) and not made
    first = batch.to_host()[0][0]
    first[:] = -1                                   # (what is handed out is the caller's)
    assert got() == rebased(ptr) and not made
    _check_matrices(batch, ptr, groups, range(4))
    assert len(made) == 1 and got() == rebased(ptr)
    other = [p - (i % 3 if 0 < i else 0) for i, p in enumerate(ptr)]
    batch.vec_row_ptr.copy_(torch.tensor(other, dtype=torch.int32))
    assert got() == rebased(other) and len(made) == 1
    batch, ptr, groups = _stacked(np.random.default_rng(12), [40, 8])
    whole = batch.vec_row_ptr                       # (before anything else was asked for)
    whole[1:] += 1
    assert got() == rebased([0] + [p + 1 for p in ptr[1:]]) and len(made) == 1


@pytest.mark.parametrize("ahead", [4096, 8, 2])
def test_extents_whatever_went_ahead(built_library, monkeypatch, ahead):
    """The row pointer, the matrices' extents or nothing on its way to the host: twenty groups of four matrices against what may be sent."""
    import sys
    monkeypatch.setattr(sys.modules["sspmm_amd.svc"], "_AHEAD", ahead)
    batch, ptr, groups = _stacked(np.random.default_rng(13), [40, 3, 8, 100])
    sent = batch._row_ptr.ahead
    assert (sent is None) == (ahead == 2) and (sent is None or sent.whole == (ahead == 4096))
    _check_matrices(batch, ptr, groups, range(4))
    assert [t[0].tolist() for t in batch.to_host()] == [[x - ptr[a] for x in ptr[a:b + 1]] for a, b in zip(groups, groups[1:])]


def test_stacks_where_the_gpu_is_the_default_device(built_library):
    """(what goes to the host lives there)"""
    with torch.device("cuda"):
        batch, ptr, groups = _stacked(np.random.default_rng(10), [40, 3, 8, 100])
        _check_matrices(batch, ptr, groups, range(4))


def _check_matrices(batch, ptr, groups, matrices):
    for i in matrices:
        own = ptr[groups[i]:groups[i + 1] + 1]
        r = batch.matrix(i)
        assert r.num_vec == own[-1] - own[0], i
        assert r.vec_row_ptr.cpu().tolist() == [p - own[0] for p in own], i
        assert torch.equal(r.vec_col, batch.vec_col[own[0]:own[-1]]), i


@pytest.mark.parametrize("how", ["in place", "data", "raw pointer", "graph", "shallow copy", "int64", "strided", "host", "inference"])
@pytest.mark.parametrize("taken", [0, 2, 4])
def test_matrices_follow_a_row_pointer_on_the_device(built_library, how, taken):
    """Extents and row pointers are those of vec_row_ptr as it is, after a caller wrote or replaced it, whether or not some
    matrices had been taken before.  (Written: entries kept in order and inside vec_col, as a merge leaves them.)"""
    import copy
    from sspmm_amd import _lib
    batch, ptr, groups = _stacked(np.random.default_rng(taken), [40, 8, 100, 33])
    assert batch.matrix(1).num_vec == ptr[groups[2]] - ptr[groups[1]]
    _check_matrices(batch, ptr, groups, range(taken))
    other = [p - (i % 3 if 0 < i else 0) for i, p in enumerate(ptr)]
    there = torch.tensor(other, dtype=torch.int32, device="cuda")
    if how == "in place":
        batch.vec_row_ptr.copy_(there)
    elif how == "data":
        batch.vec_row_ptr.data.copy_(there)
    elif how == "raw pointer":  # (this entry of the library writes groups + 1 entries of one matrix)
        one, bounds = torch.tensor([0, groups[-1]], dtype=torch.int32, device="cuda"), torch.empty(2, dtype=torch.int32, device="cuda")
        assert _lib.lib().svc_split_row_ptr(1, groups[-1], one.data_ptr(), there.data_ptr(), batch.vec_row_ptr.data_ptr(), bounds.data_ptr(),
                                            torch.cuda.current_stream().cuda_stream) == 0
    elif how == "graph":
        whole, graph = batch.vec_row_ptr, torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            whole.copy_(there)
        for _ in range(2):
            _check_matrices(batch, ptr, groups, range(4))
        graph.replay()
    elif how == "shallow copy":
        copy.copy(batch).vec_row_ptr.copy_(there)
    elif how == "int64":
        batch.vec_row_ptr = there.long()
    elif how == "strided":
        batch.vec_row_ptr = torch.stack([there, there + 1], dim=1)[:, 0]
    elif how == "host":
        batch.vec_row_ptr = there.cpu()
    else:
        with torch.inference_mode():
            batch.vec_row_ptr = there.clone()
            _check_matrices(batch, other, groups, range(4))
    _check_matrices(batch, other, groups, range(4))
    _check_matrices(batch, other, groups, range(4))


def test_a_shorter_row_pointer_is_not_read_past_its_end(built_library):
    batch, ptr, groups = _stacked(np.random.default_rng(5), [40, 8, 100, 33])
    batch.vec_row_ptr = batch.vec_row_ptr[:groups[2] + 1].clone()
    _check_matrices(batch, ptr, groups, [0, 1])


def test_row_pointers_taken_in_inference_mode_stay_there(built_library):
    """A row pointer is an inference tensor only for the caller who took it in inference mode."""
    batch, ptr, groups = _stacked(np.random.default_rng(6), [40, 8, 100])
    with torch.inference_mode():
        assert batch.matrix(0).vec_row_ptr.is_inference()
    got = batch.matrix(1).vec_row_ptr
    assert not got.is_inference()
    got.add_(1)
    _check_matrices(batch, ptr, groups, range(3))


@pytest.mark.parametrize("mat_groups", [[0, 3, 7, 5], [0, 40, 50, 60], [-4, 2, 3, 5], [9, 9, 9, 9]])
def test_split_of_a_miscounted_stack_stays_inside_its_arrays(built_library, mat_groups):
    """svc_split_row_ptr with first groups beyond `groups` or out of order, as a stack with a wrong group count leaves
    them: entries come out of the row pointer's own groups + 1 (here all below 100), and nothing else is written."""
    from sspmm_amd import _lib
    groups, count = 5, 3
    buf = torch.full((64 + groups + 1 + 64,), 10 ** 6, dtype=torch.int32, device="cuda")
    whole = buf[64:64 + groups + 1]
    whole.copy_(torch.tensor([0, 3, 9, 9, 20, 31], device="cuda"))
    out = torch.full((groups + count + 8,), -7, dtype=torch.int32, device="cuda")
    bounds = torch.full((count + 1 + 8,), -7, dtype=torch.int32, device="cuda")
    at = dev(np.array(mat_groups, np.int32))
    assert _lib.lib().svc_split_row_ptr(count, groups, at.data_ptr(), whole.data_ptr(), out.data_ptr(), bounds.data_ptr(),
                                        torch.cuda.current_stream().cuda_stream) == 0
    out, bounds = out.cpu(), bounds.cpu()
    assert (out[:groups + count].abs() < 100).all() and (bounds[:count + 1].abs() < 100).all()
    assert (out[groups + count:] == -7).all() and (bounds[count + 1:] == -7).all()


def test_split_rejects_what_it_cannot_do(built_library):
    """(valid device pointers throughout: nothing is launched for a rejected call)"""
    from sspmm_amd import _lib
    L, p = _lib.lib(), torch.zeros(64, dtype=torch.int32, device="cuda").data_ptr()
    assert L.svc_split_row_ptr(-1, 4, p, p, p, p, None) == 1 and L.svc_split_row_ptr(1, -1, p, p, p, p, None) == 1
    assert L.svc_split_row_ptr(2 ** 30, 2 ** 30, p, p, p, p, None) == 1
    for args in ((None, p, p, p), (p, None, p, p), (p, p, None, p), (p, p, p, None)):
        assert L.svc_split_row_ptr(1, 4, *args, None) == 1
    assert L.svc_split_row_ptr(0, 0, None, None, None, None, None) == 0


@pytest.mark.parametrize("most", [1, 64, 65, 300])
def test_group_table_of_more_matrices_than_a_workgroup_has_threads(built_library, most):
    """2100 matrices (three tiles of 1024 in the launch that makes the table) of 0 up to `most` groups, few of them large: either
    way in which that launch writes a tile's groups."""
    V = 8
    rng = np.random.default_rng(most)
    per = rng.integers(0, 3, 2100)
    per[rng.choice(2100, 3, replace=False)] = most
    rows = np.maximum(per * V - rng.integers(0, V, 2100) * (per > 0), 0)
    at = np.concatenate([[0], np.cumsum(rows)]).astype(np.int64)
    lens = rng.integers(0, 4, at[-1])
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(64, n, replace=False)) for n in lens]).astype(np.int32)
    batch = sspmm_amd.svc_batched(at, 64, dev(ptr), dev(col), None, V, order="sorted")
    got = batch.vec_row_ptr.cpu().numpy()
    starts = np.concatenate([np.arange(a, b, V) for a, b in zip(at[:-1], at[1:])] + [at[-1:]])
    ends = np.concatenate([np.minimum(np.arange(a, b, V) + V, b) for a, b in zip(at[:-1], at[1:])])
    want = np.concatenate([[0], np.cumsum([np.unique(col[ptr[a]:ptr[b]]).size for a, b in zip(starts, ends)])])
    assert np.array_equal(got, want)
