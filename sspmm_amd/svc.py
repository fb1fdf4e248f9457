"""Sparse Vector Compression (RowMerge) on the GPU: CSR -> CVSE.

Host-side mirror of the reference's `CVSE(ROW, COL, NNZ, colInd_list_array, vec_len)`
(reference RowMerge/sparse_matrix_format.py:94-123) over device tensors; the merge runs in the
HIP kernels behind svc_count / svc_fill of the C ABI.
"""
import collections

import torch

from . import _lib

SvcResult = collections.namedtuple("SvcResult", ["vec_row_ptr", "vec_col", "vec_val", "num_vec"])

_ORDERS = {"cpython": 0, "sorted": 1}


def svc(row_ptr, col_ind, csr_val, M, K, V, order="cpython", exact_size=True):
    """Merge every V consecutive rows of a CSR matrix into column vectors.

    row_ptr[M+1], col_ind[nnz]: int32 GPU tensors; csr_val: fp16 GPU tensor or None.
    order="cpython" gives exactly the column order the reference's RowMerge writes;
    order="sorted" gives ascending columns.
    Returns SvcResult(vec_row_ptr[int32 m_vec+1], vec_col[int32 nvec], vec_val[fp16 nvec*V] or None, nvec).

    exact_size=True reads nvec back from the device between the two phases (the call's one synchronisation) and
    returns arrays of exactly nvec vectors.  exact_size=False sizes them for the bound nvec <= nnz instead: the call
    then never waits for the device (both phases are queued on the current stream), num_vec is None, the vectors
    are the first vec_row_ptr[-1] entries of vec_col / vec_val and what lies behind them is unspecified.  The SpMM
    operators take such arrays as they are: they read the extent from vec_row_ptr on the device.
    """
    if order not in _ORDERS:
        raise ValueError("order must be 'cpython' or 'sorted'")
    if row_ptr.dtype != torch.int32 or col_ind.dtype != torch.int32:
        raise TypeError("row_ptr and col_ind must be int32")
    if csr_val is not None and csr_val.dtype != torch.float16:
        raise TypeError("csr_val must be float16")
    if not (row_ptr.is_cuda and col_ind.is_cuda):
        raise ValueError("row_ptr and col_ind must live on the GPU")
    if row_ptr.numel() != M + 1:
        raise ValueError("row_ptr must have M + 1 entries")
    L = _lib.lib()
    dev = row_ptr.device
    nnz = col_ind.numel()
    m_vec = (M + V - 1) // V
    with torch.cuda.device(dev):
        stream = torch.cuda.current_stream().cuda_stream
        ws = torch.empty(L.svc_workspace_bytes(M, nnz, V), dtype=torch.uint8, device=dev)
        # (svc_count writes every entry)
        vec_row_ptr = (torch.empty if M > 0 else torch.zeros)(m_vec + 1, dtype=torch.int32, device=dev)
        if M == 0:
            return SvcResult(vec_row_ptr, torch.empty(0, dtype=torch.int32, device=dev),
                             None if csr_val is None else torch.empty(0, dtype=torch.float16, device=dev), 0)
        _lib.check(L.svc_count(M, K, V, row_ptr.data_ptr(), col_ind.data_ptr(), nnz, _ORDERS[order],
                               vec_row_ptr.data_ptr(), ws.data_ptr(), stream), "svc_count")
        nvec = int(vec_row_ptr[-1].item()) if exact_size else None  # the one host read-back: sizes the outputs
        cap = nvec if exact_size else nnz
        vec_col = torch.empty(cap, dtype=torch.int32, device=dev)
        vec_val = None if csr_val is None else torch.empty(cap * V, dtype=torch.float16, device=dev)
        _lib.check(L.svc_fill(M, K, V, row_ptr.data_ptr(), col_ind.data_ptr(),
                              0 if csr_val is None else csr_val.data_ptr(), nnz, _ORDERS[order],
                              vec_row_ptr.data_ptr(), ws.data_ptr(), vec_col.data_ptr(),
                              0 if vec_val is None else vec_val.data_ptr(), stream), "svc_fill")
    return SvcResult(vec_row_ptr, vec_col, vec_val, nvec)


class _RowPointer:
    """The row pointer of a stack and what matrix() may keep of it: as long as it is `alone`, nobody but the batch (and
    its shallow copies, which share this object) has the tensor, so nobody can have written it."""

    ahead = None  # (for those that come out of an older pickle)

    def __init__(self, whole):
        self.whole, self.alone, self.split = whole, False, None

    def __getstate__(self):  # (deep copies and pickles: what is on its way to the host stays with the original)
        return dict(self.__dict__, ahead=None)


class _ReadBack:
    """Device values on their way to the host: what is queued behind this runs on, and wait() lasts until the copy is done.
    whole: they are the row pointer, not the matrices' extents alone."""

    def __init__(self, values, stream, whole):
        self.stream, self.whole = stream, whole
        self._host = torch.empty(values.shape, dtype=values.dtype, device="cpu", pin_memory=True)
        self._host.copy_(values, non_blocking=True)
        self._done = torch.cuda.Event()
        self._done.record()

    def wait(self):
        self._done.synchronize()
        return self._host.numpy()


# Values that svc_batched sends ahead to the host at most, 16 KB: the row pointer where it is that small, the matrices' extents (by a
# launch) where they are.  Larger copies go another way, of which the first ones keep the host waiting for 5 to 7 ms each (96 matrices
# of 12288 groups: four of the first 40 calls).
_AHEAD = 4096


def _split_row_ptr(count, groups, mat_groups, whole):
    """(all matrices' row pointers from zero, one after the other; the first vector of each and the end of the last)"""
    own, bounds = torch.empty(groups + 2 * count + 1, dtype=torch.int32, device=whole.device).split((groups + count, count + 1))
    _lib.check(_lib.call(_lib.lib().svc_split_row_ptr, whole.device, count, groups, mat_groups.data_ptr(), whole.data_ptr(),
                         own.data_ptr(), bounds.data_ptr()), "svc_split_row_ptr")
    return own, bounds


class SvcBatch:
    """The SVC of a stack of matrices (svc_batched): device arrays over the whole stack and views per matrix.

    vec_row_ptr[groups + 1] runs over all groups of all matrices; vec_col / vec_val hold the matrices' vectors one
    after the other and are sized for the bound nvec <= nnz (what lies behind vec_row_ptr[-1] vectors is
    unspecified).  `matrix(i)` returns matrix i's SvcResult as device views (its row pointer rebased to zero);
    `to_host()` brings everything over in one go and returns one (vec_row_ptr, vec_col, vec_val) numpy triple per
    matrix.  Both go by the row pointer as it is at the call, whoever wrote it and however: once `vec_row_ptr` has been
    read or assigned, matrix(i) reads its extent back every time."""

    def __init__(self, V, rows, cols, groups_of, vec_row_ptr, vec_col, vec_val, mat_groups=None):
        self.V, self.rows, self.cols = V, rows, cols
        self._groups = groups_of            # host: first group of every matrix, [count + 1]
        self._first = groups_of.tolist() if hasattr(groups_of, "tolist") else list(groups_of)
        self._mat_groups = mat_groups       # the same on the device, or None
        self._row_ptr = _RowPointer(vec_row_ptr)
        self.vec_col, self.vec_val = vec_col, vec_val

    def __setstate__(self, state):
        self.__dict__.update(state)
        self._first = [int(g) for g in self._groups]  # (older pickles have the array alone)

    @property
    def vec_row_ptr(self):
        p = self._row_ptr
        p.alone, p.split, p.ahead = False, None, None
        return p.whole

    @vec_row_ptr.setter
    def vec_row_ptr(self, whole):
        self._row_ptr = _RowPointer(whole)

    def __len__(self):
        return len(self.rows)

    def _taken(self, i, g0, g1):
        # (row pointer from zero, first vector, end) of matrix i, whose groups are g0 .. g1 - 1.  Of a row pointer that
        # svc_batched made and nobody else has seen, one launch rebases all matrices' and one read-back brings their
        # extents: twenty matrices one by one took a launch each (0.4 ms a pass, 0.3 ms like this), and with a
        # read-back each 1.2 ms.  svc_batched sends the row pointer, or the extents, to the host between its phases (`ahead`), so that the
        # host has the extents while the merge still runs and takes the next stack (twenty matrices, pass after pass 290-320 -> 195-235 us;
        # with the launch in svc_batched the same, but 14 us more for callers who never ask).  Any other one is a
        # caller's tensor (of any type, stride, length and device), written in ways that leave no trace on the host: those go one
        # by one.  A piece of the split is handed out once (what a caller writes into it is not in the next one), on the stream
        # that it was allocated on, and in the inference mode that it was made in.
        p = self._row_ptr
        whole = p.whole
        if not p.alone:
            ptr = whole[g0:g1 + 1]
            lo, hi = (int(x) for x in ptr[[0, -1]].tolist())
            return ptr - lo, lo, hi
        stream, split = _lib.stream_of(whole.device), p.split
        if split is None:
            ahead = p.ahead
            own, bounds = _split_row_ptr(len(self), self._first[-1], self._mat_groups, whole)
            if ahead is not None and ahead.stream == stream:
                bounds = ahead.wait()[self._groups] if ahead.whole else ahead.wait()
            bounds = bounds.tolist()
            sizes = [b - a + 1 for a, b in zip(self._first, self._first[1:])]
            p.split = split = (bounds, dict(enumerate(own.split(sizes))), stream, own.is_inference())
        bounds, own, own_stream, inference = split
        lo, hi = bounds[i], bounds[i + 1]
        mine = own.pop(i, None) if stream == own_stream and inference == torch.is_inference_mode_enabled() else None
        return (whole[g0:g1 + 1] - lo if mine is None else mine), lo, hi

    def matrix(self, i):
        g0, g1 = self._first[i], self._first[i + 1]
        if g1 < g0:
            raise IndexError("matrix %d of %d" % (i, len(self)))
        ptr, lo, hi = self._taken(i, g0, g1)   # (the views need their extent on the host)
        return SvcResult(ptr, self.vec_col[lo:hi], None if self.vec_val is None else self.vec_val[lo * self.V:hi * self.V], hi - lo)

    def to_host(self):
        p = self._row_ptr
        ahead = p.ahead  # (there only while it is what the device has)
        ptr = ahead.wait() if ahead is not None and ahead.whole and ahead.stream == _lib.stream_of(p.whole.device) else p.whole.cpu().numpy()
        n = int(ptr[-1])
        col = self.vec_col[:n].cpu().numpy()
        val = None if self.vec_val is None else self.vec_val[:n * self.V].cpu().numpy()
        out = []
        for i in range(len(self.rows)):
            p = ptr[self._groups[i]:self._groups[i + 1] + 1]
            lo, hi = int(p[0]), int(p[-1])
            out.append((p - p[0], col[lo:hi], None if val is None else val[lo * self.V:hi * self.V]))
        return out


def stack_csr(mats):
    """Stacks CSR matrices along the rows on the host.  mats: sequence of (M, K, row_ptr, col_ind, values or None)
    numpy arrays.  Returns (mat_rows[count + 1], K_max, row_ptr[M_total + 1], col_ind[nnz], values or None), int32 /
    fp16, the row pointer holding entry offsets into the stacked col_ind."""
    import numpy as np
    rows = np.zeros(len(mats) + 1, np.int64)
    ptrs, cols, vals, base = [np.zeros(1, np.int64)], [], [], 0
    with_values = len(mats) > 0 and all(m[4] is not None for m in mats)
    for i, (M, K, rp, ci, cv) in enumerate(mats):
        rp = np.asarray(rp, dtype=np.int64)
        if rp.size != M + 1 or rp[0] != 0 or rp[-1] != np.asarray(ci).size:
            raise ValueError("matrix %d: row_ptr does not describe col_ind" % i)
        rows[i + 1] = rows[i] + M
        ptrs.append(rp[1:] + base)
        cols.append(np.asarray(ci, dtype=np.int32))
        if with_values:
            vals.append(np.asarray(cv, dtype=np.float16))
        base += int(rp[-1])
    if base >= 1 << 28 or rows[-1] >= 1 << 31:
        raise ValueError("the stack is too large for one call: split it")
    cat = lambda parts, dt: np.concatenate(parts).astype(dt) if parts else np.zeros(0, dt)  # noqa: E731
    return (rows.astype(np.int32), max([m[1] for m in mats] + [0]), np.concatenate(ptrs).astype(np.int32),
            cat(cols, np.int32), cat(vals, np.float16) if with_values else None)


def svc_batched(mat_rows, K_max, row_ptr, col_ind, csr_val, V, order="cpython", cols=None):
    """The SVC of a stack of matrices in one chain of launches (svc_count_batched / svc_fill_batched of the C ABI).

    mat_rows: host int array [count + 1], first row of every matrix in the stack (as stack_csr returns it);
    row_ptr[M_total + 1], col_ind[nnz]: int32 GPU tensors of the stacked CSR; csr_val: fp16 GPU tensor or None.
    Nothing is waited for: both phases are queued on the current stream, between them a copy of the row pointer (or of the
    matrices' extents) to the host, for matrix().  Returns an SvcBatch."""
    import numpy as np
    if order not in _ORDERS:
        raise ValueError("order must be 'cpython' or 'sorted'")
    if row_ptr.dtype != torch.int32 or col_ind.dtype != torch.int32:
        raise TypeError("row_ptr and col_ind must be int32")
    if csr_val is not None and csr_val.dtype != torch.float16:
        raise TypeError("csr_val must be float16")
    if not (row_ptr.is_cuda and col_ind.is_cuda):
        raise ValueError("row_ptr and col_ind must live on the GPU")
    mat_rows = np.asarray(mat_rows, dtype=np.int64)
    count, M_total = mat_rows.size - 1, int(mat_rows[-1])
    rows = mat_rows[1:] - mat_rows[:-1]
    if count < 0 or row_ptr.numel() != M_total + 1 or (rows < 0).any():
        raise ValueError("mat_rows must be non-decreasing with mat_rows[-1] + 1 == len(row_ptr)")
    groups_of = np.zeros(count + 1, dtype=np.int64)
    np.cumsum((rows + V - 1) // V, out=groups_of[1:])
    groups = int(groups_of[-1])
    L = _lib.lib()
    dev = row_ptr.device
    nnz = col_ind.numel()
    with torch.cuda.device(dev):
        stream = _lib.stream_of(dev)
        d_rows, capturing, ahead = torch.from_numpy(mat_rows.astype(np.int32)), torch.cuda.is_current_stream_capturing(), None
        # (from pinned memory the copy waits for nothing; a stream that is captured refuses the other one, as it has to: a replay
        # would read the numbers from memory that has gone to others)
        d_rows = d_rows.to(dev) if capturing else d_rows.pin_memory().to(dev, non_blocking=True)
        d_groups = torch.empty(count + 1, dtype=torch.int32, device=dev)
        ws = torch.empty(L.svc_batched_workspace_bytes(count, M_total, nnz, V), dtype=torch.uint8, device=dev)
        vec_row_ptr = (torch.empty if groups > 0 else torch.zeros)(groups + 1, dtype=torch.int32, device=dev)
        vec_col = torch.empty(nnz, dtype=torch.int32, device=dev)
        vec_val = None if csr_val is None else torch.empty(nnz * V, dtype=torch.float16, device=dev)
        if groups > 0:
            _lib.check(L.svc_count_batched(count, groups, d_rows.data_ptr(), M_total, K_max, V, row_ptr.data_ptr(),
                                           col_ind.data_ptr(), nnz, _ORDERS[order], d_groups.data_ptr(),
                                           vec_row_ptr.data_ptr(), ws.data_ptr(), stream), "svc_count_batched")
            if not capturing and groups > 0 and min(groups, count) < _AHEAD:
                whole = groups < _AHEAD
                ahead = _ReadBack(vec_row_ptr if whole else _split_row_ptr(count, groups, d_groups, vec_row_ptr)[1], stream, whole)
            _lib.check(L.svc_fill_batched(count, groups, d_rows.data_ptr(), M_total, K_max, V, row_ptr.data_ptr(),
                                          col_ind.data_ptr(), 0 if csr_val is None else csr_val.data_ptr(), nnz,
                                          _ORDERS[order], vec_row_ptr.data_ptr(), ws.data_ptr(), vec_col.data_ptr(),
                                          0 if vec_val is None else vec_val.data_ptr(), stream), "svc_fill_batched")
    batch = SvcBatch(V, rows, cols, groups_of, vec_row_ptr, vec_col, vec_val, d_groups if groups > 0 else None)
    batch._row_ptr.alone, batch._row_ptr.ahead = groups > 0, ahead
    return batch
