"""Graphs in host memory: the check on the device against the host's (every
refusal with the same status and message), from the entry count where it
begins, and the upload in pieces against the same graph already on the GPU."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

LINE = 1 << 15  # entries from which the device checks


def ring(n, extra=0):
    """A ring of n vertices (2n entries), weighted."""
    v = np.arange(n, dtype=np.int64)
    adj = np.stack([(v - 1) % n, (v + 1) % n], 1).reshape(-1)
    xadj = 2 * np.arange(n + 1, dtype=np.int64)
    return xadj.astype(np.int32), adj.astype(np.int32), np.ones(2 * n, np.int32), np.ones(n, np.int32)


def call(gk, ctx, arrays, k=2, flags=0):
    """gk_partition and gk_graph_check of one raw CSR: (status, message) of each, and the partition."""
    x, a, w, v = arrays
    c = gk.Csr()
    c.n, c.nnz = len(x) - 1, len(a)
    p = [None if y is None else np.ascontiguousarray(y).ctypes.data_as(gk.I32P) for y in (x, a, w, v)]
    c.xadj, c.adjncy, c.adjwgt, c.vwgt = p
    L = gk.lib()
    prm = gk.Params()
    L.gk_params_default(ctypes.byref(prm), k)
    prm.flags |= flags
    part = np.full(c.n, -3, np.int32)
    got = L.gk_partition(ctx.handle, ctypes.byref(c), ctypes.byref(prm), part.ctypes.data_as(gk.I32P), None)
    got = (got, L.gk_last_error() if got else b"")
    exp = L.gk_graph_check(ctypes.byref(c), 0)
    return got, (exp, L.gk_last_error() if exp else b""), part


BIG = 2**31 - 1
FAULTS = {
    "none": lambda x, a, w, v: None,
    "first row": lambda x, a, w, v: x.__setitem__(1, -1),
    "row beyond the end": lambda x, a, w, v: x.__setitem__(len(x) // 2, BIG),
    "rows crossing": lambda x, a, w, v: x.__setitem__(len(x) - 2, 5),
    "neighbour -1": lambda x, a, w, v: a.__setitem__(0, -1),
    "neighbour n": lambda x, a, w, v: a.__setitem__(len(a) - 1, len(v)),
    "self loop": lambda x, a, w, v: a.__setitem__(len(a) - 1, len(v) - 1),
    "edge weight 0": lambda x, a, w, v: w.__setitem__(len(w) - 1, 0),
    "edge weight negative": lambda x, a, w, v: w.__setitem__(len(w) // 3, -BIG),
    "vertex weight 0": lambda x, a, w, v: v.__setitem__(len(v) - 1, 0),
    "vertex weights 2^31": lambda x, a, w, v: v.__setitem__(7, BIG - len(v) + 2),
    "vertex weights 2^31 - 1": lambda x, a, w, v: v.__setitem__(7, BIG - len(v) + 1),
    "edge weights 2^32": lambda x, a, w, v: w.__setitem__(slice(4, 7), BIG),
}


@pytest.mark.parametrize("n", [LINE // 2 - 1, LINE // 2, LINE // 2 + 1, 70001])
@pytest.mark.parametrize("fault", list(FAULTS))
def test_refusals(gk, ctx, n, fault):
    x, a, w, v = ring(n)
    FAULTS[fault](x, a, w, v)
    got, exp, part = call(gk, ctx, (x, a, w, v))
    assert got == exp
    assert (exp[0] == 0) == (fault in ("none", "vertex weights 2^31 - 1"))
    if exp[0]:
        assert set(part.tolist()) == {-3}


# 1 MiB pieces: an array that ends with one, and one entry on either side;
# 16 MiB: the last graph that is staged, and one that is not
@pytest.mark.parametrize("n", [131071, 131072, 131073, 262143, 599185, 700001])
@pytest.mark.parametrize("weights", [(True, True), (False, False), (True, False)])
def test_upload_pieces(gk, ctx, n, weights):
    from _dev import host, ptr
    x, a, w, v = ring(n)
    rng = np.random.default_rng(n)
    edge = rng.integers(1, 9, n).astype(np.int32)  # edge i joins i and i + 1
    w = np.stack([np.roll(edge, 1), edge], 1).reshape(-1).copy()
    v = rng.integers(1, 4, n).astype(np.int32)
    arrays = (x, a, w if weights[0] else None, v if weights[1] else None)
    got, exp, part = call(gk, ctx, arrays, k=5)
    assert got == exp == (0, b"")
    d = [None if y is None else torch.from_numpy(y).cuda() for y in arrays]
    c = gk.Csr()
    c.n, c.nnz = n, 2 * n
    c.xadj, c.adjncy, c.adjwgt, c.vwgt = [None if y is None else ptr(y) for y in d]
    prm = gk.Params()
    gk.lib().gk_params_default(ctypes.byref(prm), 5)
    out = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    assert gk.lib().gk_partition_device(ctx.handle, ctypes.byref(c), ctypes.byref(prm), ptr(out), None, None) == 0
    assert np.array_equal(part, host(out))
    assert part.min() >= 0 and part.max() == 4
