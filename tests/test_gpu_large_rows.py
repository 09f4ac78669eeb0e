"""Entry points that take several threads per row, at row counts beyond one
launch (2^32 threads): pair export (16 threads a row) from 2^28 rows on,
neighbor count and fill (4 threads a query) from 2^30."""
import ctypes as C

import pytest
import torch

from diffsph_amd import _lib
from diffsph_amd.neighborhood import CellGrid

pytestmark = pytest.mark.gpu


def test_pairs_export_beyond_one_launch():
    n, dev = (1 << 28) + 17, "cuda"
    print(f"case export {n}", flush=True)
    off = torch.zeros(n + 1, dtype=torch.int32, device=dev)
    off[1:] = 1            # row 0 has one pair, the last row two
    off[n] = 3
    q = torch.zeros(n, 2, device=dev)
    q[n - 1] = 0.25
    r = torch.tensor([[0.0, 0.1], [0.25, 0.3], [0.2, 0.25]], device=dev)
    nbr = torch.arange(3, dtype=torch.int32, device=dev)
    P = _lib.ptr
    pr = _lib.Pairs()
    pr.nq, pr.nr = n, 3
    pr.offsets, pr.nbr, pr.qpos, pr.rpos = P(off), P(nbr), P(q), P(r)
    pr.h_uniform, pr.mode = 0.5, 1
    pr.domain = _lib.make_domain((-1, -1), (1, 1), (False, False))
    i, j = torch.full((3,), -1, device=dev), torch.full((3,), -1, device=dev)
    d = torch.zeros(3, device=dev)
    x, gr = (torch.zeros(7, device=dev)[1:].view(3, 2) for _ in range(2))  # aligned to their floats only
    oo = torch.empty(n + 1, dtype=torch.int32, device=dev)
    L = _lib.lib()
    ws = torch.empty(L.dsph_pairs_export_workspace(n), dtype=torch.uint8, device=dev)
    _lib.check(L.dsph_pairs_export(C.byref(pr), None, None, None, P(oo), P(i), P(j), P(d), P(x), None, None, P(gr),
                                   P(ws), ws.numel(), _lib.stream_handle(q.device)), "pairs_export")
    assert i.tolist() == [0, n - 1, n - 1] and j.tolist() == [0, 1, 2]
    torch.testing.assert_close(d.cpu(), torch.tensor([0.2, 0.1, 0.1]))
    torch.testing.assert_close(x.cpu(), torch.tensor([[0.0, -1.0], [0.0, -1.0], [1.0, 0.0]]), rtol=0, atol=1e-5)
    assert (gr[:, 0].abs().cpu() > 0).tolist() == [False, False, True]


@pytest.mark.parametrize("what", ["count", "csr", "fixed"])
def test_search_beyond_one_launch(what):
    n, dev = (1 << 30) + 33, "cuda"
    print(f"case {what} {n}", flush=True)
    domain = _lib.make_domain((-1, -1), (1, 1), (False, False))
    ref = torch.tensor([[0.9, 0.9], [0.88, 0.9], [-0.9, 0.0]], device=dev)
    g = CellGrid.build(ref, None, domain, 0.1, h_uniform=0.1)
    q = torch.zeros(n, 2, device=dev)
    for k in (0, 1 << 29, n - 1):
        q[k] = 0.9
    L, P = _lib.lib(), _lib.ptr
    st = _lib.stream_handle(q.device)
    args = (C.byref(domain), C.byref(g.grid), P(g.cell_start), P(g.sorted_pos), None, 3, P(q), None, n, 1,
            C.c_float(0.1), 1)
    if what == "count":
        cnt = torch.full((n,), -1, dtype=torch.int32, device=dev)
        _lib.check(L.dsph_neighbor_count(*args, P(cnt), st), "neighbor_count")
        rows = torch.nonzero(cnt).flatten()
        assert rows.numel() == 3, f"{rows.numel()} rows with entries"
        assert rows.tolist() == [0, 1 << 29, n - 1] and cnt[rows].tolist() == [2, 2, 2]
    elif what == "fixed":
        # one entry a row: every row of two is cut and reported
        cnt = torch.full((n,), -1, dtype=torch.int32, device=dev)
        nsl = (n + 63) // 64
        so = torch.full((nsl + 1,), -1, dtype=torch.int32, device=dev)
        nbr = torch.full((nsl * 64,), -1, dtype=torch.int32, device=dev)
        flag = torch.zeros(1, dtype=torch.int32, device=dev)
        _lib.check(L.dsph_neighbor_fill_fixed_or(*args, 1, P(cnt), P(so), P(nbr), nbr.numel(), None, P(flag), st),
                   "neighbor_fill_fixed_or")
        assert int(flag) == 1
        assert torch.equal(so, torch.arange(0, nsl * 64 + 1, 64, dtype=torch.int32, device=dev))
        rows = torch.nonzero(cnt).flatten()
        assert rows.numel() == 3, f"{rows.numel()} rows with entries"
        assert rows.tolist() == [0, 1 << 29, n - 1] and cnt[rows].tolist() == [1, 1, 1]
        first = min(g.rank[:2].tolist())
        put = torch.nonzero(nbr >= 0).flatten()
        assert put.tolist() == rows.tolist() and nbr[put].tolist() == [first] * 3
    else:
        off = torch.full((n + 1,), 4, dtype=torch.int32, device=dev)
        off[0] = 0
        off[1: (1 << 29) + 1] = 2
        off[n] = 6
        nbr = torch.full((6,), -1, dtype=torch.int32, device=dev)
        _lib.check(L.dsph_neighbor_fill(*args, P(off), None, 6, P(nbr), 6, st), "neighbor_fill")
        assert nbr.tolist() == sorted(g.rank[:2].tolist()) * 3
