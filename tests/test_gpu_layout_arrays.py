"""Engines on layouts made from arrays (wk_layout_from_arrays) that a scan would
not give but whose arrays are valid: the products are the direct kernel's."""
import ctypes as C
import sys

import numpy as np
import pytest

from oracle import pyoracle as O
from warpkernel_amd import _capi as capi
from warpkernel_amd import engine, fe, structure, structure2
from warpkernel_amd._capi import check, lib

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def layout(variant, nrows, nznrows, rowptr, row_map, reorder, lens, tpr=None, row_off=None):
    """A structure or structure2 of group width 64 over the given arrays."""
    ptr = lambda a, t: np.ascontiguousarray(a, t).ctypes.data_as(C.c_void_p)
    rowptr = np.ascontiguousarray(rowptr, np.int32)
    offsets = np.concatenate([[0], np.cumsum(np.asarray(lens, np.int64) * 64)]).astype(np.int64)
    keep = [np.ascontiguousarray(a, t) for a, t in (
        (rowptr, np.int32), (row_map, np.int32), (reorder, np.uint32), (offsets, np.int64), (lens, np.uint32),
        (tpr if variant == 2 else [0], np.uint32), (row_off if variant == 2 else [0], np.uint32))]
    p = [a.ctypes.data_as(C.c_void_p) for a in keep]
    h = C.c_void_p()
    check(lib().wk_layout_from_arrays(variant, 64, 5 if variant == 2 else 0, 32 if variant == 2 else 0, nrows, nrows,
                                      nznrows, len(lens), len(reorder), int(offsets[-1]), *p[:5],
                                      p[5] if variant == 2 else None, p[6] if variant == 2 else None, C.byref(h)))
    s = structure(64) if variant == 1 else structure2(64)
    s._h, s._rowptr = h, rowptr
    s._load_fields()
    return s


def blocks(nodes, empty):
    """Three rows per node that share the columns of the node and the next, then
    `empty` rows without entries."""
    n = 3 * nodes + empty
    cols = [np.arange(3 * i, min(3 * i + 6, 3 * nodes)) for i in range(nodes) for _ in range(3)]
    lens = np.concatenate([[len(c) for c in cols], np.zeros(empty, int)])
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ci = np.concatenate(cols).astype(np.int32)
    return fe.CSR("blocks", n, n, rp, ci, np.random.default_rng(1).uniform(-1, 1, ci.size))


@pytest.mark.parametrize("k", [1, 4, 8, 17])
def test_group_without_entries(k):
    """Rows without entries counted among the rows with entries: a last group of
    no steps."""
    say(f"[gpu] layout with an empty group k={k}")
    m = blocks(40, 70)  # 190 rows: two groups with entries, one without
    s = structure(64).scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind)
    assert s.nznrows == 120 and s.nwarps == 2
    s = layout(1, m.nrows, m.nrows, m.rowptr, s.row_map, s.reorder_rows, list(s.max_nz_rows) + [0])
    x = fe.uniform_x(m.ncols, k, seed=4).reshape(m.ncols, k)
    ref = O.csr_spmv(m.rowptr, m.colind, m.vals, x).reshape(m.nrows, k)
    for dtype in ("f64", "f32"):
        eng = engine(s, m.vals, m.colind, dtype=dtype)
        y = torch.full((m.nrows, k), float("nan"), dtype=torch.float64, device="cuda")
        eng.launch(dev(x if dtype == "f64" else x.astype(np.float32)), y)
        if dtype == "f64":
            assert np.array_equal(y.cpu().numpy(), ref)
        else:  # inputs rounded to 24 bits: at most 2^-23 per product and six products a row
            bound = 2.0 ** -22 * O.csr_spmv(m.rowptr, m.colind, np.abs(m.vals), np.abs(x)).reshape(m.nrows, k)
            assert np.all(np.abs(y.cpu().numpy() - ref) <= bound)
        eng.close()
    s.close()


def test_groups_without_rows():
    """Split groups, none of whose rows counts as one with entries: y is 0."""
    say("[gpu] layout without rows that count")
    n, lens = 130, [2, 1]
    rp = np.minimum(np.arange(n + 1), 60).astype(np.int32)  # 60 rows of one entry
    s = layout(2, n, 0, rp, np.arange(n), np.arange(60), lens, tpr=[1, 1], row_off=[0, 64, n])
    colind = np.arange(60, dtype=np.int32)
    eng = engine(s, np.full(60, 2.0), colind)
    x = torch.ones(n, dtype=torch.float64, device="cuda")
    for cfg in (None, dict(stage_lds=0, unroll=8, nontemporal=1, rows_per_lane=1, k_tile=1)):
        y = torch.full((n,), float("nan"), dtype=torch.float64, device="cuda")
        eng.launch(x, y, cfg=cfg)
        assert torch.equal(y, torch.zeros_like(y)), cfg
    eng.close()
    s.close()
