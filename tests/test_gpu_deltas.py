"""16-bit column offsets (banded layouts of short rows) on the GPU through the C
ABI: the same products in the same order as the direct kernel, so bit-identical
to it and, in FP64 on WPK1 layouts, to the oracle; no tolerance."""
import sys

import numpy as np
import pytest

from oracle import pyoracle as O
from warpkernel_amd import _capi as capi
from warpkernel_amd import engine, fe, structure, structure2

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

OFFSETS = dict(stage_lds=0, nontemporal=1, rows_per_lane=1, k_tile=1)
DIRECT = dict(OFFSETS, nontemporal=2, unroll=8)  # nontemporal columns: always the direct kernel


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def matrix(nrows, lens, lo, hi, seed, corner=()):
    """Row r: lens[r % len(lens)] entries at columns r + [lo, hi] (clipped into
    range), plus (row, column) entries in corner."""
    rng = np.random.default_rng(seed)
    n = np.asarray([lens[r % len(lens)] for r in range(nrows)], np.int64)
    rows = np.repeat(np.arange(nrows), n)
    cols = np.clip(rows + rng.integers(lo, hi + 1, rows.size), 0, nrows - 1)
    if corner:
        c = np.asarray(corner)
        rows, cols = np.concatenate([rows, c[:, 0]]), np.concatenate([cols, c[:, 1]])
    order = np.lexsort((cols, rows))
    rows, cols = rows[order], cols[order].astype(np.int32)
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=nrows))]).astype(np.int32)
    return fe.CSR("band", nrows, nrows, rp, cols, rng.uniform(-1, 1, rows.size))


CASES = {
    # lengths around the 4-step words and the 8- and 16-step batches; empty rows
    "edges": lambda: matrix(901, [1, 3, 4, 5, 7, 8, 9, 0, 15, 16, 17, 31, 33], -8, 8, 1),
    # batches of 28 steps, their remainders, and two batches
    "long": lambda: matrix(705, [20, 27, 28, 29, 38, 1, 32], -40, 40, 6),
    "hexes": lambda: fe.hex_laplace_3d(6),
    "one_row": lambda: matrix(1, [1], 0, 0, 2),
    # offsets of exactly +-32767 fit; one of 32768 beyond does not (direct kernel)
    "widest": lambda: matrix(70000, [5], -6, 6, 3, [(33000, 233), (100, 32867), (40000, 0)]),
    "too_wide": lambda: matrix(70000, [5], -6, 6, 3, [(33000, 232)]),
    "tets": lambda: fe.tet_poisson_3d(12),
    "laplace": lambda: fe.q1_laplace_2d(37),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("variant", [1, 2])
def test_offsets_match_the_direct_kernel_and_the_oracle(name, variant):
    say(f"[gpu] column offsets {name} variant {variant}")
    m = CASES[name]()
    s = (structure(64) if variant == 1 else structure2(64)).scan(
        m.nnz, m.nrows, m.vals, m.rowptr, m.colind, *([] if variant == 1 else [5]))
    x, b = fe.uniform_x(m.ncols, seed=7), fe.uniform_x(m.nrows, seed=8)
    x[1::13] = -0.0
    ref = O.csr_spmv(m.rowptr, m.colind, m.vals, x)
    for dtype in ("f64", "f32"):
        eng = engine(s, m.vals, m.colind, dtype=dtype, adjoint=dtype == "f64")
        xd = dev(x if dtype == "f64" else x.astype(np.float32))
        nan = torch.full((m.nrows,), float("nan"), dtype=torch.float64, device="cuda")
        for acc in ((0,) if dtype == "f64" else (0, 1)):
            want = nan.clone()
            eng.launch(xd, want, cfg=dict(DIRECT, accumulate=acc))
            for u in (8, 16):
                for wpb, remap in ((1, 0), (2, 1), (8, 1)):
                    y = nan.clone()
                    eng.launch(xd, y, cfg=dict(OFFSETS, unroll=u, waves_per_block=wpb, xcd_remap=remap, accumulate=acc))
                    assert torch.equal(y, want), (dtype, acc, u, wpb, remap)
            y = nan.clone()
            eng.launch(xd, y)
            if acc == 0:
                assert torch.equal(y, want), (dtype, "default")
        if dtype == "f64":
            if variant == 1:
                assert np.array_equal(want.cpu().numpy(), ref)
            y = nan.clone()
            eng.residual(dev(b), xd, y, cfg=dict(OFFSETS, unroll=16))
            assert np.array_equal(y.cpu().numpy(), b - want.cpu().numpy())
            # the combined backward reads the transposed layout's offsets
            dx, dv, dx1, dv1 = nan.clone(), dev(np.zeros(m.nnz)), nan.clone(), dev(np.zeros(m.nnz))
            eng.backward(dev(b), xd, dx, dv)
            eng.run_adjoint(dev(b), dx1, cfg=DIRECT)
            eng.dvals(dev(b), xd, dv1)
            assert torch.equal(dx, dx1) and torch.equal(dv, dv1)
        eng.close()


def test_offsets_follow_special_values_and_column_swaps():
    say("[gpu] column offsets special values and swaps")
    m = matrix(500, [2, 9, 1], -5, 5, 9)
    s = structure(64).scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind)
    eng = engine(s, m.vals, m.colind)
    x = fe.uniform_x(m.ncols, seed=3)
    x[0], x[77], x[300] = np.inf, np.nan, -np.inf  # pads read column 0
    y0, y1 = (torch.empty(m.nrows, dtype=torch.float64, device="cuda") for _ in range(2))
    eng.launch(dev(x), y0, cfg=DIRECT)
    eng.launch(dev(x), y1, cfg=dict(OFFSETS, unroll=16))
    assert torch.equal(torch.isnan(y0), torch.isnan(y1)) and torch.isnan(y0).any()
    assert torch.equal(torch.nan_to_num(y0, nan=1.0), torch.nan_to_num(y1, nan=1.0))
    x = fe.uniform_x(m.ncols, seed=4)
    pc = eng.device_colinds
    for cols in (((pc.astype(np.int64) + 7) % m.ncols).astype(np.int32), pc):
        eng.device_colinds = cols
        eng.launch(dev(x), y0, cfg=DIRECT)
        eng.launch(dev(x), y1, cfg=dict(OFFSETS, unroll=16))
        assert torch.equal(y0, y1)
    eng.close()
