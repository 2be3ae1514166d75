"""New values into the layouts (wk_engine_update_values) at the edges of the
update kernel's tiles: row lengths around its 32 steps, empty rows, both group
widths, split rows, row-sorted and transposed layouts, FP32 values, engines
scanned on the device.  The padded values are copies, so they are equal."""
import sys

import numpy as np
import pytest

from oracle import pyoracle as O
from warpkernel_amd import _capi as capi
from warpkernel_amd import engine, fe, structure, structure2

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def matrix(nrows, lens, seed):
    rng = np.random.default_rng(seed)
    n = np.asarray([lens[r % len(lens)] for r in range(nrows)], np.int64)
    rp = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    rows = np.repeat(np.arange(nrows), n)
    ci = rng.integers(0, nrows, rows.size)
    ci = ci[np.lexsort((ci, rows))].astype(np.int32)
    return fe.CSR("update", nrows, nrows, rp, ci, rng.uniform(-1, 1, rows.size))


CASES = {
    "one": (1, [1]),
    "edges": (331, [31, 32, 33, 0, 63, 64, 65, 1]),
    "long": (70, [700, 3]),
    "partial": (129, [27]),
}


def scanned(m, variant, width):
    s = structure(width) if variant == 1 else structure2(width)
    return s.scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind, *([] if variant == 1 else [5]))


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("variant,width,dtype,adjoint", [
    (1, 64, "f64", False), (1, 64, "f32", False), (2, 64, "f64", False), (1, 32, "f64", False),
    (2, 32, "f64", False), (1, 64, "f64", True), (2, 64, "f64", True), (1, 32, "f64", True)])
def test_update_values_equals_process(name, variant, width, dtype, adjoint):
    say(f"[gpu] update {name} {variant} {width} {dtype} adjoint {adjoint}")
    m = matrix(*CASES[name], seed=3)
    s = scanned(m, variant, width)
    eng = engine(s, m.vals, m.colind, dtype=dtype, adjoint=adjoint)
    new = np.random.default_rng(9).uniform(-1, 1, m.nnz).astype(np.float64 if dtype == "f64" else np.float32)
    eng.update_values(torch.from_numpy(new).cuda())
    pv, _ = s.process_host(new.astype(np.float64), m.colind)
    assert np.array_equal(eng.download(capi.WK_ENGINE_VALUES), pv.astype(new.dtype))
    if adjoint:
        dy = fe.uniform_x(m.nrows, seed=4)
        colptr, rowind, perm = O.transpose(m.nrows, m.ncols, m.rowptr, m.colind)
        dx = torch.full((m.ncols,), float("nan"), dtype=torch.float64, device="cuda")
        eng.run_adjoint(torch.from_numpy(dy).cuda(), dx)
        ref = O.csr_spmv(colptr, rowind, new[perm], dy)
        if variant == 1:
            assert np.array_equal(dx.cpu().numpy(), ref)
        else:  # split rows: lane partials in tree order
            assert np.linalg.norm(dx.cpu().numpy() - ref) <= 1e-14 * np.linalg.norm(ref)
    eng.close()


def test_update_values_row_sorted_and_device_scanned():
    say("[gpu] update row-sorted and device-scanned")
    m = matrix(331, [31, 32, 33, 0, 5], seed=5)
    s = scanned(m, 1, 64)
    new = np.random.default_rng(10).uniform(-1, 1, m.nnz)
    d = torch.from_numpy(new).cuda()
    a = engine(s, m.vals, m.colind, rowsort=True)
    a.update_values(d)
    b = engine(s, new, m.colind, rowsort=True)
    assert np.array_equal(a.download(capi.WK_ENGINE_VALUES), b.download(capi.WK_ENGINE_VALUES))
    c = engine.from_device(*(torch.from_numpy(v).cuda() for v in (m.rowptr, m.colind, m.vals)))
    c.update_values(d)
    assert np.array_equal(c.download(capi.WK_ENGINE_VALUES), s.process_host(new, m.colind)[0])
    for e in (a, b, c):
        e.close()


@pytest.mark.parametrize("lens", [[1, 4, 3], [4], [5, 8, 1, 7], [8], [9, 7, 8]])
@pytest.mark.parametrize("variant", [1, 2])
def test_update_values_of_many_short_groups(lens, variant):
    """4,097 groups of rows: the tiles of 4 and 8 steps (one wave a group), and past them."""
    say(f"[gpu] update many {lens} {variant}")
    m = matrix(64 * 4096 + 7, lens, seed=6)
    s = scanned(m, variant, 64)
    eng = engine(s, m.vals, m.colind)
    new = np.random.default_rng(11).uniform(-1, 1, m.nnz)
    eng.update_values(torch.from_numpy(new).cuda())
    pv, _ = s.process_host(new, m.colind)
    assert np.array_equal(eng.download(capi.WK_ENGINE_VALUES), pv)
    eng.close()
