"""New values into layouts with rows far longer than the others, dense columns
(whose transposed layouts are mostly pads), and the one-wave tiles beside the
transposed layout's gather.  The padded values are copies, so they are equal."""
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


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def matrix(nrows, lens, column=0, seed=3, width=30):
    """lens[r % len(lens)] entries in row r within `width` of the diagonal; column > 0: an entry
    of column 0 in each of the first `column` rows too."""
    rng = np.random.default_rng(seed)
    n = np.asarray(lens, np.int64)[np.arange(nrows) % len(lens)]
    rows = np.concatenate([np.repeat(np.arange(nrows), n), np.arange(column)])
    near = np.clip(rows + rng.integers(-width, width + 1, rows.size), 1, nrows - 1)
    cols = np.where(np.arange(rows.size) < n.sum(), near, 0)
    order = np.lexsort((cols, rows))
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=nrows))]).astype(np.int32)
    return fe.CSR("long", nrows, nrows, rp, cols[order].astype(np.int32), rng.uniform(-1, 1, rows.size))


CASES = {
    "one_long": matrix(3000, [20000] + [9] * 2999),
    "few_long": matrix(3000, ([2000] + [3] * 99)),
    "dense": matrix(150, [900]),
    "column": matrix(6000, [5, 7], 6000),
    "column_and_row": matrix(6000, [4000] + [5] * 5999, 3000),
    "scattered": matrix(70000, [15, 17], width=300),  # 1.1M entries, far apart in the transposed layout
    "short_4": matrix(64 * 4096 + 7, [1, 4, 3]),
    "short_8": matrix(64 * 4096 + 7, [5, 8, 1, 7]),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("variant", [1, 2])
@pytest.mark.parametrize("dtype,adjoint", [("f64", False), ("f64", True), ("f32", True)])
def test_update_values_of_long_rows(name, variant, dtype, adjoint):
    say(f"[gpu] update long {name} {variant} {dtype} adjoint {adjoint}")
    m = CASES[name]
    s = structure(64) if variant == 1 else structure2(64)
    s.scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind, *([] if variant == 1 else [5]))
    eng = engine(s, m.vals, m.colind, dtype=dtype, adjoint=adjoint)
    new = np.random.default_rng(9).uniform(-1, 1, m.nnz).astype(np.float64 if dtype == "f64" else np.float32)
    eng.update_values(dev(new))
    pv, _ = s.process_host(new.astype(np.float64), m.colind)
    assert np.array_equal(eng.download(capi.WK_ENGINE_VALUES), pv.astype(new.dtype))
    if adjoint:
        # the transposed layout's values: the same sums as an engine built on them
        other = engine(s, new.astype(np.float64), m.colind, dtype=dtype, adjoint=True)
        dy = dev(fe.uniform_x(m.nrows, seed=4).astype(new.dtype))
        a, b = (torch.full((m.ncols,), float("nan"), dtype=torch.float64, device="cuda") for _ in range(2))
        eng.run_adjoint(dy, a)
        other.run_adjoint(dy, b)
        assert torch.equal(a, b)
        other.close()
    eng.close()


@pytest.mark.parametrize("name", ["short_4", "short_8", "column_and_row"])
@pytest.mark.parametrize("variant", [1, 2])
def test_update_values_of_narrow_groups(name, variant):
    """Group width 32, short rows (one wave a group) and long ones, both layouts."""
    say(f"[gpu] update narrow {name} {variant}")
    m = CASES[name]
    s = structure(32) if variant == 1 else structure2(32)
    s.scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind, *([] if variant == 1 else [5]))
    eng = engine(s, m.vals, m.colind, adjoint=True)
    new = np.random.default_rng(9).uniform(-1, 1, m.nnz)
    eng.update_values(dev(new))
    pv, _ = s.process_host(new, m.colind)
    assert np.array_equal(eng.download(capi.WK_ENGINE_VALUES), pv)
    other = engine(s, new, m.colind, adjoint=True)
    dy = dev(fe.uniform_x(m.nrows, seed=4))
    a, b = (torch.full((m.ncols,), float("nan"), dtype=torch.float64, device="cuda") for _ in range(2))
    eng.run_adjoint(dy, a)
    other.run_adjoint(dy, b)
    assert torch.equal(a, b)
    other.close()
    eng.close()


def test_one_long_row_does_not_set_the_time():
    """200,000 rows of 9 entries, with and without one of 100,000 (5% more
    entries): within a factor of ten of each other, 50 us aside."""
    say("[gpu] update, one long row")
    us = []
    for lens in ([9], [100000] + [9] * 199999):
        m = matrix(200000, lens)
        s = structure(64).scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind)
        eng = engine(s, m.vals, m.colind)
        v = dev(m.vals)
        times = []
        for _ in range(7):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(4):
                eng.update_values(v)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b) * 250)
        us.append(sorted(times)[3])
        eng.close()
    say(f"[gpu] update {us[0]:.1f} us without, {us[1]:.1f} us with the long row")
    assert us[1] < 10 * us[0] + 50
