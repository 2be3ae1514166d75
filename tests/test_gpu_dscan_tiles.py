"""Scan and process on the GPU at the edges of its tiles: row lengths around the
32 steps the fill turns at a time, column spans on both sides of the 262,144
bits of the window bitmap, pads, duplicate columns and split rows.  Every array
equals the host-scanned engine's (whole numbers and copied values: no tolerance)."""
import gc
import sys
import weakref

import numpy as np
import pytest

from warpkernel_amd import _capi as capi
from warpkernel_amd import engine, fe, structure, structure2

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

ARRAYS = (capi.WK_ENGINE_VALUES, capi.WK_ENGINE_COLS, capi.WK_ENGINE_COLS_KR, capi.WK_REORDER_ROWS,
          capi.WK_ENGINE_WIN_IDX, capi.WK_ENGINE_WIN_OFF, capi.WK_ENGINE_WIN_COLS, capi.WK_ENGINE_WIN_COLS_KR)


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def matrix(nrows, lens, span, seed):
    """Row r has lens[r % len(lens)] entries in a band of `span` columns around r
    (wrapped into range), sorted, duplicates possible."""
    rng = np.random.default_rng(seed)
    n = np.asarray([lens[r % len(lens)] for r in range(nrows)], np.int64)
    rp = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    rows = np.repeat(np.arange(nrows), n)
    ci = (rows + rng.integers(0, span, rows.size)) % nrows
    ci = ci[np.lexsort((ci, rows))].astype(np.int32)
    return fe.CSR("tiles", nrows, nrows, rp, ci, rng.uniform(-1, 1, rows.size))


CASES = {
    "short": (700, [1, 2, 0, 31], 90),
    "edges": (333, [31, 32, 33, 63, 64, 65, 0, 100], 300),
    "one_row": (1, [1], 1),
    "narrow_bitmap": (300000, [3, 5], 262080),    # most spans just inside the bitmap
    "wide": (300000, [3, 5], 300000),             # sorted keys
    "mixed": (270000, [2, 1], 262144),            # both in one layout (wrapped rows span everything)
    "no_windows": (400, [129], 400),              # groups of more than 8192 slots
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("variant,dtype", [(1, "f64"), (2, "f64"), (1, "f32")])
def test_device_scan_equals_host_scan(name, variant, dtype):
    say(f"[gpu] device scan tiles {name} variant {variant} {dtype}")
    m = matrix(*CASES[name], seed=len(name))
    s = (structure(64) if variant == 1 else structure2(64)).scan(
        m.nnz, m.nrows, m.vals, m.rowptr, m.colind, *([] if variant == 1 else [5]))
    host = engine(s, m.vals, m.colind, dtype=dtype, kr=True)
    dev = engine.from_device(*(torch.from_numpy(a).cuda() for a in (m.rowptr, m.colind, m.vals)), variant=variant,
                             threshold=5 if variant == 2 else 0, dtype=dtype, kr=True)
    for which in ARRAYS:
        a, b = host.download(which), dev.download(which)
        if name == "no_windows" and variant == 1 and which >= capi.WK_ENGINE_WIN_IDX:
            assert b.size == 0  # groups this large get no windows on the device
            continue
        assert np.array_equal(a, b), (which, a.size, b.size)
    host.close()
    dev.close()


def test_device_scanned_engine_is_freed_when_dropped():
    """Without the garbage collector; its layout keeps it alive while held."""
    say("[gpu] device-scanned engine lifetime")
    m = matrix(130, [3, 1, 7], 60, 1)
    csr = [torch.from_numpy(a).cuda() for a in (m.rowptr, m.colind, m.vals)]
    rows = structure(64).scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind).row_map
    gc.disable()
    try:
        eng = engine.from_device(*csr)
        ref = weakref.ref(eng)
        assert eng.kernel is eng.kernel or eng.kernel.nz == m.nnz
        assert np.array_equal(eng.kernel.row_map, rows) and eng.kernel.row_map is eng.kernel.row_map
        layout = eng.kernel
        del eng
        assert ref() is not None and layout.nrows == m.nrows
        assert np.array_equal(layout.row_map_inv[layout.row_map], np.arange(m.nrows))
        del layout
        assert ref() is None
        eng = engine.from_device(*csr)
        eng.close()
        assert eng.kernel.nz == m.nnz  # the scalars outlive the device arrays
    finally:
        gc.enable()


def test_rebuilt_engines_reuse_device_blocks():
    """Engines rebuilt in place keep their results while blocks change hands
    (another engine alive, launches in flight when one is destroyed), and the
    device memory held afterwards is bounded."""
    say("[gpu] rebuilt engines")
    free0 = torch.cuda.mem_get_info()[0]
    mats = [fe.hex_elastic_3d(n) for n in (24, 20, 25)]
    csr = [[torch.from_numpy(a).cuda() for a in (m.rowptr, m.colind, m.vals)] for m in mats]
    xs = [torch.from_numpy(fe.uniform_x(m.ncols, seed=i)).cuda() for i, m in enumerate(mats)]
    first = []
    for m, c, x in zip(mats, csr, xs):
        y = torch.full((m.nrows,), float("nan"), dtype=torch.float64, device="cuda")
        eng = engine.from_device(*c)
        eng.launch(x, y)
        first.append(y.clone())
    kept = engine.from_device(*csr[0])  # stays alive while the others come and go
    for rep in range(12):
        i = rep % 3
        ys = torch.full((mats[i].nrows,), float("nan"), dtype=torch.float64, device="cuda")
        eng = engine.from_device(*csr[i])
        eng.launch(xs[i], ys)
        eng.close()  # the product may still be running
        yk = torch.full((mats[0].nrows,), float("nan"), dtype=torch.float64, device="cuda")
        kept.launch(xs[0], yk)
        assert torch.equal(ys, first[i]) and torch.equal(yk, first[0]), rep
    kept.close()
    del csr, xs, first, ys, yk
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    assert free0 - torch.cuda.mem_get_info()[0] < (3 << 30)  # 2 GiB kept at most
