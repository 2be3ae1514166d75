"""Windows built on the GPU in one pass, at its edges: longest groups of 16, 32, 96
and 128 steps (registers per thread), column spans on both sides of 65,536 and
262,144 (the two bitmaps, the sort), more keys than a window may have, node
windows whose triples end inside a wave's batch.  Every array equals the
host-built one (whole numbers: no tolerance)."""
import numpy as np
import pytest

from warpkernel_amd import _capi as capi
from warpkernel_amd import engine, fe, structure, structure2

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

ARRAYS = (capi.WK_ENGINE_COLS, capi.WK_ENGINE_COLS_KR, capi.WK_ENGINE_WIN_IDX, capi.WK_ENGINE_WIN_OFF,
          capi.WK_ENGINE_WIN_COLS, capi.WK_ENGINE_WIN_COLS_KR, capi.WK_ENGINE_ND_CNT, capi.WK_ENGINE_ND_OFF,
          capi.WK_ENGINE_ND_POS)


def csr(n, rows, cols, seed):
    order = np.lexsort((cols, rows))
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int32)
    return fe.CSR("windows", n, n, rp, cols[order].astype(np.int32),
                  np.random.default_rng(seed).uniform(-1, 1, rows.size))


def band(nrows, lens, pool, seed):
    """lens[r % len(lens)] columns of row r out of a band of `pool` columns by
    64-row block, so that a group's keys are at most `pool`."""
    rng = np.random.default_rng(seed)
    n = np.asarray([lens[r % len(lens)] for r in range(nrows)], np.int64)
    rows = np.repeat(np.arange(nrows), n)
    lo = np.minimum(rows // 64 * 64, max(nrows - pool, 0))
    return csr(nrows, rows, lo + rng.integers(0, min(pool, nrows), rows.size), seed)


def spread(ncols, span, rows=128):
    """Groups whose first row reads columns 5 and 5 + span."""
    r = np.repeat(np.arange(rows), 3)
    c = np.tile([5, 17, 40], rows) + r // 3 % 64
    c[0::192], c[2::192] = 5, 5 + span
    return csr(ncols, r, c, span)


def nodes(nn, reach, seed):
    """3 rows a node, triples of columns over the nodes within `reach`."""
    rng = np.random.default_rng(seed)
    rows, cols = [], []
    for i in range(nn):
        near = np.unique(np.clip(i + rng.integers(-reach, reach + 1, 2 * reach), 0, nn - 1))
        for d in range(3):
            rows.append(np.full(3 * near.size, 3 * i + d))
            cols.append((3 * near[:, None] + np.arange(3)).ravel())
    return csr(3 * nn, np.concatenate(rows), np.concatenate(cols), seed)


CASES = {
    **{f"len{n}": (lambda n=n: band(200, [n, 3], 300, n)) for n in (16, 17, 32, 33, 96, 97, 128)},
    **{f"span{n}": (lambda n=n: spread(70000, n)) for n in (65534, 65535, 65536, 65537)},
    "ncols65536": lambda: spread(65536, 65530),
    **{f"span{n}": (lambda n=n: spread(300000, n)) for n in (262142, 262143, 262144)},
    "keys2048": lambda: csr(9000, np.repeat(np.arange(64), 32), np.arange(2048) * 4, 1),
    "keys2049": lambda: csr(9000, np.repeat(np.arange(65), 33), np.arange(65 * 33) * 4, 2),
    "nodes": lambda: nodes(130, 9, 3),
    "nodes_long": lambda: nodes(90, 22, 4),
    "elastic": lambda: fe.hex_elastic_3d(5),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("variant", [1, 2])
def test_windows_equal_the_host_built(name, variant):
    print(f"[gpu] windows {name} variant {variant}", flush=True)
    m = CASES[name]()
    s = (structure(64) if variant == 1 else structure2(64)).scan(
        m.nnz, m.nrows, m.vals, m.rowptr, m.colind, *([] if variant == 1 else [9]))
    host = engine(s, m.vals, m.colind, kr=True)
    dev = engine.from_device(*(torch.from_numpy(a).cuda() for a in (m.rowptr, m.colind, m.vals)), variant=variant,
                             threshold=9 if variant == 2 else 0, kr=True)
    for which in ARRAYS:
        a, b = host.download(which), dev.download(which)
        assert np.array_equal(a, b), (which, a.size, b.size)
    cnt, off = (host.download(w).astype(np.int64) for w in (capi.WK_ENGINE_ND_CNT, capi.WK_ENGINE_WIN_OFF))
    if cnt.size:  # the node windows' entries: as many as each group has
        at = np.concatenate([o + np.arange(c) for o, c in zip(off, cnt)])
        for which, shape in ((capi.WK_ENGINE_ND_COLS, -1), (capi.WK_ENGINE_ND_COLS_KR, (-1, 3))):
            a, b = (e.download(which).reshape(shape)[at] for e in (host, dev))
            assert np.array_equal(a, b), which
    assert (cnt.size > 0) == (variant == 1 and name in ("nodes", "nodes_long", "elastic")) or variant == 2
    x = torch.rand(m.ncols, dtype=torch.float64, device="cuda")
    y0, y1 = (torch.full((m.nrows,), float("nan"), dtype=torch.float64, device="cuda") for _ in range(2))
    host.launch(x, y0)
    dev.launch(x, y1)
    assert torch.equal(y0, y1)
    host.close()
    dev.close()


def test_long_rows_are_scanned_when_the_call_returns():
    """Rows past 128 entries have no windows: the engine built on one stream is
    whole when the call returns, for any other stream."""
    print("[gpu] device scan of long rows on a side stream", flush=True)
    m = band(20000, [300, 150], 2000, 9)
    host = engine(structure(64).scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind), m.vals, m.colind)
    a = [torch.from_numpy(v).cuda() for v in (m.rowptr, m.colind, m.vals)]
    x = torch.rand(m.ncols, dtype=torch.float64, device="cuda")
    y0, y1 = (torch.full((m.nrows,), float("nan"), dtype=torch.float64, device="cuda") for _ in range(2))
    host.launch(x, y0)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    dev = engine.from_device(*a, stream=side)
    assert side.query()
    dev.launch(x, y1)
    assert torch.equal(y0, y1)
    host.close()
    dev.close()
