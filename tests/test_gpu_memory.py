"""Device memory of destroyed engines: bounded while it is kept, and given back
on request."""
import gc
import sys

import numpy as np
import pytest

import warpkernel_amd
from warpkernel_amd import batch, engine, fe, structure

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

MIB = 1 << 20


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def free():
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return torch.cuda.mem_get_info()[0]


def test_kept_memory_is_bounded_and_given_back():
    """Five engines of about 0.6 GiB: destroyed together they leave at most 2 GiB
    behind, one rebuilt takes its memory from there, and a release returns all."""
    say("[gpu] memory of destroyed engines")
    m = fe.hex_elastic_3d(48)
    csr = [torch.from_numpy(a).cuda() for a in (m.rowptr, m.colind, m.vals)]
    x = torch.from_numpy(fe.uniform_x(m.ncols, seed=1)).cuda()
    ys = [torch.empty(m.nrows, dtype=torch.float64, device="cuda") for _ in range(2)]
    gc.collect()
    warpkernel_amd.release_memory()
    start = free()
    engines = [engine.from_device(*csr) for _ in range(5)]
    engines[0].launch(x, ys[0])
    held = start - free()
    assert held > 5 << 29  # 2.5 GiB
    for e in engines:
        e.close()
    kept = start - free()
    assert 1 << 30 < kept <= (2 << 30) + 64 * MIB
    eng = engine.from_device(*csr)
    assert start - free() <= (2 << 30) + 128 * MIB + held // 5
    eng.launch(x, ys[1])
    assert torch.equal(ys[0], ys[1])
    eng.close()
    given = warpkernel_amd.release_memory()
    assert 1 << 30 < given <= 2 << 30
    assert start - free() < 64 * MIB
    assert warpkernel_amd.release_memory() == 0


def test_release_beside_living_engines():
    say("[gpu] release beside living engines")
    m = fe.hex_elastic_3d(16)
    s = structure(64).scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind)
    x = torch.from_numpy(fe.uniform_x(m.ncols, seed=1)).cuda()
    y = [torch.empty(m.nrows, dtype=torch.float64, device="cuda") for _ in range(3)]
    a, b = engine(s, m.vals, m.colind), engine(s, m.vals, m.colind)
    a.launch(x, y[0])
    b.close()
    bt = batch([a])
    bt.bind([x], [y[2]])
    assert warpkernel_amd.release_memory() > 0
    a.launch(x, y[1])
    bt.run()
    assert torch.equal(y[0], y[1]) and torch.equal(y[0], y[2])
    bt.close()
    a.close()


@pytest.mark.parametrize("where", ["host", "device"])
def test_offsets_that_do_not_fit_are_given_back(where):
    """A band of 2M rows of 5 entries: its column offsets take 32 MB, which an
    engine keeps only if every one of them fits 16 bits."""
    say(f"[gpu] memory of offsets that do not fit, {where}")
    n = 2_000_000
    used = []
    for far in (0, 1):
        rows = np.arange(n, dtype=np.int32)
        ci = np.clip(rows[:, None] + np.arange(-2, 3, dtype=np.int32), 0, n - 1).astype(np.int32)
        if far:
            ci[n // 2, 0] = 7  # a million columns off the diagonal
        rp, vals = (5 * np.arange(n + 1)).astype(np.int32), np.ones(5 * n)
        csr = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (rp, ci.reshape(-1), vals)]
        gc.collect()
        warpkernel_amd.release_memory()
        start = free()
        if where == "host":
            s = structure(64).scan(5 * n, n, vals, rp, ci.reshape(-1))
            eng = engine(s, vals, ci.reshape(-1))
        else:
            eng = engine.from_device(*csr)
        warpkernel_amd.release_memory()
        used.append(start - free())
        x, y = torch.ones(n, dtype=torch.float64, device="cuda"), torch.empty(n, dtype=torch.float64, device="cuda")
        eng.launch(x, y)
        assert bool((y == 5).all())
        eng.close()
    assert used[0] - used[1] > 24 * MIB, used
