"""The residual written over b (wk_residual with r = b): every element of b is
read once, before its own result replaces it, whatever kernel runs.  FP64 against
the oracle, zero tolerance."""
import sys

import numpy as np
import pytest

from oracle import pyoracle as O
from warpkernel_amd import engine, fe, structure, structure2

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SETS = dict(stage_lds=6, nontemporal=1, rows_per_lane=1)


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def dev(a, ld=None):
    t = torch.from_numpy(np.ascontiguousarray(a)).cuda()
    if ld is None:
        return t
    wide = torch.full((t.shape[0], ld), float("nan"), dtype=t.dtype, device="cuda")
    wide[:, : t.shape[1]] = t
    return wide[:, : t.shape[1]]


# whole tiles, and every remainder of the tiles of 8 and 16 columns that leaves
# a lane fewer columns than it has places
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 13, 16, 17, 18, 19, 31, 32])
@pytest.mark.parametrize("name", ["elastic", "tets"])
def test_residual_over_b(name, k):
    say(f"[gpu] residual in place {name} k={k}")
    m = fe.hex_elastic_3d(6) if name == "elastic" else fe.tet_poisson_3d(9)
    x, b = fe.uniform_x(m.ncols, k, seed=30 + k), fe.uniform_x(m.nrows, k, seed=60 + k)
    x, b = x.reshape(m.ncols, k), b.reshape(m.nrows, k)
    want = b - O.csr_spmv(m.rowptr, m.colind, m.vals, x)
    eng = engine(structure(64).scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind), m.vals, m.colind)
    for cfg in (None, SETS):
        for ldx, ldr in ((None, None), (k + 1, k + 3)):
            r = dev(b, ldr)
            eng.residual(r, dev(x, ldx), r, cfg=cfg)
            assert np.array_equal(r.cpu().numpy(), want), (cfg, ldr)
    eng.close()
    s = structure2(64).scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind, 5)
    eng = engine(s, m.vals, m.colind)
    apart, over = dev(np.zeros_like(b)), dev(b)  # split rows: the same sums, into another array
    eng.residual(dev(b), dev(x), apart)
    eng.residual(over, dev(x), over)
    assert torch.equal(apart, over)
    eng.close()
