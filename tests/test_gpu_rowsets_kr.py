"""Row sets in Kr numbering: which rows share a set.  FP64 against the window
kernel on the same engine, zero tolerance."""
import sys

import numpy as np
import pytest

from warpkernel_amd import engine, fe, structure

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SETS = dict(stage_lds=6, nontemporal=1, rows_per_lane=1)
OTHER = dict(stage_lds=4, nontemporal=1, rows_per_lane=1, unroll=8, waves_per_block=1, k_tile=4)


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def out(rows, k):
    return torch.full((rows, k), float("nan"), dtype=torch.float64, device="cuda")


def test_row_sets_in_kr_numbering_tell_pads_from_column_0():
    """Row 7 ends with an entry of column 0 where row 0, next in its group and on
    the same other columns, has a pad: row 0 does not read x at column 0."""
    say("[gpu] row sets, pads and column 0 in Kr numbering")
    n, k = 192, 8
    rows = [np.array([3, 4, 5]) + 3 * (r // 3 % 60) for r in range(n)]
    rows[0] = rows[1] = np.array([3, 4, 5])
    rows[7] = np.array([3, 4, 5, 0])
    rp = np.concatenate([[0], np.cumsum([r.size for r in rows])]).astype(np.int32)
    ci = np.concatenate(rows).astype(np.int32)
    vals = np.random.default_rng(2).uniform(-1, 1, ci.size)
    s = structure(64).scan(ci.size, n, vals, rp, ci)
    assert list(s.row_map[:2]) == [7, 0]
    x = fe.uniform_x(n, k, seed=5)
    x[0] = np.inf
    eng = engine(s, vals, ci, kr=True)
    ys = []
    for cfg in (OTHER, SETS, None):
        y = out(n, k)
        eng.launch_x(dev(x[s.row_map]), y, cfg=cfg)
        ys.append(y.cpu().numpy())
    assert np.isinf(ys[0][0]).all() and np.isfinite(ys[0][1:]).all()
    assert np.array_equal(ys[0], ys[1]) and np.array_equal(ys[0], ys[2])
    eng.close()
