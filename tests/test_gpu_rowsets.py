"""Row sets (stage_lds = 6 on layouts whose neighbouring rows share their
columns) on the GPU through the C ABI: several right-hand sides on the matrix
cores.  Every row sums its slots in order by fma, so FP64 results and FP32
values with FP64 sums are bit-identical to the oracle's CSR product; the
tolerance is zero."""
import sys

import numpy as np
import pytest

from oracle import pyoracle as O
from warpkernel_amd import engine, fe, structure
from warpkernel_amd import _capi as capi

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SETS = dict(stage_lds=6, nontemporal=1, rows_per_lane=1)
OTHER = dict(stage_lds=4, nontemporal=1, rows_per_lane=1, unroll=8, waves_per_block=1, k_tile=4)


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


def out(rows, k, ld=None):
    return dev(np.full((rows, k), np.nan), ld)


def blocks(nodes, dof, degrees, seed, far=0):
    """dof x dof dense blocks over a random node graph: node i couples to itself
    and degrees[i % len] - 1 further nodes (degree 0: empty rows).  far > 0
    couples some nodes across that many columns."""
    rng = np.random.default_rng(seed)
    lens, cols = [], []
    for i in range(nodes):
        d = min(int(degrees[i % len(degrees)]), nodes)
        near = np.unique((i + np.concatenate([[0], rng.integers(-40, 41, 4 * d)])) % nodes)
        pick = np.sort(rng.permutation(near)[:d]) if d else np.zeros(0, int)
        if far and d and i % 3 == 0:
            pick = np.unique(np.append(pick, (i + far) % nodes))
        c = (pick[:, None] * dof + np.arange(dof)).reshape(-1)
        for _ in range(dof):
            lens.append(c.size)
            cols.append(c)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ci = np.concatenate(cols).astype(np.int32) if rp[-1] else np.zeros(0, np.int32)
    n = nodes * dof
    return fe.CSR("blocks", n, n, rp, ci, rng.uniform(-1, 1, int(rp[-1])))


CASES = {
    "elastic_1": lambda: fe.hex_elastic_3d(1),
    "elastic_9": lambda: fe.hex_elastic_3d(9),
    # 2, 3, 4 and 6 unknowns per node (sets of 2, 3, 4 and 4 + 2 rows); group
    # lengths around the 28-step chunks (27, 28, 29, 56, 57, 84) and empty rows
    "dof2": lambda: blocks(331, 2, [14, 1, 0, 15, 28, 29, 42], 1),
    "dof3": lambda: blocks(257, 3, [9, 10, 0, 19, 28, 27, 1], 2),
    "dof4": lambda: blocks(190, 4, [7, 14, 21, 1], 3),
    "dof6": lambda: blocks(97, 6, [14, 9, 5], 4),
    # column spans above 65,535 (int32 columns)
    "far": lambda: blocks(30000, 3, [3, 4], 5, far=25000),
    # rows of 87 entries: no row sets, the other kernels take over
    "long": lambda: blocks(120, 3, [29], 6),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("k", [2, 3, 5, 8, 9, 17, 32])
def test_row_sets_match_the_oracle(name, k):
    say(f"[gpu] row sets {name} k={k}")
    m = CASES[name]()
    s = structure(64).scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind)
    x = fe.uniform_x(m.ncols, k, seed=70 + k)
    b = fe.uniform_x(m.nrows, k, seed=90 + k)
    ref = O.csr_spmv(m.rowptr, m.colind, m.vals, x)
    perm = np.asarray(s.row_map)
    eng = engine(s, m.vals, m.colind, kr=True, adjoint=True)
    for cfg in (dict(SETS, xcd_remap=0), dict(SETS, xcd_remap=1), None):
        for ldx, ldy in ((None, None), (k + 3, k + 1)):  # rows of x off 16 bytes too
            y = out(m.nrows, k, ldy)
            eng.launch(dev(x, ldx), y, cfg=cfg)
            assert np.array_equal(y.cpu().numpy(), ref), (cfg, ldx)
            if ldy:
                assert torch.isnan(y._base if y._base is not None else y)[:, k:].all()  # nothing past column k
        y = out(m.nrows, k)
        eng.launch_x(dev(x[perm]), y, cfg=cfg)
        assert np.array_equal(y.cpu().numpy(), ref[perm]), (cfg, "run_x")
        eng.residual(dev(b), dev(x), y, cfg=cfg)
        assert np.array_equal(y.cpu().numpy(), b - ref), (cfg, "residual")
    colptr, rowind, perm_t = O.transpose(m.nrows, m.ncols, m.rowptr, m.colind)
    y = out(m.ncols, k)
    eng.run_adjoint(dev(x), y, cfg=SETS)
    assert np.array_equal(y.cpu().numpy(), O.csr_spmv(colptr, rowind, m.vals[perm_t], x)), "adjoint"
    eng.close()
    e32 = engine(s, m.vals, m.colind, dtype="f32", kr=True)
    vq, xq = m.vals.astype(np.float32), x.astype(np.float32)
    ref = O.csr_spmv(m.rowptr, m.colind, vq.astype(np.float64), xq.astype(np.float64))
    for ldx in (None, k + 1):
        y = out(m.nrows, k)
        e32.launch(dev(xq, ldx), y, cfg=dict(SETS, accumulate=capi.WK_ACC_F64))
        assert np.array_equal(y.cpu().numpy(), ref), ("f32", ldx)
    e32.launch_x(dev(xq[perm]), y, cfg=dict(SETS, accumulate=capi.WK_ACC_F64))
    assert np.array_equal(y.cpu().numpy(), ref[perm]), ("f32", "run_x")
    e32.close()


@pytest.mark.parametrize("k", [5, 16])
def test_row_sets_read_special_values_as_the_other_kernels(k):
    """Infinities, NaN, signed zeros and subnormals in x (pads read column 0):
    as the window kernels, bit for bit where the result is a number."""
    say(f"[gpu] row sets special values k={k}")
    m = blocks(211, 3, [9, 4, 19, 28], 7)
    s = structure(64).scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind)
    vals = m.vals.copy()
    vals[::7] = -0.0
    vals[::11] *= 1e-310
    x = fe.uniform_x(m.ncols, k, seed=5)
    x[::5] = 0.0
    x[1::9] = -0.0
    x[2::31] *= 1e-300
    x[100, 0], x[230, k - 1], x[0, 1] = np.inf, np.nan, -np.inf
    eng = engine(s, vals, m.colind)
    y0, y1 = out(m.nrows, k), out(m.nrows, k)
    eng.launch(dev(x), y0, cfg=OTHER)
    eng.launch(dev(x), y1, cfg=SETS)
    a, c = y0.cpu().numpy(), y1.cpu().numpy()
    assert np.array_equal(np.isnan(a), np.isnan(c)) and np.isnan(a).any()
    ok = ~np.isnan(a)
    assert np.array_equal(a[ok].view(np.int64), c[ok].view(np.int64))
    eng.close()


def test_row_sets_default_and_column_swap():
    """The default uses the row sets from k = 5 on elasticity; swapped columns
    turn them off, and the scanned ones back on."""
    say("[gpu] row sets default and column swap")
    m = fe.hex_elastic_3d(6)
    s = structure(64).scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind)
    x = fe.uniform_x(m.ncols, 8, seed=6)
    eng = engine(s, m.vals, m.colind)
    assert eng.get_launch(k=8).stage_lds == 6
    pc = eng.device_colinds
    other = ((pc.astype(np.int64) + 3) % m.ncols).astype(np.int32)
    y = out(m.nrows, 8)
    for cols, shift in ((other, 3), (pc, 0)):
        eng.device_colinds = cols
        eng.launch(dev(x), y, cfg=SETS)
        ci = ((m.colind.astype(np.int64) + shift) % m.ncols).astype(np.int32)
        ref = O.csr_spmv(m.rowptr, ci, m.vals, x)
        # pads hold value 0: 0 * x[column] adds +-0, which no nonzero sum sees
        assert np.array_equal(y.cpu().numpy(), ref), shift
    eng.close()
    e32 = engine(s, m.vals, m.colind, dtype="f32")
    xq, vq = x.astype(np.float32), m.vals.astype(np.float32)
    ref = O.csr_spmv(m.rowptr, m.colind, vq.astype(np.float64), xq.astype(np.float64))
    e32.launch(dev(xq), y)
    assert np.array_equal(y.cpu().numpy(), ref)  # FP64 sums by default here
    e32.close()


@pytest.mark.parametrize("where", ["host", "device"])
def test_row_sets_are_built_when_the_call_returns(where):
    """An engine built on one stream is whole when the call returns, for any other."""
    say(f"[gpu] row sets built on a side stream, {where}")
    m = fe.hex_elastic_3d(24)
    s = structure(64).scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind)
    x = fe.uniform_x(m.ncols, 8, seed=6)
    a = [dev(v) for v in (m.rowptr, m.colind, m.vals)]
    dx, y = dev(x), out(m.nrows, 8)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    if where == "host":
        eng = engine(s, m.vals, m.colind, stream=side)
    else:
        eng = engine.from_device(*a, stream=side)
    assert side.query()
    eng.launch(dx, y, cfg=SETS)
    assert np.array_equal(y.cpu().numpy(), O.csr_spmv(m.rowptr, m.colind, m.vals, x))
    eng.close()


@pytest.mark.parametrize("k", [5, 8, 9, 16])
def test_compensated_sums_on_request(k):
    """An FP32 engine asked for compensated sums on top of its default: the
    windows' sums, bit for bit, each row's in the same order."""
    say(f"[gpu] row sets, compensated sums k={k}")
    m = fe.hex_elastic_3d(7)
    s = structure(64).scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind)
    eng = engine(s, m.vals, m.colind, dtype="f32")
    assert eng.get_launch(k=k).accumulate == capi.WK_ACC_F64
    x = dev(fe.uniform_x(m.ncols, k, seed=8).astype(np.float32))
    y0, y1, y2, y3 = (out(m.nrows, k) for _ in range(4))
    eng.launch(x, y0, cfg=dict(OTHER, accumulate=capi.WK_ACC_TWOSUM))
    eng.launch(x, y1, cfg=dict(accumulate=capi.WK_ACC_TWOSUM))
    eng.launch(x, y2)
    eng.set_launch(dict(accumulate=capi.WK_ACC_TWOSUM), k=k)
    eng.launch(x, y3)
    a, b, c, d = (t.cpu().numpy() for t in (y0, y1, y2, y3))
    assert np.array_equal(a, b) and np.array_equal(a, d) and not np.array_equal(a, c)
    eng.close()
