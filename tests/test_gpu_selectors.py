"""Which kernel a launch configuration names (wk_launch stage_lds, read back by
wk_last_kernels): stage 6 is the row sets from three right-hand sides where the
layout has them and 8 never, 0 the column offsets and 9 never, and an explicit
configuration runs as given.  FP64 and FP64 sums against the oracle, zero
tolerance; compensated sums equal those of another kernel bit for bit."""
import sys

import numpy as np
import pytest

from oracle import pyoracle as O
from warpkernel_amd import _capi as capi
from warpkernel_amd import engine, fe, structure

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

BASE = dict(nontemporal=1, rows_per_lane=1, unroll=8, waves_per_block=1, k_tile=4, xcd_remap=1, blocks_per_cu=0)


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def out(rows, k):
    return torch.full((rows, k), float("nan"), dtype=torch.float64, device="cuda")


def scan(m):
    return structure(64).scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind)


def ran(launch, x, y, cfg):
    launch(x, y, cfg=cfg)
    return capi.lib().wk_last_kernels()


def windows(kernels):
    """The window kernel, with or without node windows for a rest of one column."""
    return kernels & ~capi.WK_KERNEL_NODES == capi.WK_KERNEL_WINDOWS


@pytest.mark.parametrize("k", [2, 3, 4, 5, 8, 9, 16, 32])
def test_stage_6_and_8_on_block_rows(k):
    """Elasticity, groups of 81 steps: both kernels, run, run_x and the residual."""
    say(f"[gpu] stages 6 and 8 k={k}")
    m = fe.hex_elastic_3d(7)
    s = scan(m)
    x, b = fe.uniform_x(m.ncols, k, seed=3), fe.uniform_x(m.nrows, k, seed=4)
    ref = O.csr_spmv(m.rowptr, m.colind, m.vals, x)
    perm = np.asarray(s.row_map)
    eng = engine(s, m.vals, m.colind, kr=True)
    want = {6: capi.WK_KERNEL_ROW_SETS if k >= 3 else capi.WK_KERNEL_REGISTERS, 8: capi.WK_KERNEL_REGISTERS}
    for stage in (6, 8):
        for wpb in (1, 4):
            cfg = dict(BASE, stage_lds=stage, waves_per_block=wpb)
            y = out(m.nrows, k)
            got = ran(eng.launch, dev(x), y, cfg)
            assert np.array_equal(y.cpu().numpy(), ref), cfg
            if k >= 4 or (k == 3 and stage == 6):  # (two, three: no whole tile of the register kernel)
                assert got & want[stage] and not got & ~want[stage] & (want[6] | want[8]), (cfg, got)
            else:
                assert not got & capi.WK_KERNEL_ROW_SETS
            y = out(m.nrows, k)
            eng.launch_x(dev(x[perm]), y, cfg=cfg)
            assert np.array_equal(y.cpu().numpy(), ref[perm]), (cfg, "run_x")
            eng.residual(dev(b), dev(x), y, cfg=cfg)
            assert np.array_equal(y.cpu().numpy(), b - ref), (cfg, "residual")
    eng.close()


@pytest.mark.parametrize("k", [8, 9, 16, 32])
def test_fp32_sums_and_stages(k):
    """FP32 values: stage 6 with compensated sums is the register kernel, as asked;
    compensated sums on top of the default are the windows'."""
    say(f"[gpu] FP32 stages k={k}")
    m = fe.hex_elastic_3d(7)
    eng = engine(scan(m), m.vals, m.colind, dtype="f32")
    xq = fe.uniform_x(m.ncols, k, seed=5).astype(np.float32)
    ref = O.csr_spmv(m.rowptr, m.colind, m.vals.astype(np.float32).astype(np.float64), xq.astype(np.float64))
    x, y0 = dev(xq), out(m.nrows, k)
    comp = dict(BASE, accumulate=capi.WK_ACC_TWOSUM)
    assert windows(ran(eng.launch, x, y0, dict(comp, stage_lds=4)))
    for stage in (6, 8):
        for wpb in (1, 2, 4):
            y = out(m.nrows, k)
            assert ran(eng.launch, x, y, dict(comp, stage_lds=stage, waves_per_block=wpb)) & capi.WK_KERNEL_REGISTERS
            assert torch.equal(y, y0), (stage, wpb)
    for cfg in (dict(accumulate=capi.WK_ACC_TWOSUM), dict(accumulate=capi.WK_ACC_TWOSUM, xcd_remap=0)):
        y = out(m.nrows, k)
        assert windows(ran(eng.launch, x, y, cfg)), cfg
        assert torch.equal(y, y0), cfg
    for stage, kernel in ((6, capi.WK_KERNEL_ROW_SETS), (8, capi.WK_KERNEL_REGISTERS)):
        y = out(m.nrows, k)
        assert ran(eng.launch, x, y, dict(comp, stage_lds=stage, accumulate=capi.WK_ACC_F64)) & kernel
        assert np.array_equal(y.cpu().numpy(), ref), stage
    eng.close()


@pytest.mark.parametrize("k", [4, 16, 32])
def test_registers_without_row_sets(k):
    """Rows of 37 to 84 steps that share no columns: the register kernel's long form."""
    say(f"[gpu] stage 6 without row sets k={k}")
    n = 700
    rng = np.random.default_rng(7)
    rows = [np.sort(rng.choice(np.arange(max(0, r - 60), min(n, r + 61)), 37 + r % 25, replace=False)) for r in range(n)]
    rp = np.concatenate([[0], np.cumsum([r.size for r in rows])]).astype(np.int32)
    ci = np.concatenate(rows).astype(np.int32)
    m = fe.CSR("long", n, n, rp, ci, rng.uniform(-1, 1, ci.size))
    s = scan(m)
    x = fe.uniform_x(n, k, seed=6)
    for dtype in ("f64", "f32"):
        eng = engine(s, m.vals, m.colind, dtype=dtype)
        dt = np.float64 if dtype == "f64" else np.float32
        v, xq = m.vals.astype(dt).astype(np.float64), x.astype(dt)
        y = out(n, k)
        got = ran(eng.launch, dev(xq), y, dict(BASE, stage_lds=6, accumulate=capi.WK_ACC_F64))
        assert got & capi.WK_KERNEL_REGISTERS if k * dt().itemsize >= 32 else got == capi.WK_KERNEL_WINDOWS
        assert np.array_equal(y.cpu().numpy(), O.csr_spmv(rp, ci, v, xq.astype(np.float64)))
        eng.close()


def test_stage_0_and_9():
    say("[gpu] stages 0 and 9")
    m = fe.tet_poisson_3d(9)
    eng = engine(scan(m), m.vals, m.colind)
    x = fe.uniform_x(m.ncols, seed=8)
    ref = O.csr_spmv(m.rowptr, m.colind, m.vals, x)
    for stage, unroll, nt, kernel in ((0, 8, 1, capi.WK_KERNEL_OFFSETS), (0, 16, 1, capi.WK_KERNEL_OFFSETS),
                                      (9, 8, 1, capi.WK_KERNEL_DIRECT), (9, 16, 1, capi.WK_KERNEL_DIRECT),
                                      (0, 8, 2, capi.WK_KERNEL_DIRECT)):
        y = torch.full((m.nrows,), float("nan"), dtype=torch.float64, device="cuda")
        cfg = dict(BASE, k_tile=1, stage_lds=stage, unroll=unroll, nontemporal=nt)
        assert ran(eng.launch, dev(x), y, cfg) == kernel, cfg
        assert np.array_equal(y.cpu().numpy(), ref), cfg
    for stage in (-1, 10):
        with pytest.raises(capi.WKError) as e:
            eng.launch(dev(x), y, cfg=dict(BASE, k_tile=1, stage_lds=stage))
        assert e.value.code == capi.WK_ERR_ARG
    eng.close()


@pytest.mark.parametrize("nodes", [60, 175000])
def test_fp32_default_sums_do_not_depend_on_the_size(nodes):
    """8,204 groups as one: FP64 sums from five right-hand sides where rows share
    their columns, compensated ones below."""
    say(f"[gpu] FP32 default sums, {nodes} nodes")
    n = 3 * nodes
    node = np.arange(nodes)
    nb = np.sort(np.stack([node, (node + 1) % nodes], 1), 1)
    ci = np.repeat((nb[:, :, None] * 3 + np.arange(3)).reshape(nodes, 6), 3, 0).reshape(-1).astype(np.int32)
    m = fe.CSR("pairs", n, n, (6 * np.arange(n + 1)).astype(np.int32), ci,
               np.random.default_rng(1).uniform(-1, 1, ci.size))
    eng = engine(scan(m), m.vals, m.colind, dtype="f32")
    v = m.vals.astype(np.float32).astype(np.float64)
    for k in (4, 5, 8, 9):
        assert eng.get_launch(k=k).accumulate == (capi.WK_ACC_F64 if k >= 5 else capi.WK_ACC_TWOSUM), k
        xq = fe.uniform_x(n, k, seed=9).astype(np.float32)
        y = out(n, k)
        eng.launch(dev(xq), y)
        if k >= 5:
            assert np.array_equal(y.cpu().numpy(), O.csr_spmv(m.rowptr, ci, v, xq.astype(np.float64))), k
        eng.launch(dev(xq), y, cfg=dict(accumulate=capi.WK_ACC_TWOSUM))
        other = out(n, k)
        eng.launch(dev(xq), other, cfg=dict(BASE, stage_lds=4, accumulate=capi.WK_ACC_TWOSUM))
        assert torch.equal(y, other), k
    eng.close()


@pytest.mark.parametrize("dof,nodes,k,sets", [(2, 20800, 5, False), (2, 20800, 16, True), (2, 3200, 5, True),
                                              (3, 44800, 8, False), (4, 11200, 5, True)])
def test_default_on_short_block_rows(dof, nodes, k, sets):
    """One dof x dof block a node, and two for dof 2: the row sets where they pay."""
    say(f"[gpu] default, dof {dof}, {nodes} nodes, k={k}")
    n, w = dof * nodes, 2 if dof == 2 else 1
    node = np.arange(nodes)
    nb = np.sort(np.stack([(node + i) % nodes for i in range(w)], 1), 1)
    ci = np.repeat((nb[:, :, None] * dof + np.arange(dof)).reshape(nodes, -1), dof, 0).reshape(-1).astype(np.int32)
    m = fe.CSR("short", n, n, (w * dof * np.arange(n + 1)).astype(np.int32), ci,
               np.random.default_rng(1).uniform(-1, 1, ci.size))
    x = fe.uniform_x(n, k, seed=9)
    for dtype in ("f64", "f32"):
        dt = np.float64 if dtype == "f64" else np.float32
        v, xq = m.vals.astype(dt), x.astype(dt)
        eng = engine(scan(m), m.vals, m.colind, dtype=dtype)
        y = out(n, k)
        got = ran(eng.launch, dev(xq), y, None)
        assert bool(got & capi.WK_KERNEL_ROW_SETS) == sets, (dtype, got)
        assert np.array_equal(y.cpu().numpy(), O.csr_spmv(m.rowptr, ci, v.astype(np.float64), xq.astype(np.float64)))
        eng.close()


@pytest.mark.parametrize("groups,lens,kernel", [
    (1280, [39], capi.WK_KERNEL_PACKED), (313, [39], capi.WK_KERNEL_OFFSETS), (1280, [16], capi.WK_KERNEL_OFFSETS),
    (2304, [20], capi.WK_KERNEL_PACKED), (1280, [1, 3, 9, 17, 33, 39], capi.WK_KERNEL_PACKED),
    (1280, [1, 3, 9, 17], capi.WK_KERNEL_OFFSETS)])
def test_default_on_bands(groups, lens, kernel):
    """One right-hand side on bands of random columns: column offsets or x windows."""
    say(f"[gpu] default on bands, {groups} groups, {lens}")
    n = 64 * groups
    rng = np.random.default_rng(3)
    cnt = np.asarray(lens)[np.arange(n) % len(lens)]
    rows = np.repeat(np.arange(n), cnt)
    cols = np.clip(rows + rng.integers(-30, 31, rows.size), 0, n - 1)
    ci = cols[np.lexsort((cols, rows))].astype(np.int32)
    m = fe.CSR("band", n, n, np.concatenate([[0], np.cumsum(cnt)]).astype(np.int32), ci, rng.uniform(-1, 1, ci.size))
    x = fe.uniform_x(n, seed=2)
    eng = engine(scan(m), m.vals, m.colind)
    y = torch.full((n,), float("nan"), dtype=torch.float64, device="cuda")
    assert ran(eng.launch, dev(x), y, None) == kernel
    assert np.array_equal(y.cpu().numpy(), O.csr_spmv(m.rowptr, ci, m.vals, x))
    eng.close()


def test_default_where_row_sets_do_not_reach():
    """x as eight columns of an array of more than 4 GiB: the windows' choice."""
    say("[gpu] default on columns of a wide array")
    m = fe.hex_elastic_3d(7)
    k = 8
    x = fe.uniform_x(m.ncols, k, seed=3)
    eng = engine(scan(m), m.vals, m.colind)
    wide = torch.empty((m.ncols, (1 << 32) // (8 * m.ncols) + 1), dtype=torch.float64, device="cuda")
    wide[:, 5:5 + k] = dev(x)
    near = torch.empty((m.ncols, 2 * k), dtype=torch.float64, device="cuda")
    near[:, :k] = dev(x)
    ref = O.csr_spmv(m.rowptr, m.colind, m.vals, x)
    for xd, sets in ((wide[:, 5:5 + k], False), (near[:, :k], True)):
        y = out(m.nrows, k)
        got = ran(eng.launch, xd, y, None)
        assert got == capi.WK_KERNEL_ROW_SETS if sets else windows(got), got
        assert np.array_equal(y.cpu().numpy(), ref)
    eng.close()


def test_layouts_that_have_offsets_and_row_sets():
    """The layouts of test_gpu_deltas and test_gpu_rowsets hold what they are there
    for, also where the rows do not fill the last group."""
    say("[gpu] offsets and row sets are there")
    from test_gpu_deltas import CASES as BANDS
    from test_gpu_rowsets import CASES as BLOCKS
    for name, make in BANDS.items():
        m = make()
        eng = engine(scan(m), m.vals, m.colind)
        y = torch.empty(m.nrows, dtype=torch.float64, device="cuda")
        want = capi.WK_KERNEL_DIRECT if name == "too_wide" else capi.WK_KERNEL_OFFSETS
        assert ran(eng.launch, dev(fe.uniform_x(m.ncols)), y, dict(BASE, k_tile=1, stage_lds=0)) == want, name
        eng.close()
    for name, make in BLOCKS.items():
        m = make()
        eng = engine(scan(m), m.vals, m.colind)
        got = ran(eng.launch, dev(fe.uniform_x(m.ncols, 8)), out(m.nrows, 8), dict(BASE, stage_lds=6))
        say(name, got)
        assert (got == capi.WK_KERNEL_ROW_SETS) == (name != "long"), (name, got)
        eng.close()
