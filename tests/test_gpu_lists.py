"""Rounds swept from row lists in dense bound sets, at the sizes where the lists end: one column
of very high degree is fixed, so that few changed columns mark many rows (more than a row list
holds) and these touch many columns (more than the touched list holds).  Against the oracle's
Jacobi twin: bit-exact bounds, verdicts, rounds and counts."""
import time

import numpy as np
import pytest

import scip_amd as sa
from oracle import oracle as orc
from tests.test_zz_no_alloc import DeviceArray

pytestmark = pytest.mark.gpu


# a tile of the sweep holds at most 256 nonzeros, and only sets of many tiles list rows: with these
# rows beside them (64 of 1,000 further columns each, never binding) 4,375 tiles at least
IDLE = 17_500


def star(n, force, idle=0):
    """x0 + y_i + y_(i+1) <= 1 over binaries for i = 1..n, then (force) the row x0 >= 1: its round
    changes one column, whose n rows then fix every y; then rows that never change anything."""
    rows = n + (1 if force else 0) + idle
    length = np.concatenate([np.full(n, 3), [1] if force else [], np.full(idle, 64)]).astype(np.int64)
    rowptr = np.concatenate([[0], np.cumsum(length)]).astype(np.int64)
    i = np.arange(1, n + 1)
    colidx = np.stack([np.zeros(n, np.int64), i, i + 1], 1).reshape(-1)
    rest = n + 2 + np.sort((np.arange(64) * 15 + np.arange(idle)[:, None]) % 1000, axis=1).reshape(-1)
    colidx = np.concatenate([colidx, [0] if force else [], rest]).astype(np.int32)
    lhs, rhs = np.full(rows, -1e20), np.full(rows, 1.0)
    if force:
        lhs[n], rhs[n] = 1.0, 1e20
    rhs[rows - idle:] = 100.0
    cols = n + 2 + (1000 if idle else 0)
    return sa.Instance(rowptr=rowptr, colidx=colidx, vals=np.ones(len(colidx)), lhs=lhs, rhs=rhs,
                       integral=np.ones(cols, dtype=np.uint8), lb=np.zeros(cols), ub=np.ones(cols))


# rows of one length bin and touched columns: within every list; beyond the no-allocation
# entry point's lists (2^15); beyond the touched list (2^16); beyond a row list (2^17)
@pytest.mark.parametrize("n", [32_700, 33_000, 70_000, 131_000, 135_000])
def test_lists_end(gpu_ctx, n):
    print(f"[case] lists n={n}", flush=True)
    inst = star(n, force=True, idle=IDLE)
    ol, ou, orr = orc.propagate_jacobi(orc.OMatrix.from_instance(inst), inst.lb, inst.ub)
    assert not orr["cutoff"] and orr["rounds"] == 3 and orr["nchgbds"] == n + 2
    mat = sa.Matrix(gpu_ctx, inst)
    lb, ub, st = mat.propagate()
    assert np.array_equal(lb, ol) and np.array_equal(ub, ou)
    assert (st["rounds"], st["nchgbds"], st["rows_swept"]) == (orr["rounds"], orr["nchgbds"], orr["rows_swept"])
    dl, du = DeviceArray(inst.lb), DeviceArray(inst.ub)
    st = mat.propagate_device_noalloc(dl.data_ptr(), du.data_ptr())
    assert np.array_equal(dl.numpy(), ol) and np.array_equal(du.numpy(), ou)
    assert (st["rounds"], st["nchgbds"], st["rows_swept"]) == (orr["rounds"], orr["nchgbds"], orr["rows_swept"])
    dl.free()
    du.free()
    mat.close()


@pytest.mark.parametrize("n", [70_000, 135_000])
def test_lists_end_from_overlays(gpu_ctx, n):
    # the same rows marked by a node's overlay, next to a node with a single marked row pair and
    # one that is cut off, in one dense set; then again on the same set
    print(f"[case] lists from overlays n={n}", flush=True)
    inst = star(n, force=False, idle=IDLE)
    mat = sa.Matrix(gpu_ctx, inst)
    base = sa.Bounds(mat, 1)
    base.upload(inst.lb, inst.ub)
    nodes = sa.Bounds(mat, 3, sa.SAP_MODE_DENSE)
    p = sa.default_params(flags=sa.SAP_FLAG_BASE_IS_FIXPOINT)
    for _ in range(2):
        out = nodes.propagate_nodes(base, 0, [0, 1, 2, 4], [0, 5, 7, 8], [1.0] * 4, [1.0] * 4, params=p,
                                    chgcap=2 * n + 64)
        assert out["result"].tolist() == [sa.SAP_REDUCEDDOM, sa.SAP_REDUCEDDOM, sa.SAP_CUTOFF]
        assert out["rounds"][:2].tolist() == [2, 2]
        a, b, c = out["chgptr"][1:].tolist()
        assert np.array_equal(out["chgcol"][:a], np.arange(1, n + 2)) and np.all(out["chgub"][:a] == 0.0)
        assert out["chgcol"][a:b].tolist() == [0, 4, 6] and np.all(out["chgub"][a:b] == 0.0) and b == c
    nodes.close()
    base.close()
    mat.close()


# a dense set that never lists from marking: the rows of the overlay columns are shared out over the
# workgroup; around one pass of 256 rows, and a column so long that one thread walking it would
# be a chain of thousands of steps
@pytest.mark.parametrize("n", [255, 256, 257, 40_000])
def test_long_overlay_column(gpu_ctx, n):
    print(f"[case] long overlay column n={n}", flush=True)
    inst = star(n, force=False)
    om = orc.OMatrix.from_instance(inst)
    mat = sa.Matrix(gpu_ctx, inst)
    base = sa.Bounds(mat, 1)
    base.upload(inst.lb, inst.ub)
    nodes = sa.Bounds(mat, 1, sa.SAP_MODE_DENSE)   # at most 21 rows of three to a tile: 1,905 tiles
    p = sa.default_params(flags=sa.SAP_FLAG_BASE_IS_FIXPOINT)
    for c, x in (([0], [1.0]), ([2], [1.0]), ([0, 7, n], [0.0, 1.0, 1.0]), ([0, 9], [1.0, 1.0])):
        out = nodes.propagate_nodes(base, 0, [0, len(c)], c, x, x, params=p, chgcap=n + 64)
        lb, ub = inst.lb.copy(), inst.ub.copy()
        lb[c] = ub[c] = x
        ol, ou, orr = orc.propagate_jacobi(om, lb, ub)
        assert (out["result"][0] == sa.SAP_CUTOFF) == bool(orr["cutoff"]) == (c == [0, 9])
        if not orr["cutoff"]:
            lb[out["chgcol"]], ub[out["chgcol"]] = out["chglb"], out["chgub"]
            assert np.array_equal(lb, ol) and np.array_equal(ub, ou), c
    if n == 40_000:
        # 40,000 tags by 256 threads are 157 steps of under 1 us; a call takes about 100 us without them
        def best(col):
            t = []
            for _ in range(20):
                t0 = time.perf_counter()
                nodes.propagate_nodes(base, 0, [0, 1], [col], [0.0], [0.0], params=p, chgcap=64)
                t.append(time.perf_counter() - t0)
            return min(t)
        short, long = best(5), best(0)
        assert long < 10 * short, (short, long)
    nodes.close()
    base.close()
    mat.close()


def test_clustered_changes(gpu_ctx):
    # which rounds are listed follows from how many columns changed, not from where they are: a system
    # with its changing columns first, last and spread, and the time of a call on each
    inst = sa.gen_mixed(130_000, 65_000, seed=11, planted=True)   # 65,536 columns: one workgroup a counter
    mat = sa.Matrix(gpu_ctx, inst)
    lb, ub, st = mat.propagate()
    mat.close()
    changed = (lb != inst.lb) | (ub != inst.ub)
    row = np.repeat(np.arange(inst.nrows), np.diff(inst.rowptr))
    took = {}
    for name, order in (("spread", np.random.default_rng(1).permutation(inst.ncols)),
                        ("first", np.argsort(~changed, kind="stable")), ("last", np.argsort(changed, kind="stable"))):
        print(f"[case] changed columns {name}", flush=True)
        at = np.empty_like(order)
        at[order] = np.arange(inst.ncols)
        col = at[inst.colidx].astype(np.int32)
        o = np.lexsort((col, row))
        one = sa.Instance(rowptr=inst.rowptr, colidx=col[o], vals=inst.vals[o], lhs=inst.lhs, rhs=inst.rhs,
                          integral=inst.integral[order], lb=inst.lb[order], ub=inst.ub[order])
        ol, ou, orr = orc.propagate_jacobi(orc.OMatrix.from_instance(one), one.lb, one.ub)
        mat = sa.Matrix(gpu_ctx, one)
        root, work = sa.Bounds(mat, 1, sa.SAP_MODE_DENSE), sa.Bounds(mat, 1, sa.SAP_MODE_DENSE)
        root.upload(one.lb, one.ub)
        ms = []
        for _ in range(20):
            work.copy_from(root)
            st = work.propagate()
            ms.append(st["device_ms"])
        gl, gu = work.download()
        assert np.array_equal(gl, ol) and np.array_equal(gu, ou)
        assert st["rounds"] == orr["rounds"] and st["nchgbds"] == orr["nchgbds"]
        took[name] = min(ms)
        work.close()
        root.close()
        mat.close()
    # the same rows are swept in the same rounds; what may differ is how the gathers fall into cache lines
    assert max(took["first"], took["last"]) < 1.3 * took["spread"], took


# more columns than one pass of the marking takes (2^20), few enough tiles that the set never lists
@pytest.mark.parametrize("ncols", [1_048_576, 1_048_577, 1_100_003])
def test_many_columns(gpu_ctx, ncols):
    print(f"[case] many columns ncols={ncols}", flush=True)
    part = sa.gen_mixed(3000, 3000, seed=5, planted=True)
    at = np.linspace(0, ncols - 1, 3000).astype(np.int64)
    whole = {}
    for k, fill in (("lb", 0.0), ("ub", 1.0), ("integral", 0)):
        whole[k] = np.full(ncols, fill, dtype=getattr(part, k).dtype)
        whole[k][at] = getattr(part, k)
    inst = sa.Instance(rowptr=part.rowptr, colidx=at[part.colidx].astype(np.int32), vals=part.vals, lhs=part.lhs,
                       rhs=part.rhs, **whole)
    ol, ou, orr = orc.propagate_jacobi(orc.OMatrix.from_instance(inst), inst.lb, inst.ub)
    assert not orr["cutoff"] and orr["rounds"] >= 3
    mat = sa.Matrix(gpu_ctx, inst)
    b = sa.Bounds(mat, 1, sa.SAP_MODE_DENSE)
    b.upload(inst.lb, inst.ub)
    st = b.propagate()
    gl, gu = b.download()
    assert np.array_equal(gl, ol) and np.array_equal(gu, ou)
    assert (st["rounds"], st["nchgbds"], st["rows_swept"]) == (orr["rounds"], orr["nchgbds"], orr["rows_swept"])
    b.close()
    mat.close()
