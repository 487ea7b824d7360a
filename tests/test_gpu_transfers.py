"""Host bound arrays to the device and back at the sizes where their route changes: one chunk of
32,768 columns (staged in one piece, read back with the call's own wait), two and more chunks
(copied out by helper threads), more chunks than there are slots.  Every value comes back as it
was, a NaN anywhere is refused and changes nothing, and the calls on host arrays agree with the
oracle's Jacobi twin."""
import os
import threading
import time

import numpy as np
import pytest

import scip_amd as sa
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

SIZES = [1, 32_767, 32_768, 32_769, 65_537, 98_304, 262_144, 262_145, 300_001]


@pytest.mark.parametrize("ncols", SIZES)
def test_round_trip(gpu_ctx, ncols):
    print(f"[case] transfer ncols={ncols}", flush=True)
    rng = np.random.default_rng(ncols)
    inst = sa.Instance(rowptr=np.array([0, 1], np.int64), colidx=np.array([ncols - 1], np.int32), vals=np.ones(1),
                       lhs=np.array([-1e20]), rhs=np.array([1e20]), integral=np.zeros(ncols, np.uint8),
                       lb=-rng.random(ncols), ub=rng.random(ncols))
    inst.lb[0] = -1e20
    mat = sa.Matrix(gpu_ctx, inst)
    b = sa.Bounds(mat, 2)
    b.upload(inst.lb, inst.ub)
    b.upload(inst.lb - 1.0, inst.ub + 1.0, v=1)   # the staging of the first upload is free again
    for v, off in ((0, 0.0), (1, 1.0)):
        lb, ub = b.download(v)
        assert np.array_equal(lb, inst.lb - off) and np.array_equal(ub, inst.ub + off), v
    for at in {0, ncols // 2, ncols - 1}:
        for side in (0, 1):
            bad = [inst.lb + 5.0, inst.ub + 5.0]
            bad[side][at] = np.nan
            with pytest.raises(sa.SapError) as e:
                b.upload(*bad, v=0)
            assert e.value.rc == sa.SAP_INVALIDDATA
            with pytest.raises(sa.SapError):
                mat.propagate(*bad)
    lb, ub = b.download(0)
    assert np.array_equal(lb, inst.lb) and np.array_equal(ub, inst.ub)
    b.close()
    mat.close()


def boxes(ncols):
    rng = np.random.default_rng(ncols)
    return sa.Instance(rowptr=np.array([0, 1], np.int64), colidx=np.array([ncols - 1], np.int32), vals=np.ones(1),
                       lhs=np.array([-1e20]), rhs=np.array([1e20]), integral=np.zeros(ncols, np.uint8),
                       lb=-rng.random(ncols), ub=rng.random(ncols))


@pytest.mark.parametrize("ncols", [1, 257, 32_768, 32_769])
def test_all_vectors(gpu_ctx, ncols):
    # one pair of arrays into every vector of a set
    print(f"[case] upload into all vectors ncols={ncols}", flush=True)
    inst = boxes(ncols)
    mat = sa.Matrix(gpu_ctx, inst)
    b = sa.Bounds(mat, 67)
    b.upload(inst.lb - 2.0, inst.ub + 2.0)
    b.upload(inst.lb, inst.ub, v=33)
    for v in (0, 1, 32, 33, 34, 66):
        off = 0.0 if v == 33 else 2.0
        lb, ub = b.download(v)
        assert np.array_equal(lb, inst.lb - off) and np.array_equal(ub, inst.ub + off), v
    b.close()
    mat.close()


def test_all_vectors_cost(gpu_ctx):
    # the vectors are filled on the device, whichever way the arrays came there: on the two sides of
    # the line between the routes an upload into many vectors takes about as long
    took = []
    for ncols in (32_000, 33_000):
        print(f"[case] upload into 256 vectors ncols={ncols}", flush=True)
        inst = boxes(ncols)
        mat = sa.Matrix(gpu_ctx, inst)
        b = sa.Bounds(mat, 256)
        t = []
        for _ in range(20):
            t0 = time.perf_counter()
            b.upload(inst.lb, inst.ub)
            t.append(time.perf_counter() - t0)
        took.append(min(t))
        b.close()
        mat.close()
    assert took[0] < 2.0 * took[1], took


@pytest.mark.parametrize("ncols", [32_768, 32_769, 262_145])
def test_calls(gpu_ctx, ncols):
    print(f"[case] calls ncols={ncols}", flush=True)
    inst = sa.gen_mixed(ncols // 4, ncols, seed=ncols % 97, planted=True)
    ol, ou, orr = orc.propagate_jacobi(orc.OMatrix.from_instance(inst), inst.lb, inst.ub)
    assert not orr["cutoff"] and orr["nchgbds"] > 1024   # more than the history entries that come with the bounds
    mat = sa.Matrix(gpu_ctx, inst)
    for flags in (0, sa.SAP_FLAG_HOSTLOOP):
        lb, ub, st = mat.propagate(params=sa.default_params(flags=flags))
        assert np.array_equal(lb, ol) and np.array_equal(ub, ou) and st["rounds"] == orr["rounds"]
    r = mat.propagate_reasons()
    assert np.array_equal(r["lb"], ol) and np.array_equal(r["ub"], ou) and r["nhist"] == orr["nchgbds"]
    r = mat.propagate_reasons(ol, ou)   # nothing left to do: an empty history
    assert np.array_equal(r["lb"], ol) and np.array_equal(r["ub"], ou) and r["nhist"] == 0
    mat.close()
    # packed: instance 0 changes, instance 1 is at its fixpoint, instance 2 has no rows
    done = sa.Instance(**{**inst.__dict__, "lb": ol, "ub": ou})
    none = sa.Instance(rowptr=np.zeros(1, np.int64), colidx=np.zeros(0, np.int32), vals=np.zeros(0), lhs=np.zeros(0),
                       rhs=np.zeros(0), integral=np.zeros(7, np.uint8), lb=np.zeros(7), ub=np.ones(7))
    packed = sa.PackedMatrix(gpu_ctx, [inst, done, none])
    lb, ub, res, rnd, _ = packed.propagate_packed()
    assert res.tolist() == [sa.SAP_REDUCEDDOM, sa.SAP_DIDNOTFIND, sa.SAP_DIDNOTFIND]
    assert rnd[0] == orr["rounds"]
    assert np.array_equal(lb, np.concatenate([ol, ol, none.lb])) and np.array_equal(ub, np.concatenate([ou, ou, none.ub]))
    packed.close()


def test_many_calls(gpu_ctx):
    # more calls than the redundant-row generations (255) on one matrix: the calls that start the
    # generations again take the bounds over apart from the reset
    inst = sa.gen_covering_packing(40, 60, 8, seed=3)
    mat = sa.Matrix(gpu_ctx, inst)
    om = orc.OMatrix.from_instance(inst)
    rng = np.random.default_rng(4)
    print("[case] 520 calls on one matrix", flush=True)
    for _ in range(520):
        lb, ub = inst.lb.copy(), inst.ub.copy()
        j = rng.choice(60, size=4, replace=False)
        lb[j[:2]], ub[j[2:]] = 1.0, 0.0
        ol, ou, orr = orc.propagate_jacobi(om, lb, ub)
        gl, gu, st = mat.propagate(lb, ub)
        assert (st["result"] == sa.SAP_CUTOFF) == bool(orr["cutoff"])
        if not orr["cutoff"]:
            assert np.array_equal(gl, ol) and np.array_equal(gu, ou) and st["nchgbds"] == orr["nchgbds"]
        else:
            assert np.array_equal(gl, lb) and np.array_equal(gu, ub)
    mat.close()


def test_helper_threads_keep_to_the_affinity(gpu_ctx):
    # a caller confined to one CPU gets no helper threads, and the same values
    inst = boxes(600_001)
    mat = sa.Matrix(gpu_ctx, inst)
    b = sa.Bounds(mat, 1)
    b.upload(inst.lb, inst.ub)
    b.download()
    go, end, wrong = threading.Event(), threading.Event(), []

    def caller():
        os.sched_setaffinity(0, {min(os.sched_getaffinity(0))})   # this thread only
        go.wait(60)
        while not end.is_set():
            b.upload(inst.lb, inst.ub)
            lb, ub = b.download()
            if not (np.array_equal(lb, inst.lb) and np.array_equal(ub, inst.ub)):
                wrong.append(1)

    print("[case] transfers of a caller on one CPU", flush=True)
    t = threading.Thread(target=caller)
    t.start()
    time.sleep(0.2)
    threads = len(os.listdir("/proc/self/task"))
    go.set()
    until, most = time.perf_counter() + 1.0, 0
    while time.perf_counter() < until:
        most = max(most, len(os.listdir("/proc/self/task")))
    end.set()
    t.join(60)
    b.close()
    mat.close()
    assert not wrong and most == threads, (most, threads)
