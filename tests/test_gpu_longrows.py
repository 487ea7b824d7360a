"""Rows around the lengths at which a wavefront or a workgroup takes another chunk of 256 positions:
activities and propagation against the oracle, value for value, scanned and listed, with the rows
swept by wavefronts (the default) and by whole workgroups (longrow 64)."""
import numpy as np
import pytest

import scip_amd as sa
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

LENGTHS = [65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 319, 511, 512, 513, 767, 1023, 1024, 1025, 1280, 2047, 2049, 4100]


def long_instance(seed, extra, n):
    """Two rows of every length and `extra` short ones over n columns, planted."""
    rng = np.random.default_rng(seed)
    integral = (rng.random(n) < 0.4).astype(np.uint8)
    lb = np.where(integral, 0.0, -1e4 * rng.random(n))
    ub = np.where(integral, rng.integers(1, 1000, size=n).astype(float), 1e4 * rng.random(n))
    point = np.where(integral, np.floor(lb + (ub - lb) * rng.random(n)), lb + (ub - lb) * rng.random(n))
    free = (integral == 0) & (rng.random(n) < 0.002)
    ub[free] = 1e20
    rows = [np.sort(rng.choice(n, size=L, replace=False)) for L in 2 * LENGTHS + list(rng.integers(2, 20, size=extra))]
    col = np.concatenate(rows).astype(np.int32)
    ptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int64)
    val = 10.0 ** rng.uniform(-3, 3, size=len(col)) * rng.choice([-1.0, 1.0], size=len(col))
    act = np.add.reduceat(val * point[col], ptr[:-1])
    span = np.add.reduceat(np.abs(val) * np.minimum(ub - lb, 1e5)[col], ptr[:-1])
    side = span * rng.choice([0.002, 0.05, 0.3], size=len(rows))
    return sa.Instance(rowptr=ptr, colidx=col, vals=val, lhs=act - side, rhs=act + side, integral=integral, lb=lb, ub=ub)


# 60 and 40,000 short rows: the device holds every workgroup at once.  112,000 and 160,000: the tiles
# alone fill it (1,024 workgroups of four tiles), so the long rows' workgroups start first, with
# the tiles' in ascending and in descending order (1.3 and 1.9 tiles per wavefront); late rounds
# of these are listed (over 4,096 tiles, columns of low degree)
@pytest.mark.parametrize("extra", [60, 40_000, 112_000, 160_000])
@pytest.mark.parametrize("longrow", [1024, 64])
def test_long_rows(gpu_ctx, extra, longrow):
    print(f"[case] long rows extra={extra} longrow={longrow}", flush=True)
    inst = long_instance(7 + extra, extra, 5000 if extra <= 40_000 else 100_000)
    # lanes of four nonzeros, packed nearly without gaps into tiles of 64; 980 to 1,010 of the
    # workgroups are the tiles'
    length = np.diff(inst.rowptr)
    tiles = np.sum((length[length <= 64] + 3) // 4) / 64
    if extra == 112_000:
        assert tiles > 4 * 1024 and tiles / (4 * 980) < 1.7
    if extra == 160_000:
        assert 1.8 < tiles / (4 * 1010) and tiles / (4 * 980) < 1.95
    om = orc.OMatrix.from_instance(inst)
    ol, ou, orr = orc.propagate_jacobi(om, inst.lb, inst.ub)
    assert not orr["cutoff"] and orr["rounds"] >= 3
    ctx = sa.Context(0)
    ctx.set_tuning(longrow=longrow)
    mat = sa.Matrix(ctx, inst)
    for mode in (sa.SAP_MODE_DENSE, sa.SAP_MODE_SPARSE):
        b = sa.Bounds(mat, 1, mode)
        b.upload(inst.lb, inst.ub)
        st = b.propagate()
        gl, gu = b.download(0)
        assert np.array_equal(gl, ol) and np.array_equal(gu, ou)
        for k in ("rounds", "nchgbds", "rows_swept", "nnz_swept", "nrecompute"):
            assert st[k] == orr[k], (mode, k)
        b.close()
    got = mat.row_activities()
    want = orc.row_activities(om, inst.lb, inst.ub)
    for g, w in zip(got, want):
        assert np.array_equal(np.asarray(g).reshape(-1), np.asarray(w).reshape(-1))
    mat.close()
    ctx.close()
