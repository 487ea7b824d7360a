"""The propagation work that users of this engine have it do, as cases that can be timed.

Every case is one call sequence of the public Python entry points (which are the C ABI's, one
for one) on an instance made from a seed:

  plain     sap_propagate: host bounds in, host bounds out
  reasons   sap_propagate_reasons: the SCIP plugin's call at a node of the tree
  resident  the root bounds copied on the device and propagated there, then read back
  device    sap_propagate_device_noalloc: bounds in tensors of the caller
  nodes     sap_propagate_nodes: node bound vectors as overlays on a resident root fixpoint
  probe     sap_probe: both branches of many binaries
  split     sap_probe_split: the propagation part of strong branching
  packed    sap_propagate_packed: many instances in one matrix, host bounds in and out
  serve     sap_server_replay: node requests of several resident problems, continuously batched

Two families of instances: "cover" (covering and packing rows over binaries, 10 nonzeros a row)
and "mixed" (log-normal or uniform row lengths, 40 % integer columns, coefficients of magnitude
10^U[-3,3], two-sided rows); the sides of a mixed instance are centred on a hidden feasible
point (planted) or on the middle of the activity span (above ~10^4 rows usually infeasible).
"""
from __future__ import annotations

import math

import numpy as np
import torch

import scip_amd as sa

FIXPOINT = sa.SAP_FLAG_BASE_IS_FIXPOINT


def listed():
    return [
        # a node of one small pure-binary problem, host bounds in and out: launches and waits count
        dict(name="plain_cover_2k", kind="plain", family="cover", rows=2_000, cols=5_000, node=20),
        # presolving's root propagation of a middle-sized problem (PROPPRESOL)
        dict(name="plain_mixed_100k", kind="plain", family="mixed", rows=100_003, cols=120_011, planted=True, node=0),
        # the large instance propagated to its fixpoint, host bounds in and out
        dict(name="plain_mixed_1m", kind="plain", family="mixed", rows=1_000_000, cols=1_000_000, planted=True, node=0),
        # a node of the tree as the SCIP plugin propagates it by default (PROPEXEC): the root
        # fixpoint plus the node's branchings, ranged rows on, a reason for every change
        dict(name="reasons_mixed_30k", kind="reasons", family="mixed", rows=30_011, cols=25_013, node=12),
        # the same instance from root bounds resident in HBM, where its fixpoint stays as the base
        # of node calls; the fixpoint is also read back for branching
        dict(name="resident_mixed_1m", kind="resident", family="mixed", rows=1_000_000, cols=1_000_000),
        # bounds already in the caller's device tensors, no allocation allowed
        dict(name="device_mixed_300k", kind="device", family="mixed", rows=300_007, cols=450_001),
        # 1,024 open nodes of one tree, each fixing 1..50 binaries, in one call
        dict(name="nodes_cover_1024", kind="nodes", family="cover", rows=200_000, cols=300_000, nvec=1024),
        # one node at a time from a resident fixpoint: the latency of a small change
        dict(name="nodes_mixed_1", kind="nodes", family="mixed", rows=100_003, cols=90_001, nvec=1),
        # presolve probing: 8,192 binaries, 2,048 branch vectors per launch
        dict(name="probe_cover_8k", kind="probe", family="cover", rows=200_000, cols=300_000, nvec=2048, nprobe=8192),
        # strong branching: both children of 100 candidates of a mixed problem
        dict(name="split_mixed_20k", kind="split", family="mixed", rows=20_011, cols=30_013, nvec=200, nprobe=100),
        # 24 independent instances of 500 to 60,000 rows propagated together
        dict(name="packed_24", kind="packed", family="mixed", count=24, most=60_000),
        # 2,000 waiting node requests, half of one covering problem, half of four mixed ones
        dict(name="serve_2k", kind="serve", family="cover", rows=50_000, cols=75_000, slots=64, requests=2000, others=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed kinds, sizes uniform in their logarithm."""
    kind = rng.choice(["plain", "plain", "plain", "reasons", "resident", "device", "nodes", "nodes", "probe", "split",
                       "packed", "serve"])
    family = rng.choice(["cover", "mixed"])
    most = {"plain": 600_000, "resident": 900_000, "reasons": 100_000, "device": 600_000}.get(kind, 200_000)
    rows = _log(rng, 700, most)
    cols = max(400, int(rows * rng.uniform(0.7, 1.6))) if family == "mixed" else int(rows * rng.uniform(1.4, 2.5)) | 1
    c = dict(kind=kind, family=family, rows=rows, cols=cols)
    if kind == "plain" and family == "cover":
        c["node"] = rng.randrange(1, 50)
    elif kind == "plain":
        c.update(planted=rng.random() < 0.8, node=rng.choice([0, 0, rng.randrange(1, 30)]),
                 ranged=rng.random() < 0.3, tighten=rng.random() < 0.85)
        if c["ranged"]:
            c.update(rows=min(rows, 60_000), cols=min(cols, 60_000))
        c["node"] = c["node"] if c["planted"] else 0
    elif kind in ("reasons", "device", "split", "packed"):
        c["family"] = "mixed"
        c["cols"] = max(400, int(rows * rng.uniform(0.7, 1.6)))
        if kind == "reasons":
            c["node"] = rng.randrange(0, 30)
    elif kind == "resident":
        c["family"] = "mixed"
        c["cols"] = max(400, int(rows * rng.uniform(0.7, 1.6)))
    if kind == "nodes":
        c["nvec"] = _log(rng, 1, 1024)
        if family == "mixed":
            c.update(rows=min(rows, 80_000), cols=min(cols, 80_000), nvec=min(c["nvec"], 300))
    elif kind == "probe":
        c.update(family="cover", cols=int(rows * rng.uniform(1.4, 2.5)) | 1, nvec=2 * _log(rng, 8, 1024))
        c["nprobe"] = min(_log(rng, 20, 8000), c["cols"] // 2)
    elif kind == "split":
        c.update(rows=min(rows, 50_000), cols=min(c["cols"], 60_000), nprobe=_log(rng, 5, 100))
        c["nvec"] = 2 * rng.randrange(max(1, c["nprobe"] // 2), c["nprobe"] + 1)
    elif kind == "packed":
        c = dict(kind=kind, family="mixed", count=rng.randrange(3, 25), most=_log(rng, 2_000, 60_000))
    elif kind == "serve":
        c.update(family="cover", rows=min(rows, 50_000), cols=min(rows, 50_000) * 3 // 2, slots=rng.choice([16, 33, 64]),
                 requests=_log(rng, 200, 2000), others=rng.randrange(1, 5))
    return c


# ---- instances -----------------------------------------------------------------------------
def mixed(rows, cols, seed, planted, uniform=None):
    """A mixed instance: row lengths log-normal (median 8, sigma 1, at most 10,000) or uniform in
    a range, distinct ascending columns in each row, sides at 0.3 of the row's finite span
    around the activity of a hidden feasible point or around the middle of the span."""
    dev = "cuda"
    g = torch.Generator(device=dev)
    g.manual_seed(seed)

    def u(n):
        return torch.rand(n, generator=g, device=dev, dtype=torch.float64)

    if uniform is None:
        length = torch.exp(math.log(8.0) + torch.randn(rows, generator=g, device=dev, dtype=torch.float64)).round().long()
        length = length.clamp(1, 10_000)
    else:
        length = (uniform[0] + (u(rows) * (uniform[1] - uniform[0] + 1)).long()).clamp(max=uniform[1])
    length = length.clamp(max=cols)
    row = torch.repeat_interleave(torch.arange(rows, device=dev), length)
    key = torch.unique(row * cols + (u(len(row)) * cols).long().clamp(max=cols - 1))   # sorted, without repeats
    row, col = key // cols, key % cols
    integral = u(cols) < 0.4
    top = (1 + (u(cols) * 1000).long()).clamp(max=1000).double()
    lb = torch.where(integral, 0.0, -1e4 * u(cols))
    ub = torch.where(integral, top, 1e4 * u(cols))
    open_side = u(cols)
    lb = torch.where(~integral & (open_side < 0.025), -1e20, lb)
    ub = torch.where(~integral & (open_side >= 0.025) & (open_side < 0.05), 1e20, ub)
    lo = torch.where(lb <= -1e20, ub - 1e4, lb)
    hi = torch.where(ub >= 1e20, lb + 1e4, ub)
    point = lo + (hi - lo) * u(cols)
    point = torch.where(integral, point.round(), point)
    n = len(row)
    val = torch.pow(10.0, -3.0 + 6.0 * u(n)) * torch.where(u(n) < 0.5, -1.0, 1.0)
    small = torch.where(val > 0, lb[col], ub[col])
    large = torch.where(val > 0, ub[col], lb[col])
    rowptr = np.concatenate([[0], np.cumsum(np.bincount(row.cpu().numpy(), minlength=rows))]).astype(np.int64)

    def total(x):   # per row, on the host: the same bits every time (every row has a nonzero)
        return np.add.reduceat(x.cpu().numpy(), rowptr[:-1])

    least = total(torch.where(small.abs() < 1e20, val * small, 0.0))
    most = total(torch.where(large.abs() < 1e20, val * large, 0.0))
    centre = total(val * point[col]) if planted else 0.5 * (least + most)
    return sa.Instance(rowptr, col.int().cpu().numpy(), val.cpu().numpy(), centre - 0.3 * (most - least),
                       centre + 0.3 * (most - least), *(t.cpu().numpy() for t in (integral.to(torch.uint8), lb, ub)))


def instance(case, seed):
    if case["family"] == "cover":
        return sa.gen_covering_packing(case["rows"], case["cols"], seed=seed)
    return mixed(case["rows"], case["cols"], seed, case.get("planted", True))


def packed_rows(case):
    """Rows of each packed instance, 500 to the most, evenly spread in their logarithm, large and
    small ones in turn."""
    size = [int(round(500 * (case["most"] / 500) ** (i / (case["count"] - 1)))) for i in range(case["count"])]
    return size[::2] + size[1::2][::-1]


def branched(inst, lb, ub, count, rng):
    """Bounds of a node: `count` branchings on unfixed integer columns (a half of the domain)."""
    lb, ub = lb.copy(), ub.copy()
    free = np.nonzero((inst.integral != 0) & (ub - lb >= 1.0))[0]
    for j in rng.choice(free, size=min(count, len(free)), replace=False) if len(free) else []:
        mid = math.floor((lb[j] + ub[j]) / 2)
        if rng.random() < 0.5:
            ub[j] = mid
        else:
            lb[j] = mid + 1
    return lb, ub


# ---- what a user's program has in hand before the call ---------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    s = dict(kind=kind)
    if kind == "serve":
        return prepare_serve(case, seed, rng, s)
    s["ctx"] = ctx = sa.Context(0)
    if kind == "packed":
        parts = [mixed(m, int(1.5 * m), seed * 64 + i, True, uniform=(4, 64)) for i, m in enumerate(packed_rows(case))]
        s["mat"] = sa.PackedMatrix(ctx, parts)
        s["params"] = sa.default_params()
        s["lb"], s["ub"] = s["mat"].inst.lb, s["mat"].inst.ub
        return s
    inst = instance(case, seed)
    s["mat"] = mat = sa.Matrix(ctx, inst)
    if kind in ("plain", "reasons"):
        flags = (sa.SAP_FLAG_RANGEDROWS if case.get("ranged", kind == "reasons") else 0) \
            | (0 if case.get("tighten", True) else sa.SAP_FLAG_NOTIGHTEN)
        s["params"] = sa.default_params(flags=flags)
        s["lb"], s["ub"] = inst.lb, inst.ub
        if case.get("node", 0):
            lb, ub, _ = mat.propagate()
            s["lb"], s["ub"] = branched(inst, lb, ub, case["node"], rng)
    elif kind == "device":
        s["params"] = sa.default_params()
        s["lb0"], s["ub0"] = torch.from_numpy(inst.lb).cuda(), torch.from_numpy(inst.ub).cuda()
        s["lb"], s["ub"] = s["lb0"].clone(), s["ub0"].clone()
    elif kind == "resident":
        s["params"] = sa.default_params()
        s["root"], s["work"] = sa.Bounds(mat, 1), sa.Bounds(mat, 1)
        s["root"].upload(inst.lb, inst.ub)
    else:   # calls on a resident root fixpoint
        s["root"] = root = sa.Bounds(mat, 1)
        root.upload(inst.lb, inst.ub)
        root.propagate()
        lb, ub = root.download()
        s["params"] = sa.default_params(flags=FIXPOINT)
        s["set"] = sa.Bounds(mat, case["nvec"])
        free = np.nonzero((inst.integral != 0) & (ub - lb >= 1.0))[0]
        if kind == "nodes":
            # a node fixes 1..50 binaries, or halves the domains of as many integer columns
            size = rng.integers(1, 51, size=case["nvec"]) if case["nvec"] > 1 else [25]
            col = np.concatenate([rng.choice(free, size=int(min(n, len(free))), replace=False) for n in size])
            mid, down = np.floor((lb[col] + ub[col]) / 2), rng.random(len(col)) < 0.5
            ptr = np.concatenate([[0], np.cumsum(np.minimum(size, len(free)))])
            # room for the change lists: a binary node changes few columns, a mixed one many
            s["cap"] = case["nvec"] * 64 + 1024 if case["family"] == "cover" else case["nvec"] * 2048 + 8192
            s["ov"] = (ptr, col, np.where(down, lb[col], mid + 1), np.where(down, mid, ub[col]))
        else:
            pick = np.sort(rng.choice(free, size=min(case["nprobe"], len(free)), replace=False)).astype(np.int32)
            s["cols"] = pick
            s["cap"] = 16 * len(pick) + 1024 if kind == "probe" else 2048 * len(pick) + 8192
            s["down"] = s["up"] = None
            if kind == "split":
                s["down"] = np.floor(lb[pick] + (ub[pick] - lb[pick] - 1.0) * rng.random(len(pick)))
                s["up"] = s["down"] + 1.0
    return s


def prepare_serve(case, seed, rng, s):
    s["server"] = server = sa.Server(0, nstreams=4, hbm_budget=16 << 30, slots=case["slots"])
    probs = [sa.gen_covering_packing(case["rows"], case["cols"], seed=seed)]
    probs += [mixed(2_000 * (i + 1) + 7, 3_000 * (i + 1) + 5, seed * 8 + i, True) for i in range(case["others"])]
    for p in probs:
        server.warm(server.add_problem(p))
    n = case["requests"]
    which = np.where(rng.random(n) < 0.5, 0, 1 + rng.integers(0, case["others"], size=n)).astype(np.int32)
    ints = [np.nonzero(p.integral)[0] for p in probs]
    cols = [np.unique(rng.choice(ints[w], size=int(rng.integers(1, 51)))) for w in which]
    ptr = np.concatenate([[0], np.cumsum([len(c) for c in cols])])
    fix = rng.integers(0, 2, size=int(ptr[-1])).astype(np.float64)
    s["trace"] = (np.zeros(n), which, ptr, np.concatenate(cols).astype(np.int32), fix, fix)
    s["params"] = sa.default_params(flags=FIXPOINT)
    return s


def whole(a):
    """A returned list with the unused rest of its buffer (zeros): its length is then the
    caller's room, not the number of entries that these inputs happen to give."""
    return a if a.base is None else a.base


# ---- one pass ---------------------------------------------------------------------------------
def run(s):
    kind, params = s["kind"], s["params"]
    if kind == "plain":
        lb, ub, st = s["mat"].propagate(s["lb"], s["ub"], params)
        return dict(lb=lb, ub=ub, result=st["result"], rounds=st["rounds"])
    if kind == "reasons":
        r = s["mat"].propagate_reasons(s["lb"], s["ub"], params)
        out = {k: whole(r[k]) for k in ("round", "col", "bound", "val", "row", "rule")}
        return dict(out, lb=r["lb"], ub=r["ub"], conflict=r["conflict"], nhist=r["nhist"], result=r["stats"]["result"], rounds=r["stats"]["rounds"])
    if kind == "resident":
        s["work"].copy_from(s["root"])
        st = s["work"].propagate(params)
        lb, ub = s["work"].download()
        return dict(lb=lb, ub=ub, result=st["result"], rounds=st["rounds"])
    if kind == "device":
        s["lb"].copy_(s["lb0"])
        s["ub"].copy_(s["ub0"])
        torch.cuda.current_stream().synchronize()   # the engine works on a stream of its own
        st = s["mat"].propagate_device_noalloc(s["lb"].data_ptr(), s["ub"].data_ptr(), params)
        return dict(lb=s["lb"], ub=s["ub"], result=st["result"], rounds=st["rounds"])
    if kind == "nodes":
        r = s["set"].propagate_nodes(s["root"], 0, *s["ov"], params=params, chgcap=s["cap"])
        return {k: whole(r[k]) for k in ("result", "rounds", "chgptr", "chgcol", "chglb", "chgub")}
    if kind in ("probe", "split"):
        r = s["set"].probe(s["root"], 0, s["cols"], params, downub=s["down"], uplb=s["up"], dedcap=s["cap"])
        return {k: whole(r[k]) for k in ("verdict", "rounds", "dedptr", "dedcol", "dlb0", "dub0", "dlb1", "dub1")}
    if kind == "packed":
        lb, ub, res, rounds, _ = s["mat"].propagate_packed(s["lb"], s["ub"], params)
        return dict(lb=lb, ub=ub, result=res, rounds=rounds)
    r = s["server"].replay(*s["trace"], mode=sa.SAP_SERVE_CONTINUOUS, params=params, want_changes=True)
    return {k: whole(r[k]) for k in ("result", "rounds", "nchg", "chgptr", "chgcol", "chglb", "chgub")}


def work(case):
    """Bytes: a nonzero is 8 (value) + 4 (column), a row 16 (sides) + 4 (pointer), a column 16 in
    and 16 out (bounds); a call on a fixpoint base reads only the rows of the columns it
    changes.  Operations: about 20 per nonzero (both activities in double-double)."""
    kind = case["kind"]
    if kind == "packed":
        rows = sum(packed_rows(case))
        nnz, cols = 34 * rows, 1.5 * rows
    else:
        rows, cols = case["rows"], case["cols"]
        nnz = rows * (10 if case["family"] == "cover" else 13.2)
    if kind in ("plain", "reasons", "resident", "device", "packed"):
        return dict(bytes=12 * nnz + 20 * rows + 32 * cols, flops=20 * nnz)
    changed = {"nodes": 25.5 * case.get("nvec", 0), "serve": 25.5 * case.get("requests", 0)}.get(kind, 2 * case.get("nprobe", 0))
    touched = changed * nnz / cols               # rows of the changed columns
    each = nnz / rows
    return dict(bytes=touched * (28 * each + 24) + 40 * changed, flops=20 * touched * each)


def binary_fixpoint(inst, lb, ub):
    """The fixpoint of a covering/packing system from given bounds; None if it is infeasible."""
    lb, ub = lb.copy(), ub.copy()
    row = np.repeat(np.arange(inst.nrows), np.diff(inst.rowptr))
    col, a = inst.colidx, inst.vals
    while True:
        least = np.add.reduceat(a * lb[col], inst.rowptr[:-1])
        most = np.add.reduceat(a * ub[col], inst.rowptr[:-1])
        if ((least > inst.rhs + 1e-3) | (most < inst.lhs - 1e-3)).any():   # sides are multiples of 0.4
            return None
        free = ub[col] - lb[col] > 0.5
        off = free & (a > (inst.rhs - least)[row] + 1e-3)
        on = free & (a > (most - inst.lhs)[row] + 1e-3)
        if not off.any() and not on.any():
            return lb, ub
        ub[col[off]] = 0.0
        lb[col[on]] = 1.0
        if (lb > ub).any():
            return None


def exact(case, seed):
    """A covering/packing system's fixpoint is unique: a row whose remaining slack is smaller than
    an unfixed binary's coefficient fixes that binary.  A mixed system's fixpoint depends on the
    order in which the 5 % improvement rule accepts bounds, and lists of changes follow from
    it, so those have no value of their own."""
    if case["kind"] != "plain" or case["family"] != "cover":
        return None
    inst = instance(case, seed)
    lb, ub = branched(inst, *binary_fixpoint(inst, inst.lb, inst.ub), case["node"], np.random.default_rng(seed))
    end = binary_fixpoint(inst, lb, ub)
    return dict(lb=lb if end is None else end[0], ub=ub if end is None else end[1], result=None, rounds=None)
