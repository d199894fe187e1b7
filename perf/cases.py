"""The work a user of this library has it do, as cases that can be timed.

Every case goes through a public entry point: the device-resident batch
stream (Context), the one-shot driver (run_dynlp), the batched runner and the
serving loop (Multi), the IrLP baseline and the five step launchers on device
pointers.  Sizes are those of the benchmark, the tests and the reference's own
run targets (5K, 50K and 500K vertices), and larger ones for the HBM-bound end.

    listed()             the cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what a program has in hand before the call
    run(state)           one pass; its outputs
    work(case)           bytes and operations one pass cannot do without
    exact(case, seed)    the outputs in 64-bit arithmetic, where they have one
"""
import ctypes as C

import numpy as np
import torch

import labelpropcuda_amd as L
from labelpropcuda_amd._lib import check, load

DELTA = 1e-4
DEV = "cuda"


# ------------------------------------------------------------------------
# cases
# ------------------------------------------------------------------------
def listed():
    return [
        # the reference's small run and the CPU-comparable configuration:
        # latency of a whole short stream, every frontier small
        {"name": "stream_5k", "kind": "stream", "n": 5000, "degree": 5, "batches": 10,
         "max_iter": 100000, "on_device": False},
        # the reference's default run target
        {"name": "stream_50k", "kind": "stream", "n": 50000, "degree": 5, "batches": 10,
         "max_iter": 100000, "on_device": False},
        # the benchmark's workload: every frontier size from a handful of
        # vertices to most of the graph
        {"name": "stream_500k", "kind": "stream", "n": 500000, "degree": 7, "batches": 10,
         "max_iter": 100000, "on_device": False},
        # a graph far beyond the caches, with an iteration cap as a user
        # short of time sets it: large frontiers, HBM-bound
        {"name": "stream_6m", "kind": "stream", "n": 6000011, "degree": 7, "batches": 8,
         "max_iter": 1000, "on_device": True},
        # a resident tenant that receives small updates one after another:
        # the fixed cost of a batch
        {"name": "updates_400k", "kind": "updates", "n": 400000, "degree": 5, "updates": 24,
         "smallest": 100, "largest": 1000},
        # one call from host arrays to host labels, as the command line and
        # the C++ driver make it: upload, creation, every batch, read-back
        {"name": "driver_20k", "kind": "driver", "n": 20000, "degree": 5, "batches": 5,
         "max_iter": 100000},
        # many small graphs of uneven size advanced together
        {"name": "batched_40", "kind": "batched", "graphs": 40, "smallest": 2000,
         "largest": 16000, "batches": 8},
        # tenants served as their requests arrive (all at once: saturated)
        {"name": "serve_12", "kind": "serve", "tenants": 12, "smallest": 10000,
         "largest": 200000, "requests": 32, "least": 100, "most": 20000},
        # the full-recompute baseline on the benchmark graph's size
        {"name": "irlp_500k", "kind": "irlp", "n": 500000, "degree": 7},
        # the same, far beyond the caches
        {"name": "irlp_8m", "kind": "irlp", "n": 8000009, "degree": 7},
        # one batch through the five step launchers, by a caller that may
        # not allocate device memory (the allocation-free propagation)
        {"name": "steps_20k", "kind": "steps", "n": 20001, "degree": 5, "max_iter": 100000,
         "noalloc": True},
        # the same launchers on a large graph
        {"name": "steps_2m", "kind": "steps", "n": 2000003, "degree": 7, "max_iter": 500,
         "noalloc": False},
    ]


def _between(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))


def draw(rng):
    kind = rng.choice(["stream", "stream", "stream", "large", "updates", "driver", "batched",
                       "serve", "irlp", "irlp", "steps", "steps"])
    degree = rng.choice([3, 5, 6, 7, 7])
    if kind == "stream":
        n = _between(rng, 3000, 500000)
        return {"kind": "stream", "n": n, "degree": degree, "batches": rng.randint(4, 10),
                "max_iter": 100000 if n <= 50000 else 10000, "on_device": False}
    if kind == "large":
        return {"kind": "stream", "n": _between(rng, 1000000, 6000000), "degree": degree,
                "batches": rng.randint(4, 8), "max_iter": rng.randint(200, 1000),
                "on_device": True}
    if kind == "updates":
        return {"kind": "updates", "n": _between(rng, 50000, 400000), "degree": 5,
                "updates": rng.randint(8, 24), "smallest": rng.randint(50, 200),
                "largest": rng.randint(400, 1000)}
    if kind == "driver":
        return {"kind": "driver", "n": _between(rng, 2000, 20000), "degree": degree,
                "batches": rng.randint(3, 6), "max_iter": 100000}
    if kind == "batched":
        return {"kind": "batched", "graphs": rng.randint(8, 40), "smallest": 2000,
                "largest": _between(rng, 4000, 16000), "batches": rng.randint(4, 8)}
    if kind == "serve":
        return {"kind": "serve", "tenants": rng.randint(3, 12), "smallest": 10000,
                "largest": _between(rng, 20000, 200000), "requests": rng.randint(8, 32),
                "least": 100, "most": _between(rng, 2000, 20000)}
    if kind == "irlp":
        return {"kind": "irlp", "n": _between(rng, 3000, 8000000), "degree": degree}
    n = _between(rng, 3000, 2000000)
    return {"kind": "steps", "n": n, "degree": degree,
            "max_iter": 100000 if n <= 50000 else 500,
            "noalloc": n <= 500000 and rng.random() < 0.5}


# ------------------------------------------------------------------------
# graphs made on the device
# ------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _graph(n, degree, g):
    """A random spanning tree plus uniform random edges to the average
    degree, symmetric; true labels Bernoulli(0.5); weights U[0.5, 1) within
    a class, U[0, 0.5) across: the synthetic graphs of the reference's
    generator.  Returns CSR arrays, labels and the edges u < v."""
    perm = torch.randperm(n, generator=g, device=DEV)
    at = torch.arange(1, n, device=DEV)
    parent = torch.minimum((torch.rand(n - 1, generator=g, device=DEV, dtype=torch.float64)
                            * at).long(), at - 1)
    a, b = perm[1:], perm[parent]
    tree = torch.sort(torch.minimum(a, b) * n + torch.maximum(a, b)).values
    extra = max(0, n * degree // 2 - (n - 1))
    x = torch.randint(n, (extra + extra // 50 + 64,), generator=g, device=DEV)
    y = torch.randint(n, (len(x),), generator=g, device=DEV)
    key = torch.unique((torch.minimum(x, y) * n + torch.maximum(x, y))[x != y])
    key = key[tree[torch.searchsorted(tree, key).clamp_max(n - 2)] != key]
    key = key[torch.randperm(len(key), generator=g, device=DEV)[:extra]]
    key = torch.sort(torch.cat([tree, key])).values
    u, v = key // n, key % n
    truth = (torch.rand(n, generator=g, device=DEV) >= 0.5).float()
    r = 0.5 * torch.rand(len(u), generator=g, device=DEV)
    w = torch.where(truth[u] == truth[v], r + 0.5, r)
    src, dst, ww = torch.cat([u, v]), torch.cat([v, u]), torch.cat([w, w])
    order = torch.argsort(src * n + dst)
    row = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    row[1:] = torch.cumsum(torch.bincount(src, minlength=n), 0)
    return (row.int(), dst[order].int().contiguous(), ww[order].contiguous(), truth, u, v, w)


def _stream_inputs(n, degree, batches, seed):
    """The reference's batch stream (balanced ground truth first, then equal
    shares of new vertices with 1 % ground truth and 9 % deletions; an edge
    arrives with its later end) over a graph made on the device."""
    g = _gen(seed)
    row, col, val, truth, u, v, w = _graph(n, degree, g)
    order = torch.randperm(n, generator=g, device=DEV)
    half = max(2, n // 100) // 2
    first = torch.cat([order[truth[order] == c][:half] for c in (0.0, 1.0)])
    batch = torch.full((n,), -1, dtype=torch.int64, device=DEV)
    batch[first] = 0
    rest = order[batch[order] < 0]
    ins, gt, dels = [first], [first], [first[:0]]
    free = torch.zeros(n, dtype=torch.bool, device=DEV)
    for b, part in enumerate(torch.tensor_split(rest, batches - 1), 1):
        batch[part] = b
        k = max(1, len(part) // 100)
        ins.append(part)
        gt.append(part[:k])
        free[part[k:]] = True
        pool = torch.nonzero(free).flatten()
        gone = pool[torch.randperm(len(pool), generator=g, device=DEV)[:len(part) * 9 // 100]]
        free[gone] = False
        dels.append(gone)
    arrives = torch.maximum(batch[u], batch[v])
    by = torch.argsort(arrives, stable=True)

    def host(t, dtype):
        return np.ascontiguousarray(t.cpu().numpy().astype(dtype, copy=False))

    def offsets(lens):
        return np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)

    return L.Inputs(
        rowPtr=host(row, np.int32), colInd=host(col, np.int32), values=host(val, np.float32),
        trueLabels=host(truth, np.float32),
        insOff=offsets([len(t) for t in ins]), ins=host(torch.cat(ins), np.int32),
        gtOff=offsets([len(t) for t in gt]), gtIds=host(torch.cat(gt), np.int32),
        gtLab=host(truth[torch.cat(gt)], np.float32),
        delOff=offsets([len(t) for t in dels]), dels=host(torch.cat(dels), np.int32),
        eOff=offsets(torch.bincount(arrives, minlength=batches).tolist()),
        eSrc=host(u[by], np.int32), eDst=host(v[by], np.int32), eW=host(w[by], np.float32))


# ------------------------------------------------------------------------
# prepare
# ------------------------------------------------------------------------
def prepare(case, seed):
    return {"stream": _prep_stream, "updates": _prep_updates, "driver": _prep_driver,
            "batched": _prep_batched, "serve": _prep_serve, "irlp": _prep_irlp,
            "steps": _prep_steps}[case["kind"]](case, int(seed))


def _prep_stream(c, seed):
    if c["on_device"]:
        inp = _stream_inputs(c["n"], c["degree"], c["batches"], seed)
    else:
        inp = L.generate(c["n"], c["degree"], c["batches"], seed % (1 << 31))
    return {"kind": "stream", "ctx": L.Context(inp, L.make_config(inp, maxIterations=c["max_iter"]))}


def _prep_updates(c, seed):
    sizes = _sizes(np.random.default_rng(seed), c["smallest"], c["largest"], c["updates"])
    inp = L.generate_stream(c["n"], c["degree"], [0] + sizes, seed % (1 << 31))
    return {"kind": "stream", "ctx": L.Context(inp, L.make_config(inp))}


def _prep_driver(c, seed):
    inp = L.generate(c["n"], c["degree"], c["batches"], seed % (1 << 31))
    return {"kind": "driver", "inputs": inp,
            # tau given, so that the call prints nothing
            "cfg": L.make_config(inp, tau=0.5, maxIterations=c["max_iter"])}


def _sizes(rng, smallest, largest, count):
    """`count` whole numbers spread over the logarithm of [smallest, largest]."""
    return [int(k) for k in np.rint(np.exp(rng.uniform(np.log(smallest), np.log(largest), count)))]


def _prep_batched(c, seed):
    """Graph sizes and degrees belong to the case, the graphs to the seed."""
    rng = np.random.default_rng(42)
    sizes = _sizes(rng, c["smallest"], c["largest"], c["graphs"])
    degrees = [int(d) for d in rng.choice([3, 5, 7], c["graphs"])]
    return {"kind": "batched",
            "multi": L.Multi([L.generate(n, d, c["batches"], (seed + i) % (1 << 31))
                              for i, (n, d) in enumerate(zip(sizes, degrees))])}


def _prep_serve(c, seed):
    """Tenants' and requests' sizes belong to the case, the graphs to the
    seed."""
    rng = np.random.default_rng(1042)
    sizes = _sizes(rng, c["smallest"], c["largest"], c["tenants"])
    who = rng.integers(0, c["tenants"], c["requests"])
    size = _sizes(rng, c["least"], c["most"], c["requests"])
    tenants = [L.generate_stream(n, 5, [0] + [k for k, w in zip(size, who) if w == t],
                                 (seed + t) % (1 << 31)) for t, n in enumerate(sizes)]
    return {"kind": "serve", "multi": L.Multi(tenants), "requests": [(int(t), 0.0) for t in who]}


def _status(n, g):
    """Status and ground-truth class of an evolved graph: 1 % ground truth,
    9 % deleted."""
    r = torch.rand(n, generator=g, device=DEV)
    return torch.where(r < 0.01, 2, torch.where(r < 0.10, 1, 0)).int()


def _irlp_inputs(c, seed):
    g = _gen(seed)
    row, col, val, truth, _, _, _ = _graph(c["n"], c["degree"], g)
    status = _status(c["n"], g)
    gt = torch.where(status == 2, truth.int(), -1).int()
    labels = torch.where(status == 2, truth, 0.5).float()
    return row, col, val, status, gt, labels


def _prep_irlp(c, seed):
    row, col, val, status, gt, labels = _irlp_inputs(c, seed)
    return {"kind": "irlp", "row": row, "col": col, "val": val, "status": status, "gt": gt,
            "start": labels, "labels": labels.clone()}


def _prep_steps(c, seed):
    """One batch as the reference's driver hands it to its launchers: the
    active CSR with the new vertices (a tenth of the graph) in it, the edges
    that arrive with them, the deletions, and labels of the old vertices
    that have settled near their class."""
    n, g = c["n"], _gen(seed)
    row, col, val, truth, u, v, w = _graph(n, c["degree"], g)
    order = torch.randperm(n, generator=g, device=DEV)
    k = n // 10
    new = order[:k].contiguous()
    is_new = torch.zeros(n, dtype=torch.int32, device=DEV)
    is_new[new] = 1
    status = torch.zeros(n, dtype=torch.int32, device=DEV)
    gt_ids = torch.cat([new[:max(1, k // 100)], order[k:k + n // 100]])
    status[gt_ids] = 2
    gt = torch.full((n,), -1, dtype=torch.int32, device=DEV)
    gt[gt_ids] = truth[gt_ids].int()
    gone = order[n - max(1, k * 9 // 100):].int().contiguous()
    near = truth + (0.5 - truth) * torch.rand(n, generator=g, device=DEV)
    labels = torch.where(is_new == 1, 0.5, near)
    labels[gt_ids] = truth[gt_ids]
    arrives = (is_new[u] + is_new[v]) > 0
    m = max(int(arrives.sum()), n * c["degree"] // 8)

    def ints(size):
        return torch.zeros(size, dtype=torch.int32, device=DEV)

    return {"kind": "steps", "n": n, "max_iter": c["max_iter"], "noalloc": c["noalloc"],
            "row": row, "col0": col, "col": col.clone(), "val": val, "status0": status,
            "status": status.clone(), "affected": ints(n), "gone": gone,
            "new": new.int().contiguous(), "is_new": is_new, "eu": u[arrives].int(),
            "ev": v[arrives].int(), "ew": w[arrives].contiguous(), "gt": gt,
            "labels0": labels.float(), "labels": labels.float().clone(),
            "buffer": torch.empty(n, device=DEV), "comp": ints(n), "sub_src": ints(2 * m),
            "sub_dst": ints(2 * m), "sub_w": torch.zeros(2 * m, device=DEV),
            "sub_row": ints(n + 1), "tau": float(val.mean())}


# ------------------------------------------------------------------------
# run
# ------------------------------------------------------------------------
def run(state):
    return {"stream": _run_stream, "driver": _run_driver, "batched": _run_batched,
            "serve": _run_serve, "irlp": _run_irlp, "steps": _run_steps}[state["kind"]](state)


_COUNTS = ("numSubEdges", "numComponents", "numMarked", "frontier0", "iterations", "numTouched",
           "updates")


def _run_stream(s):
    ctx = s["ctx"]
    ctx.run_all()
    labels = ctx.labels()
    st = [ctx.stats(b) for b in range(ctx.inputs.numBatches)]
    return {"labels": labels, "counts": np.array([[x[k] for k in _COUNTS] for x in st], np.int64),
            "accuracy": np.array([x["accuracy"] for x in st], np.float32)}


def _run_driver(s):
    labels, _, accuracy = L.run_dynlp(s["inputs"], s["cfg"])
    return {"labels": labels, "accuracy": accuracy}


def _tenants(m, skip=0):
    counts, accuracy = [], []
    for t, g in enumerate(m.graphs):
        for b in range(skip, g.numBatches):
            x = m.stats(t, b)
            counts.append([x[k] for k in _COUNTS])
            accuracy.append(x["accuracy"])
    return {"labels": np.concatenate([m.labels(t) for t in range(len(m.graphs))]),
            "counts": np.array(counts, np.int64), "accuracy": np.array(accuracy, np.float32)}


def _run_batched(s):
    m = s["multi"]
    m.run_all()
    m.synchronize()
    return _tenants(m)


def _run_serve(s):
    m = s["multi"]
    m.reset()
    m.run_next(list(range(len(m.graphs))))  # every tenant's ground-truth seed
    m.serve(s["requests"])
    m.synchronize()
    return _tenants(m, 1)


def _p(t):
    return C.c_void_p(t.data_ptr())


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _run_irlp(s):
    s["labels"].copy_(s["start"])
    used = C.c_int(0)
    check(load().dlp_irlp(_p(s["row"]), _p(s["col"]), _p(s["val"]), _p(s["labels"]),
                          _p(s["status"]), _p(s["gt"]), len(s["status"]), C.c_float(DELTA),
                          100000, C.byref(used), _stream()))
    return {"labels": s["labels"], "iterations": used.value}


def _run_steps(s):
    lib, n, q = load(), s["n"], _stream()
    for dst, src in (("col", "col0"), ("status", "status0"), ("labels", "labels0")):
        s[dst].copy_(s[src])
    s["affected"].zero_()
    check(lib.dlp_mark_deletions(_p(s["row"]), _p(s["col"]), _p(s["status"]), _p(s["affected"]),
                                 _p(s["gone"]), len(s["gone"]), n, q))
    nodes, edges, comps, used = C.c_int(0), C.c_int(0), C.c_int(0), C.c_int(0)
    check(lib.dlp_build_sparsified_subgraph(
        _p(s["row"]), _p(s["col"]), _p(s["val"]), _p(s["affected"]), _p(s["status"]), _p(s["eu"]),
        _p(s["ev"]), _p(s["ew"]), len(s["eu"]), _p(s["new"]), len(s["new"]), _p(s["is_new"]),
        C.c_float(s["tau"]), _p(s["sub_row"]), _p(s["sub_dst"]), _p(s["sub_w"]),
        _p(s["sub_src"]), C.byref(nodes), C.byref(edges), q))
    check(lib.dlp_connected_components(_p(s["sub_src"]), _p(s["sub_dst"]), edges.value,
                                       _p(s["new"]), len(s["new"]), _p(s["comp"]),
                                       C.byref(comps), n, q))
    check(lib.dlp_label_initialization(
        _p(s["row"]), _p(s["col"]), _p(s["val"]), _p(s["labels"]), _p(s["status"]),
        _p(s["comp"]), comps.value, _p(s["new"]), len(s["new"]), _p(s["gt"]), n, q))
    propagate = (lib.dlp_iterative_propagation_noalloc if s["noalloc"]
                 else lib.dlp_iterative_propagation)
    check(propagate(_p(s["row"]), _p(s["col"]), _p(s["val"]), _p(s["labels"]), _p(s["buffer"]),
                    _p(s["status"]), _p(s["gt"]), _p(s["affected"]), n, C.c_float(DELTA),
                    s["max_iter"], C.byref(used), q))
    return {"labels": s["labels"], "col": s["col"], "status": s["status"],
            "affected": s["affected"], "sub_src": s["sub_src"], "sub_dst": s["sub_dst"],
            "sub_w": s["sub_w"], "comp": s["comp"], "edges": edges.value,
            "components": comps.value, "iterations": used.value}


# ------------------------------------------------------------------------
# work
# ------------------------------------------------------------------------
def _graph_work(n, degree):
    """Row pointers, columns and weights once; a multiply and two additions
    per stored entry."""
    return 4 * (n + 1) + 8 * n * degree, 3 * n * degree


def work(case):
    """Each input read once and each output written once, with one sweep's
    arithmetic: how many iterations a stream needs is known only by running
    it."""
    c, kind = case, case["kind"]
    if kind == "batched":
        mean = (c["largest"] - c["smallest"]) / np.log(c["largest"] / c["smallest"])
        n, degree = int(c["graphs"] * mean), 5
    elif kind == "serve":
        mean = (c["largest"] - c["smallest"]) / np.log(c["largest"] / c["smallest"])
        n, degree = int(c["tenants"] * mean), 5
    else:
        n, degree = c["n"], c["degree"]
    b, f = _graph_work(n, degree)
    if kind in ("stream", "driver", "batched"):
        # true labels in, labels out, every vertex and edge in its batch list
        b += 8 * n + 4 * n + 12 * (n * degree // 2)
    elif kind in ("updates", "serve"):
        b += 8 * n  # labels out, true labels in: the lists are small
    elif kind == "irlp":
        b += 16 * n  # status, ground truth, labels in and out
    else:
        # status, ground truth, affected, components, labels; the new edges
        # in (a fifth of all) and the columns out
        b += 28 * n + 12 * (n * degree // 10) + 4 * n * degree
    return {"bytes": float(b), "flops": float(f)}


# ------------------------------------------------------------------------
# exact
# ------------------------------------------------------------------------
def exact(case, seed):
    """IrLP converges to values that 64-bit arithmetic gives too.  The other
    paths decide by a threshold on every label and every iteration which
    vertices go on, so another rounding follows another trajectory (the
    64-bit twin of a stream ends up to 2e-2 away): they have no such value."""
    if case["kind"] != "irlp":
        return None
    row, col, val, status, gt, labels = _irlp_inputs(case, int(seed))
    n = len(status)
    src = torch.repeat_interleave(torch.arange(n, device=DEV), (row[1:] - row[:-1]).long())
    dst, w = col.long(), val.double()
    w = torch.where(status[dst] == 1, 0.0, w)
    total = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, src, w)
    live = (status == 0) & (gt < 0)
    old = labels.double()
    for _ in range(100000):
        s = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, src, w * old[dst])
        new = torch.where(live & (total > 1e-10), s / total, old).clamp(0.0, 1.0)
        moved = float(((new - old).abs() * live).max())
        old = new
        if moved <= DELTA:
            break
    return {"labels": old, "iterations": None}
