"""Batches that run into the iteration cap alternate between two states: the
propagation kernels count the iterations that repeat the state of two
iterations before bit for bit instead of running them.  Labels, iteration and
update counts must stay the oracle's, which runs every one of them, for every
engine and for an even and an odd number of iterations left."""
import time

import numpy as np
import pytest

import labelpropcuda_amd as L
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.int32)


def from_rows(rows, labels, prefix, batches):
    """Inputs of a graph given as {neighbour: weight} rows, through the graph
    text files and the reference batch generator."""
    rows = [sorted(r.items()) for r in rows]
    for name, vals in (("RowPtr", np.cumsum([0] + [len(r) for r in rows])),
                       ("ColInd", [v for r in rows for v, _ in r]),
                       ("Values", [f"{w:.6f}" for r in rows for _, w in r]),
                       ("TrueLabels", [f"{i} {c}" for i, c in enumerate(labels)])):
        with open(prefix + name + ".txt", "w") as f:
            f.write("\n".join(map(str, vals)) + "\n")
    return L.dynlp.from_graph_files(prefix, batches, 42)


def star_tree(prefix, hubs=40, leaves=30, seed=2, batches=6):
    """A random tree of hubs, each with about `leaves` leaves: deletions
    detach bipartite subtrees, whose labels alternate; the hubs' rows are
    longer than one lane sums."""
    rng = np.random.default_rng(seed)
    n = hubs * (leaves + 1)
    ids = rng.permutation(n)
    rows = [{} for _ in range(n)]
    for x in range(1, n):
        u, v = int(ids[x]), int(ids[rng.integers(min(x, hubs))])
        rows[u][v] = rows[v][u] = float(rng.uniform(0.05, 1.0))
    return from_rows(rows, rng.permutation(np.arange(n) % 2), prefix, batches)


def one_sided(inp, prefix, share=0.1, seed=2):
    """`inp`'s graph with a share of its entries dropped on one side."""
    rng = np.random.default_rng(seed)
    rows = [{int(v): float(w) for v, w in zip(inp.colInd[a:b], inp.values[a:b])
             if rng.random() >= share}
            for a, b in zip(inp.rowPtr[:-1], inp.rowPtr[1:])]
    return from_rows(rows, inp.trueLabels.astype(int), prefix, 8)


_ORACLE = {}


def oracle_run(key, inp, cap):
    """(labels bits, iterations, updates) after every batch."""
    if (key, cap) not in _ORACLE:
        orc = Oracle(inp, maxIterations=cap)
        res = []
        for b in range(inp.numBatches):
            orc.run_batch(b)
            st = orc.stats()
            res.append((bits(orc.labels()).copy(), st["iterations"], st["updates"]))
        assert any(r[1] == cap for r in res), "no batch reaches the cap"
        _ORACLE[key, cap] = res
    return _ORACLE[key, cap]


def graph(kind, tmp_path):
    if kind == "random":
        return L.generate(5000, 5, 6, 42)
    if kind == "sparse":
        return L.generate(2000, 3, 8, 3)
    if kind == "long rows":
        return star_tree(str(tmp_path / "star_"))
    if kind == "hubs":
        return star_tree(str(tmp_path / "hubs_"), 12, 90, 5, 8)
    return one_sided(L.generate(2000, 3, 8, 3), str(tmp_path / "one_"))


def check(kind, inp, cap, skips=True, **tuning):
    want = oracle_run(kind, inp, cap)
    with L.Context(inp, L.make_config(inp, maxIterations=cap)) as ctx:
        ctx.set_tuning(**tuning)
        for _ in range(2):  # the second pass starts from the first one's device state
            ctx.reset()
            for b in range(inp.numBatches):
                ctx.run_batch(b)
                st = ctx.stats(b)
                assert (st["iterations"], st["updates"]) == want[b][1:], f"batch {b}"
                assert np.array_equal(bits(ctx.labels()), want[b][0]), f"batch {b}: labels"
        it, up = ctx.skipped()
        if skips:
            assert 0 < it < sum(r[1] for r in want) and 0 < up < sum(r[2] for r in want)
        elif skips is not None:
            assert (it, up) == (0, 0)


CAPS = [20000, 20001]


@pytest.mark.parametrize("cap", CAPS)
@pytest.mark.parametrize("kind,tuning", [
    ("random", dict()),                                       # register-mask kernels
    ("random", dict(localOwnerAfter=1)),
    ("random", dict(localOwnerAfter=1, maskOwnerMax=-1)),     # flags, one vertex per thread
    ("random", dict(localOwnerAfter=1, maskOwnerMax=-1, localShape=4)),  # several per thread
    ("sparse", dict(localOwnerAfter=1)),
    ("long rows", dict(localOwnerAfter=1)),                   # rows summed by a wave
    ("one-sided", dict(localOwnerAfter=1)),                   # one wave, rows OR-reduced
])
def test_owner_kernels(gpu_available, tmp_path, kind, tuning, cap):
    check(kind, graph(kind, tmp_path), cap, **tuning)


@pytest.mark.parametrize("cap", CAPS)
@pytest.mark.parametrize("kind,tuning,skips", [
    ("random", dict(), True),
    ("random", dict(chunk=3), True),              # a cycle in the middle of a chunk
    ("random", dict(chunk=1), True),
    ("sparse", dict(), True),
    ("one-sided", dict(), True),
    ("long rows", dict(), True),                  # more than two entries a lane
    ("hubs", dict(), True),                       # rows summed by a wave
    ("hubs", dict(blockRowMin=64), False),        # hub rows: the queue kernel
])
def test_multi_block_kernels(gpu_available, tmp_path, kind, tuning, skips, cap):
    """One launch per iteration, frontier as flags (or, with rows for the
    work-group tier, as a queue, which runs every iteration)."""
    check(kind, graph(kind, tmp_path), cap, skips, localThreshold=-1, **tuning)


def swapping_stars(k, n):
    """k paths of six vertices, ground truth of either class at their ends,
    among n vertices; the last batch deletes the second and the fifth and hangs
    a seventh on the third.  That one and its two neighbours, which no other
    vertex holds now, swap labels for ever (equal weights: with no rounding)."""
    rng = np.random.default_rng(1)
    base = 7 * np.arange(k, dtype=np.int32)[:, None]
    w = rng.uniform(0.1, 1.0, (k, 6)).astype(np.float32)
    w[:, [2, 5]] = 1.0
    # edges 0-1, 1-2, 2-3, 3-4, 4-5 and 2-6, as rows
    rowLen = np.zeros(n, np.int64)
    rowLen[:7 * k] = np.tile([1, 2, 3, 2, 2, 1, 1], k)
    col = base + np.array([1, 0, 2, 1, 3, 6, 2, 4, 3, 5, 4, 2], np.int32)
    val = w[:, [0, 0, 1, 1, 2, 5, 2, 3, 3, 4, 4, 5]]
    truth = np.zeros(n, np.float32)
    truth[:7 * k] = np.tile([0, 0, 0, 1, 1, 1, 0], k)
    ends, inner, late, gone = (base + np.array(x, np.int32)
                               for x in ([0, 5], [1, 2, 3, 4], [6], [1, 4]))
    none = np.zeros(0, np.int32)

    def batches(*lists):
        return np.cumsum([0] + [x.size for x in lists]).astype(np.int64), \
            np.ascontiguousarray(np.concatenate([x.ravel() for x in lists]))

    insOff, ins = batches(ends, inner, late)
    gtOff, gtIds = batches(ends, none, none)
    delOff, dels = batches(none, none, gone)
    path = base + np.arange(5, dtype=np.int32)
    eOff, eSrc = batches(none, path, base + 2)
    return L.Inputs(
        rowPtr=np.concatenate([[0], np.cumsum(rowLen)]).astype(np.int32),
        colInd=col.ravel(), values=val.ravel(), trueLabels=truth, insOff=insOff, ins=ins,
        gtOff=gtOff, gtIds=gtIds, gtLab=truth[gtIds], delOff=delOff, dels=dels, eOff=eOff,
        eSrc=eSrc, eDst=batches(none, path + 1, base + 6)[1],
        eW=np.concatenate([w[:, :5].ravel(), w[:, 5]]))


@pytest.mark.parametrize("cap", [3000, 3001])
@pytest.mark.parametrize("n,thin", [((1 << 20) + 1, True), (1 << 19, False)])
def test_flagged_cycles_by_walk(gpu_available, n, thin, cap):
    """A cycle of some 2,600 vertices found by the walk over flags alone (beyond
    2^20 vertices) and by the one that loads every vertex's row place."""
    inp = swapping_stars(6000, n)
    orc = Oracle(inp, maxIterations=cap)
    with L.Context(inp, L.make_config(inp, maxIterations=cap)) as ctx:
        ctx.set_tuning(localThreshold=-1)
        for b in range(inp.numBatches):
            ctx.set_profiling(1)
            ctx.run_batch(b)
            orc.run_batch(b)
            st, ost = ctx.stats(b), orc.stats()
            assert (st["iterations"], st["updates"]) == (ost["iterations"], ost["updates"])
            assert np.array_equal(bits(ctx.labels()), bits(orc.labels())), f"batch {b}"
        f = ctx.flag_profile()
        assert st["iterations"] == cap and f["idleLaunches"] > 0
        assert f["thinLaunches"] == (f["launches"] if thin else 0)
        it, up = ctx.skipped()
        assert cap - 1200 < it < cap - 1000 and up == orc.frontier_sizes()[-1] * it


@pytest.mark.parametrize("cap", CAPS)
def test_step_propagation(gpu_available, lib, cap):
    """The step entry points: labels, second buffer, exit flags, iterations."""
    import ctypes as C

    import oracle.oracle as O
    from labelpropcuda_amd import _lib
    inp = graph("random", None)
    o = Oracle(inp, maxIterations=cap)
    o.run_batch(0)
    o.run_batch(1)  # runs into the cap
    rp, ci, vv = o.csr()
    d, _, g = o.status()
    init, aff = o.init_labels(), o.affected()
    want = O.propagate(rp, ci, vv, init, d, g, aff, 1e-4, cap)
    assert want[3] == cap
    for fn in (lib.dlp_iterative_propagation, lib.dlp_iterative_propagation_noalloc) * 2:
        dev = [_lib.DeviceArray(x) for x in (rp, ci, vv, init, np.zeros_like(init), d, g, aff)]
        it = C.c_int()
        _lib.check(fn(*[x.ptr for x in dev], inp.numNodes, C.c_float(1e-4), cap, C.byref(it),
                      None))
        assert it.value == cap
        assert np.array_equal(bits(dev[3].numpy()), bits(want[0]))
        assert np.array_equal(bits(dev[4].numpy()), bits(want[1]))
        assert np.array_equal(dev[7].numpy(), want[2])
        # the same state after 40,000,000 iterations more, which run one by
        # one would take half a minute
        t0 = time.perf_counter()
        dev = [_lib.DeviceArray(x) for x in (rp, ci, vv, init, np.zeros_like(init), d, g, aff)]
        _lib.check(fn(*[x.ptr for x in dev], inp.numNodes, C.c_float(1e-4), cap + 40000000,
                      C.byref(it), None))
        assert it.value == cap + 40000000 and time.perf_counter() - t0 < 5.0
        assert np.array_equal(bits(dev[3].numpy()), bits(want[0]))
        assert np.array_equal(bits(dev[4].numpy()), bits(want[1]))


def test_trace_runs_every_iteration(gpu_available):
    """A trace records every iteration's frontier size, so nothing is passed
    over while one is on."""
    inp, cap = L.generate(5000, 5, 4, 42), 6000
    orc = Oracle(inp, maxIterations=cap)
    with L.Context(inp, L.make_config(inp, maxIterations=cap)) as ctx:
        tr = ctx.enable_trace(maxFrontierSizes=cap)
        ctx.reset()
        for b in range(inp.numBatches):
            ctx.run_batch(b)
            orc.run_batch(b)
            assert np.array_equal(tr.snapshot()["frontierSizes"], orc.frontier_sizes())
        assert ctx.skipped() == (0, 0)


@pytest.mark.parametrize("cap", CAPS)
@pytest.mark.parametrize("slices", [0, 700])
@pytest.mark.parametrize("shape", [3, 1, 5])
def test_shared_launch(gpu_available, tmp_path, shape, slices, cap):
    """Many graphs in one launch (queue iterations in LDS), in lockstep and
    stopped and resumed every 700 iterations by the serving loop."""
    kinds = ["random", "sparse", "long rows", "one-sided"]
    graphs = [graph(k, tmp_path) for k in kinds]
    want = [oracle_run(k, g, cap) for k, g in zip(kinds, graphs)]
    with L.Multi(graphs, [L.make_config(g, maxIterations=cap) for g in graphs]) as m:
        m.set_tuning(localShape=shape)
        if slices:
            m.reset()
            reqs = [(i, 0.0) for i, g in enumerate(graphs) for _ in range(g.numBatches)]
            m.serve(reqs, sliceIterations=slices, sliceMs=-1.0, handBackAfter=-1)
        else:
            m.run_all()
        m.synchronize()
        for i, g in enumerate(graphs):
            assert [(s["iterations"], s["updates"])
                    for s in (m.stats(i, b) for b in range(g.numBatches))] == \
                [r[1:] for r in want[i]], kinds[i]
            assert np.array_equal(bits(m.labels(i)), want[i][-1][0]), kinds[i]
            it, up = m.skipped(i)
            assert 0 < it < sum(r[1] for r in want[i]) and 0 < up, kinds[i]


@pytest.mark.parametrize("cap", [1021, 1024, 1025, 1047, 2047, 2049])
def test_caps_around_the_looking_iterations(gpu_available, tmp_path, cap):
    """The owner kernels look for cycles in the last 6 of 64 iterations, the
    shared launch in passes of the last 16 of 1,024."""
    kinds = ["random", "sparse", "long rows"]
    graphs = [graph(k, tmp_path) for k in kinds]
    for kind, g in zip(kinds, graphs):
        check(kind, g, cap, None, localOwnerAfter=1)
        check(kind, g, cap, None, localOwnerAfter=1, maskOwnerMax=-1)
    want = [oracle_run(k, g, cap) for k, g in zip(kinds, graphs)]
    with L.Multi(graphs, [L.make_config(g, maxIterations=cap) for g in graphs]) as m:
        m.run_all()
        m.synchronize()
        for i, g in enumerate(graphs):
            got = [(s["iterations"], s["updates"])
                   for s in (m.stats(i, b) for b in range(g.numBatches))]
            assert got == [r[1:] for r in want[i]], kinds[i]
            assert np.array_equal(bits(m.labels(i)), want[i][-1][0]), kinds[i]


def test_moving_frontier_leaves_the_lds_kernels(gpu_available):
    """A frontier that leaves one LDS working set after another goes on in
    launches for a while and comes back: engine switches in the middle of a
    batch, oracle results."""
    inp, cap = L.generate(70000, 3, 5, 7), 1500
    with L.Context(inp, L.make_config(inp, maxIterations=cap)) as ctx:
        orc = Oracle(inp, maxIterations=cap)
        ctx.set_profiling(True)
        ctx.reset()
        for b in range(inp.numBatches):
            ctx.run_batch(b)
            orc.run_batch(b)
            st, ost = ctx.stats(b), orc.stats()
            assert (st["iterations"], st["updates"]) == (ost["iterations"], ost["updates"])
            assert np.array_equal(bits(ctx.labels()), bits(orc.labels())), f"batch {b}"
        p = ctx.prop_profile()
        assert p["localLaunches"] > 0 and p["launches"] > 256


@pytest.mark.parametrize("degree,sizes,seed", [(4, (8091, 8727), 9), (4, (5968, 7766), 16),
                                               (5, (6375, 6789), 7)])
def test_growing_core_stays_in_the_lds_kernels(gpu_available, degree, sizes, seed):
    """A small frontier whose core still grows is not one that moves: every
    iteration of the last batch runs in the LDS kernels, to the iteration
    cap, with the oracle's results."""
    cap = 1500
    inp = L.generate_stream(70001, degree, [0, *sizes], seed)
    orc = Oracle(inp, maxIterations=cap)
    with L.Context(inp, L.make_config(inp, maxIterations=cap)) as ctx:
        for b in range(inp.numBatches):
            ctx.set_profiling(1)
            ctx.run_batch(b)
            orc.run_batch(b)
            st, ost = ctx.stats(b), orc.stats()
            assert (st["iterations"], st["updates"]) == (ost["iterations"], ost["updates"])
            assert np.array_equal(bits(ctx.labels()), bits(orc.labels())), f"batch {b}"
        assert max(orc.frontier_sizes()) <= ctx.tuning()["localThreshold"]
        p = ctx.prop_profile()
        assert st["iterations"] == cap and p["localLaunches"] > 0 and p["launches"] == 0
