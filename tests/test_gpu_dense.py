"""Iterations over a flagged frontier (one byte per vertex, no claims) against
the oracle and against the queue iterations: sizes around the tiles of 64 and
1,024 vertices, thick and thin frontiers, the touched list made from the
stamps, the work counters and the recorded frontier sizes."""
import numpy as np
import pytest

import labelpropcuda_amd as L
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.int32)


@pytest.mark.parametrize("n,degree", [(63, 3), (64, 5), (65, 5), (257, 17), (1023, 4), (4099, 30)])
@pytest.mark.parametrize("cap", [3, 400])
def test_sizes_around_the_tiles(gpu_available, n, degree, cap):
    inp = L.generate(n, degree, 4, n)
    orc = Oracle(inp, maxIterations=cap)
    with L.Context(inp, L.make_config(inp, maxIterations=cap)) as ctx:
        ctx.set_tuning(localThreshold=-1)  # every iteration a launch
        tr = ctx.enable_trace(maxFrontierSizes=cap)
        ctx.reset()
        for b in range(inp.numBatches):
            ctx.run_batch(b)
            orc.run_batch(b)
            assert np.array_equal(tr.snapshot()["frontierSizes"], orc.frontier_sizes()), f"batch {b}"
            assert np.array_equal(bits(ctx.labels()), bits(orc.labels())), f"batch {b}"
            st, ost = ctx.stats(b), orc.stats()
            assert (st["updates"], st["accuracy"]) == (ost["updates"], ost["accuracy"])


def test_thick_and_thin_frontiers_match_the_queue(gpu_available):
    """1,200,003 vertices: batch 1 walks the flags in tiles of 1,024, the
    later ones load every vertex's row place along; a wave-tier limit below
    every hub keeps the same stream in queue iterations."""
    inp = L.generate(1200003, 5, 6, 9)
    runs = []
    for blockRowMin in (-1, 64):  # flags; queue (the graph counts as having hub rows)
        with L.Context(inp, L.make_config(inp, maxIterations=60)) as ctx:
            ctx.set_tuning(localThreshold=-1, blockRowMin=blockRowMin)
            ctx.set_profiling(True)
            ctx.run_all()
            p, f = ctx.prop_profile(), ctx.flag_profile()
            if blockRowMin < 0:  # both walks, and little else
                assert 0 < f["thinLaunches"] < f["launches"] and f["idleLaunches"] == 0
                assert 0.8 * p["edges"] < f["edges"] <= p["edges"]
            else:
                assert f == dict.fromkeys(f, 0) and p["appended"] > 0
            st = [ctx.stats(b) for b in range(inp.numBatches)]
            runs.append((bits(ctx.labels()),
                         [[s[k] for k in ("iterations", "updates", "frontier0", "numTouched",
                                          "accuracy")] for s in st],
                         p["edges"], p["changedEdges"]))
    sizes = [s[1] / max(s[0], 1) for s in runs[0][1]]
    assert min(sizes[1:]) * 16 < inp.numNodes < max(sizes) * 16
    assert np.array_equal(runs[0][0], runs[1][0])
    assert runs[0][1:] == runs[1][1:]


@pytest.mark.parametrize("n,degree", [(1 << 14, 4), ((1 << 14) + 1, 4), (1 << 16, 3),
                                      ((1 << 16) + 1, 3), (5003, 40)])
def test_vertices_a_wave_takes(gpu_available, n, degree):
    """Eight vertices a wave up to 16,384, sixteen up to 65,536, 64 beyond;
    rows of 40 entries: flagged launches against the oracle."""
    cap = 60
    inp = L.generate(n, degree, 5, n)
    orc = Oracle(inp, maxIterations=cap)
    with L.Context(inp, L.make_config(inp, maxIterations=cap)) as ctx:
        ctx.set_tuning(localThreshold=-1)
        ctx.set_profiling(1)
        for b in range(inp.numBatches):
            ctx.run_batch(b)
            orc.run_batch(b)
            st, ost = ctx.stats(b), orc.stats()
            assert (st["iterations"], st["updates"]) == (ost["iterations"], ost["updates"])
            assert np.array_equal(bits(ctx.labels()), bits(orc.labels())), f"batch {b}"
        f = ctx.flag_profile()
        assert f["launches"] > 100 and f["thinLaunches"] == 0


@pytest.mark.parametrize("n,thin", [(1 << 19, False), ((1 << 19) + 1, True), ((3 << 18) + 1, True)])
def test_walk_by_graph_size(gpu_available, n, thin):
    """Frontiers of a few thousand: beyond 524,288 vertices flags alone are
    walked, up to there every vertex's row place along with its flag."""
    inp = L.generate(n, 3, 6, 9)
    runs = []
    for blockRowMin in (-1, 64):  # flags; queue
        with L.Context(inp, L.make_config(inp, maxIterations=60)) as ctx:
            ctx.set_tuning(localThreshold=-1, blockRowMin=blockRowMin)
            ctx.set_profiling(True)
            ctx.run_all()
            st = [ctx.stats(b) for b in range(inp.numBatches)]
            f = ctx.flag_profile()
            runs.append((bits(ctx.labels()), [(s["iterations"], s["updates"]) for s in st]))
        if blockRowMin < 0:
            assert f["launches"] > 0 and (f["thinLaunches"] > 0) == thin
    assert np.array_equal(runs[0][0], runs[1][0]) and runs[0][1] == runs[1][1]


@pytest.mark.parametrize("cap,flagged", [(6, 0), (7, 1), (60, 54)])
def test_flags_are_set_up_for_long_excursions(gpu_available, cap, flagged):
    """The first six launches of a batch take the queue, in chunks of one, two or doubling."""
    inp = L.generate(5000, 5, 4, 42)
    orc = Oracle(inp, maxIterations=cap)
    for b in range(3):
        orc.run_batch(b)
    for chunk in (1, 2, 1024):
        with L.Context(inp, L.make_config(inp, maxIterations=cap)) as ctx:
            ctx.set_tuning(localThreshold=-1, chunk=chunk)
            ctx.run_batch(0)
            ctx.run_batch(1)
            ctx.set_profiling(1)
            ctx.run_batch(2)
            ctx.synchronize()
            assert (ctx.prop_profile()["launches"], ctx.flag_profile()["launches"]) == (cap, flagged)
            assert np.array_equal(bits(ctx.labels()), bits(orc.labels()))
