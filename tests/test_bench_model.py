"""bench.py's byte models and engine split, on figures made up for the test."""
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)


@pytest.fixture
def bench(monkeypatch):
    """bench.py, which sets the hardware queue count on import."""
    monkeypatch.setenv("GPU_MAX_HW_QUEUES", os.environ.get("GPU_MAX_HW_QUEUES", "4"))
    monkeypatch.setattr(sys, "argv", ["bench.py"])
    sys.modules.pop("bench", None)
    import bench
    return bench


def test_flagged_and_queue_launches_are_priced_apart(bench):
    prof = dict(launches=110, kernelMs=3.0, edges=7000, changedEdges=3000, appended=40,
                localLaunches=2, localKernelMs=1.0, localUpdates=500, localEdges=3000,
                localChangedEdges=100, localAppended=10)
    flags = dict(launches=100, thinLaunches=0, idleLaunches=20, updates=900, edges=6000,
                 changedEdges=2000, kernelMs=2.0)
    p = bench.with_flags(prof, flags)
    assert (p["launches"], p["kernelMs"], p["edges"], p["changedEdges"]) == (10, 1.0, 1000, 1000)
    eng = bench.engine_rooflines(p, 1600, 5000)
    assert set(eng) == {"k_dense", "k_propagate", "k_propagate_local"}
    d, q = eng["k_dense"], eng["k_propagate"]
    assert d["launches_per_step"] == 80 and d["avg_launch_us"] == 25.0
    assert d["algorithmic_bytes_per_launch"] * 80 == 5000 * 80 + 21 * 900 + 12 * 6000 + 2000
    assert q["algorithmic_bytes_per_launch"] * 10 == 20 * 200 + 12 * 1000 + 4 * 1000 + 4 * 40
    rates = {"load_per_s": 1e9, "store_per_s": 1e8, "atomic_max_per_s": 1e7}
    args = (900, 6000, 2000, 80, rates)
    stores = bench.random_access_floor_us(*args, "store_per_s")
    atomics = bench.random_access_floor_us(*args, "atomic_max_per_s")
    assert abs(stores - 1e6 * (8700e-9 + 9e-6 + 2e-5) / 80) < 1e-9 and atomics > stores


def test_measured_traffic_is_read_for_every_engine(bench):
    for name in ("k_dense", "k_propagate", "k_propagate_local"):
        assert bench.measured_traffic(name) > 0
    assert bench.measured_traffic("no_such_kernel") is None
