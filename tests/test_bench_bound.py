"""CPU: the bound that bench.py names for a per-ray kernel comes from counters where there are some,
else from the counted operations, and is unknown without either.
"""
import importlib.util
from pathlib import Path
from types import SimpleNamespace

import pytest


@pytest.fixture(scope="module")
def bench():
    spec = importlib.util.spec_from_file_location(
        "bench_bound", Path(__file__).resolve().parent.parent / "bench.py")
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


@pytest.mark.parametrize("visits,facts,bound", [
    (None, {}, None), (10, {}, "hbm"), (10 ** 9, {}, "valu"),
    (None, {"valu-busy": 0.7, "traffic-per-launch": 1e6}, "valu"),
    (None, {"valu-busy": 0.01, "traffic-per-launch": 7e9}, "hbm")])
def test_bound(bench, monkeypatch, visits, facts, bound):
    monkeypatch.setattr(bench, "profile_facts", lambda *_: facts)
    st = None if visits is None else SimpleNamespace(visits=visits, tests=0, culls=0, rays=1,
                                                     chains=0)
    out = bench.per_ray_roofline("k", 1.0, 10 ** 6, 1000, 0, "none", st)
    assert out["bound"] == bound
