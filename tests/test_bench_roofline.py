"""bench.py rates the one-launch SOR by the operations it issues, not by bytes
per iteration it does not move; a step's bytes follow the kernels it runs."""
import importlib.util
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def bench():
    spec = importlib.util.spec_from_file_location("bench_mod", ROOT / "bench.py")
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


def test_one_launch_solve_is_not_rated_by_bytes_per_iteration(bench):
    n = 300 * 300 * 90
    r = bench.sor_roofline(n, 50.0, 656e-6, True)
    assert (r["bound"], r["unit"]) == ("valu", "Top/s")
    assert r["alg_bytes_per_launch"] == 16 * n
    assert r["achieved"] == pytest.approx(17 * 50 * n / 656e-6 / 1e12, rel=1e-3)
    assert r["frac"] == pytest.approx(r["achieved"] / r["peak"], rel=1e-2) and r["frac"] < 1
    p = bench.sor_roofline(n, 2, 43e-6, False)
    assert (p["bound"], p["alg_bytes_per_launch"]) == ("hbm", 24 * n)
    assert p["frac"] == pytest.approx(24 * n / 43e-6 / 8e12, rel=1e-3)


def test_step_bytes_follow_the_kernels(bench):
    assert bench.step_bytes(1000, 50, False) == 1000 * (316 + 12 * 50)
    assert bench.step_bytes(1000, 50, True) == 1000 * (316 + 16)
