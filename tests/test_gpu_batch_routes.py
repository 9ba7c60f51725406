"""The batched and tuned paths of domains that do not solve in one launch
(LES_SOR_RESIDENT=0: one SOR iteration per launch for the whole batch, its
first steps and joins, the tuned launch shapes), and batches of both kinds."""
import dataclasses
import os

import numpy as np
import pytest

import test_gpu_batch as batch
from lesamd import api, setup_gen

pytestmark = pytest.mark.gpu


@pytest.fixture
def per_iteration(monkeypatch):
    monkeypatch.setenv("LES_SOR_RESIDENT", "0")


@pytest.mark.parametrize("graph", [True, False], ids=["graph", "eager"])
def test_batch_equals_alone(graph, per_iteration, monkeypatch):
    batch.test_batch_equals_alone(graph, False, monkeypatch)


def test_batch_staggered_joins(per_iteration, monkeypatch):
    batch.test_batch_staggered_joins(monkeypatch)


@pytest.mark.parametrize("case", [dict(im=90, jm=40, km=24, seed=31), dict(im=61, jm=27, km=18, seed=32)],
                         ids=lambda c: f"{c['im']}x{c['jm']}x{c['km']}")
def test_a_tuned_domain_steps_like_an_untuned_one(case, per_iteration):
    s = setup_gen.build(setup_gen.small_workload(**case))
    print(f"\n[tuned, per iteration] {case}", flush=True)
    a, b = api.Domain(s), api.Domain(s)
    r = a.autotune(reps=4)
    assert r["rows"] in ((1, 2, 4) if case["jm"] % 2 == 0 else (1,)), r
    assert 0.0 < r["us_per_iter"] <= r["us_per_iter_default"], r
    for n in range(1, 5):
        a.step(n, 4)
        b.step(n, 4)
    for f in batch.FIELDS:
        assert np.array_equal(a.download(f), b.download(f)), f
    x, y = a.press_stats(), b.press_stats()
    assert x["iters"] == y["iters"]
    np.testing.assert_allclose(x["sor"], y["sor"], rtol=1e-12, atol=0)
    a.close()
    b.close()


@pytest.mark.parametrize("graph", [True, False], ids=["graph", "eager"])
def test_a_batch_of_both_kinds(graph):
    """Domains whose grid is uniform in i and j solve in one launch, the others
    of the batch (cn2l or cn3s not uniform, the one-launch form off) one
    iteration per launch, all of them staged: each as alone, first steps, joins
    and caps included."""
    setups = []
    for q, (im, jm, km) in enumerate(((40, 28, 14), (48, 30, 20), (33, 26, 17), (36, 22, 14), (64, 40, 12))):
        w = dataclasses.replace(setup_gen.small_workload(im, jm, km, seed=61 + q), nmaxp=(50, 7, 50, 1, 20)[q])
        s = setup_gen.build(w, dense=False)
        if q in (1, 2):  # cn1 follows from the metrics, so the press stays the defined one
            c = dict(s.coeffs)
            name = "cn2l" if q == 1 else "cn3s"
            c[name] = c[name].copy()
            c[name][5] *= np.float32(1.125)
            s = dataclasses.replace(s, coeffs=c)
        setups.append(s)

    def make(q, mode):
        os.environ["LES_SOR_RESIDENT"] = str(mode)
        try:
            return api.Domain(setups[q])
        finally:
            os.environ.pop("LES_SOR_RESIDENT")

    print(f"\n[batch both kinds] graph {graph}", flush=True)
    n = len(setups)
    alone = [make(q, 0) for q in range(n)]
    doms = [make(q, 0 if q == 4 else 1) for q in range(n)]
    start = [0, 0, 0, 2, 2]  # the step of the batch's clock after which each joins
    last, members, b = 6, None, None
    for t in range(1, last + 1):
        act = [q for q in range(n) if t > start[q]]
        if act != members:
            if b is not None:
                b.close()
            b, members = api.Batch([doms[q] for q in act], graph=graph), act
        b.step([t - start[q] for q in act], [last] * len(act))
        for q in act:
            alone[q].step(t - start[q], last)
    b.synchronize()
    for q in range(n):
        for f in batch.FIELDS:
            assert np.array_equal(alone[q].download(f), doms[q].download(f)), (q, f)
        x, y = alone[q].press_stats(), doms[q].press_stats()
        assert (x["iters"], x["nonfinite"]) == (y["iters"], y["nonfinite"]), q
        np.testing.assert_allclose(x["sor"], y["sor"], rtol=1e-12, atol=0)
        assert doms[q].solve_fallbacks() == 0
    b.close()
    for d in alone + doms:
        d.close()
