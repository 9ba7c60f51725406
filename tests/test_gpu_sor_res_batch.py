"""A batched step whose domains solve side by side in one launch (k_sor_res
over a table of domains) against the same domains stepping alone with the
launch-per-iterations kernels: every field bit for bit, the same iteration
counts, the stop-test sums to the rounding of their order."""
import dataclasses
import os

import numpy as np
import pytest

from lesamd import api, setup_gen

pytestmark = pytest.mark.gpu
FIELDS = ("p", "u", "v", "w", "rhs")


def _domain(s, mode):
    os.environ["LES_SOR_RESIDENT"] = str(mode)
    try:
        return api.Domain(s)
    finally:
        os.environ.pop("LES_SOR_RESIDENT")


BATCHES = {
    "one": [(24, 20, 16)],
    "pair": [(24, 20, 16), (2, 2, 2)],
    "odd": [(23, 19, 9), (40, 27, 9), (61, 30, 9)],                       # odd im and jm
    "levels": [(40, 28, 5), (48, 40, 24), (33, 16, 18), (20, 60, 61)],    # no common division of the levels
    "nine": [(a, b, 64) for a in (96, 128, 160) for b in (96, 128, 160)],
    "two launches": [(160, 160, 64)] * 8 + [(150, 149, 90)] * 2,           # more cells than fit at once
}


@pytest.mark.parametrize("mode", [1, 2], ids=["resident", "tickets"])
@pytest.mark.parametrize("graph", [True, False], ids=["graph", "eager"])
@pytest.mark.parametrize("name", list(BATCHES))
def test_batch_equals_alone(name, graph, mode):
    if mode == 2 and (graph or name in ("nine", "two launches")):
        pytest.skip("the slow form is covered by the small batches")
    caps, relax = (50, 1, 2, 7), (1.0, 1.0, 1.4)
    setups = []
    for q, (im, jm, km) in enumerate(BATCHES[name]):
        w = setup_gen.small_workload(im, jm, km, seed=11 + q)
        if name == "levels":  # caps, relaxation and a threshold met at once, by domain
            w = dataclasses.replace(w, nmaxp=caps[q % 4], omega=relax[q % 3], pjuge=1e30 if q == 1 else 1e-30)
        elif im >= 96:
            w = dataclasses.replace(w, nmaxp=8)
        setups.append(setup_gen.build(w, dense=False))
    print(f"\n[sor res batch] {name} graph {graph} mode {mode}", flush=True)
    alone = [_domain(s, 0) for s in setups]
    doms = [_domain(s, mode) for s in setups]
    b = api.Batch(doms, graph=graph)
    for n in range(1, 5):
        b.step([n] * len(doms), [4] * len(doms))
        for d in alone:
            d.step(n, 4)
        if n == 3:  # between two batched steps a domain steps by itself as well
            alone[0].stage("press", n, 4)
            doms[0].stage("press", n, 4)
    b.synchronize()
    for q, (x, y) in enumerate(zip(alone, doms)):
        for f in FIELDS:
            assert np.array_equal(x.download(f), y.download(f)), (q, f)
        sx, sy = x.press_stats(), y.press_stats()
        assert (sx["iters"], sx["nonfinite"]) == (sy["iters"], sy["nonfinite"]), q
        np.testing.assert_allclose(sx["sor"], sy["sor"], rtol=1e-12, atol=0)
    b.close()
    for d in alone + doms:
        d.close()
