"""The decision of the one-launch SOR (k_sor_res) to solve by tickets when its
blocks are not all running in time, forced with LES_SOR_RESIDENT=3 (each block
waits for one block more than the launch has; 4: until one such solve is noted),
and what the domain does after it: the next steps run the launch-per-iterations
kernels, twice as many after each further solve of that kind, then one step
tries the one launch again.  Fields bit for bit as with
LES_SOR_RESIDENT=0, the stop-test sums to the rounding of their order."""
import dataclasses
import os

import numpy as np
import pytest

from lesamd import api, setup_gen

pytestmark = pytest.mark.gpu
FIELDS = ("p", "u", "v", "w", "rhs")
PAUSE = 256  # steps without the one-launch solve after the first that went by tickets
PROBE = 32   # ... and after the step that tries it again


def _domain(s, mode):
    os.environ["LES_SOR_RESIDENT"] = str(mode)
    try:
        return api.Domain(s)
    finally:
        os.environ.pop("LES_SOR_RESIDENT")


def _same(a, b, tag):
    for f in FIELDS:
        assert np.array_equal(a.download(f), b.download(f)), (tag, f)
    sa, sb = a.press_stats(), b.press_stats()
    assert (sa["iters"], sa["nonfinite"]) == (sb["iters"], sb["nonfinite"]), tag
    np.testing.assert_allclose(sa["sor"], sb["sor"], rtol=1e-12, atol=0)


@pytest.mark.parametrize("graph", [False, True], ids=["eager", "graph"])
@pytest.mark.parametrize("dims", [(40, 28, 14), (61, 27, 13)], ids=["even", "odd"])
def test_a_solve_without_room_pauses_the_one_launch_form(dims, graph):
    s = setup_gen.build(dataclasses.replace(setup_gen.small_workload(*dims, seed=3), nmaxp=6), dense=False)
    print(f"\n[sor fallback] {dims} graph {graph}", flush=True)
    ref, dom = _domain(s, 0), _domain(s, 3)
    dom.set_graph(graph)
    nmax = 4 * PAUSE + 8
    seen = []
    for n in range(1, nmax + 1):
        ref.step(n, nmax)
        dom.step(n, nmax)
        seen.append(dom.solve_fallbacks())  # waits, so that the next step knows
        if n < 4 or n > nmax - 2 or seen[-1] != seen[-2]:
            _same(ref, dom, n)
    # one at step 1, the next after the pause, the one after that after twice the pause
    assert [n + 1 for n in range(nmax) if n == 0 or seen[n] != seen[n - 1]] == [1, PAUSE + 2, 3 * PAUSE + 3], seen
    assert seen[0] == 1 and seen[-1] == 3
    assert ref.solve_fallbacks() == 0
    ref.close()
    dom.close()


@pytest.mark.parametrize("graph", [False, True], ids=["eager", "graph"])
def test_room_again_brings_the_one_launch_form_back(graph):
    """The first solve finds no room, later ones do.  The launches per step
    tell the form: one SOR launch in the one-launch form."""
    s = setup_gen.build(dataclasses.replace(setup_gen.small_workload(40, 28, 14, seed=9), nmaxp=6), dense=False)
    print(f"\n[sor fallback] room again, graph {graph}", flush=True)
    ref, dom = _domain(s, 0), _domain(s, 4)
    dom.set_graph(graph)
    nmax = PAUSE + PROBE + 12
    for n in range(1, nmax + 1):
        ref.step(n, nmax)
        at = (1, 2, PAUSE + 1, PAUSE + 2, PAUSE + 3, PAUSE + PROBE + 1, PAUSE + PROBE + 2, nmax)
        if n in at:
            dom.set_timing(True)
        dom.step(n, nmax)
        if n in at:
            kt = dom.timing()
            one = (kt["sor"][1], kt["sor1"][1]) == (1, 0)
            dom.set_timing(False)
            assert one == (n in (1, PAUSE + 2, PAUSE + PROBE + 2, nmax)), n
            _same(ref, dom, n)
        assert dom.solve_fallbacks() == 1
    ref.close()
    dom.close()


def test_steps_enqueued_before_the_pause_all_complete():
    s = setup_gen.build(dataclasses.replace(setup_gen.small_workload(40, 28, 14, seed=5), nmaxp=6), dense=False)
    print("\n[sor fallback] enqueued ahead", flush=True)
    ref, dom = _domain(s, 0), _domain(s, 3)
    dom.set_graph(True)
    ref.run(1, 12, 12)
    dom.run(1, 12, 12)
    _same(ref, dom, 12)
    n = dom.solve_fallbacks()
    assert 1 <= n <= 12
    dom.step(13, 20)  # one pause for all of them
    ref.step(13, 20)
    _same(ref, dom, 13)
    assert dom.solve_fallbacks() == n
    ref.close()
    dom.close()


def test_inner_solves_of_the_defect_correction_without_room():
    s = setup_gen.build(dataclasses.replace(setup_gen.small_workload(40, 28, 14, seed=7), pjuge=1e-30), dense=False)
    print("\n[sor fallback] defect correction", flush=True)
    ref, dom = _domain(s, 0), _domain(s, 3)
    for d in (ref, dom):
        d.set_press_mode(1, outer=3, inner=4)
    for n in (1, 2, 3):
        for d in (ref, dom):
            d.step(n, 3)
        _same(ref, dom, n)
        assert dom.solve_fallbacks() == 3
    ref.close()
    dom.close()


@pytest.mark.parametrize("graph", [False, True], ids=["eager", "graph"])
def test_a_batch_pauses_as_one(graph):
    """One domain of the batch finds no room: all of them change over, and
    back, together."""
    setups = [setup_gen.build(dataclasses.replace(setup_gen.small_workload(*d, seed=11), nmaxp=6), dense=False)
              for d in ((40, 28, 14), (33, 26, 17), (24, 21, 12))]
    print(f"\n[sor fallback] batch graph {graph}", flush=True)
    refs = [_domain(s, 0) for s in setups]
    doms = [_domain(s, 3 if q == 1 else 1) for q, s in enumerate(setups)]
    b = api.Batch(doms, graph=graph)
    nmax = PAUSE + 6
    seen = []
    for n in range(1, nmax + 1):
        b.step([n] * 3, [nmax] * 3)
        for r in refs:
            r.step(n, nmax)
        b.synchronize()
        seen.append(doms[1].solve_fallbacks())
        if n < 4 or n > nmax - 2 or seen[-1] != seen[-2]:
            for q, (r, d) in enumerate(zip(refs, doms)):
                _same(r, d, (n, q))
    assert [n + 1 for n in range(nmax) if n == 0 or seen[n] != seen[n - 1]] == [1, PAUSE + 2], seen
    assert doms[0].solve_fallbacks() == doms[2].solve_fallbacks() == 0
    b.close()
    for d in refs + doms:
        d.close()
