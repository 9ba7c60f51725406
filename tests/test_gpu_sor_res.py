"""The one-launch SOR (k_sor_res, the default where a domain fits and its grid
is uniform in i and j) against the launch-per-iterations kernels
(LES_SOR_RESIDENT=0), whose iterates are pinned to the colour sweeps: every
field bit for bit, the same iteration counts, the stop-test sums to the
rounding of their order.  Both forms of the launch: resident boxes, and the
sweeps by tickets it falls back to (LES_SOR_RESIDENT=2)."""
import dataclasses
import os

import numpy as np
import pytest

from lesamd import api, setup_gen

pytestmark = pytest.mark.gpu
FIELDS = ("p", "u", "v", "w", "rhs")


def _domain(s, **env):
    os.environ.update({k: str(v) for k, v in env.items()})
    try:
        return api.Domain(s)
    finally:
        for k in env:
            os.environ.pop(k)


def _same(a, b, n):
    for f in FIELDS:
        assert np.array_equal(a.download(f), b.download(f), equal_nan=True), (n, f)
    sa, sb = a.press_stats(), b.press_stats()
    assert (sa["iters"], sa["nonfinite"]) == (sb["iters"], sb["nonfinite"]), n
    np.testing.assert_allclose(sa["sor"], sb["sor"], rtol=1e-12, atol=0)
    return sa


# box edges: one box; a few; as many as the device takes; im and jm odd and
# even; levels per box 1 to 18; a row of 2; the largest that fits
SIZES = [(2, 2, 2), (3, 3, 3), (24, 20, 16), (23, 19, 9), (9, 2, 5), (20, 3, 7), (48, 40, 24), (65, 33, 17),
         (130, 31, 9), (16, 250, 12), (250, 29, 20), (600, 16, 11), (128, 128, 64), (203, 117, 61), (300, 300, 90)]


@pytest.mark.parametrize("mode", [1, 2], ids=["resident", "tickets"])
@pytest.mark.parametrize("dims", SIZES, ids=lambda d: "x".join(map(str, d)))
def test_equals_the_iteration_kernels(dims, mode):
    im, jm, km = dims
    w = dataclasses.replace(setup_gen.small_workload(im, jm, km, seed=3), nmaxp=9 if im >= 200 else 50)
    s = setup_gen.build(w, dense=False)
    print(f"\n[sor res] {w.name} mode {mode}", flush=True)
    ref, res = _domain(s, LES_SOR_RESIDENT=0), _domain(s, LES_SOR_RESIDENT=mode)
    res.set_graph(True)
    for n in range(1, 5):
        ref.step(n, 4)
        res.step(n, 4)
        _same(ref, res, n)
    ref.close()
    res.close()


@pytest.mark.parametrize("mode", [1, 2], ids=["resident", "tickets"])
@pytest.mark.parametrize("nmaxp,omega", [(1, 1.0), (2, 1.5), (3, 1.0), (1024, 1.0)])
def test_iteration_caps_and_relaxation(nmaxp, omega, mode):
    w = dataclasses.replace(setup_gen.small_workload(40, 28, 14, seed=41), nmaxp=nmaxp, omega=omega, pjuge=1e-30)
    s = setup_gen.build(w, dense=False)
    print(f"\n[sor res cap] {nmaxp} omega {omega} mode {mode}", flush=True)
    ref, res = _domain(s, LES_SOR_RESIDENT=0), _domain(s, LES_SOR_RESIDENT=mode)
    for n in (1, 2):
        ref.step(n, 2)
        res.step(n, 2)
        _same(ref, res, n)
    ref.close()
    res.close()


@pytest.mark.parametrize("mode", [1, 2], ids=["resident", "tickets"])
@pytest.mark.parametrize("stop_at", [1, 2, 3, 12, 49, 50])
def test_stops_where_the_iteration_kernels_stop(stop_at, mode):
    """pjuge between the residuals of iterations stop_at - 1 and stop_at of step 1."""
    base = setup_gen.small_workload(im=40, jm=28, km=14, seed=41)
    probe = _domain(setup_gen.build(dataclasses.replace(base, pjuge=1e-30), dense=False), LES_SOR_RESIDENT=0)
    probe.step(1, 2)
    h = probe.press_stats()["sor"]
    probe.close()
    lo, hi = h[stop_at - 1], min(h[: stop_at - 1]) if stop_at > 1 else 4 * h[0]
    assert lo < hi
    s = setup_gen.build(dataclasses.replace(base, pjuge=float(np.sqrt(lo * hi))), dense=False)
    print(f"\n[sor res stop] at {stop_at} mode {mode}", flush=True)
    ref, res = _domain(s, LES_SOR_RESIDENT=0), _domain(s, LES_SOR_RESIDENT=mode)
    for n in (1, 2):
        ref.step(n, 2)
        res.step(n, 2)
        st = _same(ref, res, n)
        if n == 1:
            assert st["iters"] == stop_at
    ref.close()
    res.close()


@pytest.mark.parametrize("mode", [1, 2], ids=["resident", "tickets"])
@pytest.mark.parametrize("dims", [(64, 48, 20), (61, 27, 13)], ids=["even", "odd"])
@pytest.mark.parametrize("face", ["all", "i0", "im1", "j0", "jm1", "k0", "km1", "nan"])
def test_reads_the_entry_ghosts(face, dims, mode):
    """An upload of p whose ghosts differ from their boundp copies (or a NaN
    in the interior: both solves stop at iteration 1 as diverged)."""
    w = setup_gen.Workload("sor-res-entry", *dims, seed=43)
    s = setup_gen.build(w, dense=False)
    print(f"\n[sor res entry] {face} {dims} mode {mode}", flush=True)
    ref, res = _domain(s, LES_SOR_RESIDENT=0), _domain(s, LES_SOR_RESIDENT=mode)
    for n in (1, 2):
        ref.step(n, 6)
        res.step(n, 6)
    p = ref.download("p")
    im, jm, km = dims
    faces = {"i0": np.s_[0, 1:jm + 1, 1:km + 1], "im1": np.s_[im + 1, 1:jm + 1, 1:km + 1],
             "j0": np.s_[1:im + 1, 0, 1:km + 1], "jm1": np.s_[1:im + 1, jm + 1, 1:km + 1],
             "k0": np.s_[1:im + 1, 1:jm + 1, 0], "km1": np.s_[1:im + 1, 1:jm + 1, km + 1]}
    rng = np.random.default_rng(8)
    for f in (faces if face == "all" else [face] if face in faces else []):
        p[faces[f]] += rng.uniform(-0.5, 0.5, p[faces[f]].shape).astype(np.float32)
    if face == "nan":
        p[im // 2, jm // 2, 3] = np.nan
    for d in (ref, res):
        d.upload("p", p)
        d.stage("press", 3, 6)
    _same(ref, res, 3)
    ref.close()
    res.close()


def test_domains_in_turn_and_a_grid_that_does_not_qualify():
    """Solves of several domains issued together are ordered one after the
    other (each needs the whole device); a domain whose grid is not uniform
    in i keeps the other kernels."""
    ss = [setup_gen.build(setup_gen.small_workload(*d, seed=7), dense=False) for d in ((96, 64, 32), (61, 47, 20),
                                                                                       (40, 200, 16))]
    print("\n[sor res] three domains in turn", flush=True)
    refs, ress = [_domain(s, LES_SOR_RESIDENT=0) for s in ss], [api.Domain(s) for s in ss]
    for d in ress:
        d.set_graph(True)
    for n in range(1, 9):
        for d in refs + ress:
            d.step(n, 8)
    for q, (a, b) in enumerate(zip(refs, ress)):
        _same(a, b, q)
    for d in refs + ress:
        d.close()
    s = ss[0]
    c = dict(s.coeffs, cn2l=s.coeffs["cn2l"].copy())
    c["cn2l"][5] *= np.float32(1.25)
    s = dataclasses.replace(s, coeffs=c)
    a, b = _domain(s, LES_SOR_RESIDENT=0), api.Domain(s)
    for n in (1, 2):
        a.step(n, 2)
        b.step(n, 2)
        _same(a, b, n)
    assert np.array_equal(a.press_stats()["sor"], b.press_stats()["sor"])  # the same kernel: the same order of sums
    a.close()
    b.close()


@pytest.mark.parametrize("mode", [1, 2], ids=["resident", "tickets"])
@pytest.mark.parametrize("dims,outer,inner,omega", [((40, 28, 14), 1, 1, 1.0), ((61, 27, 13), 3, 2, 1.0),
                                                    ((96, 64, 32), 2, 50, 1.0), ((40, 28, 14), 4, 7, 1.6),
                                                    ((40, 28, 14), 6, 20, 1.0)])
def test_inner_solves_of_the_defect_correction(dims, outer, inner, omega, mode):
    """The inner solves from zero (the last case meets the stop threshold of
    step 1 at its fourth norm, so later outer steps are skipped)."""
    base = dataclasses.replace(setup_gen.small_workload(*dims, seed=5), pjuge=1e-30)
    if outer == 6:
        probe = _domain(setup_gen.build(base, dense=False), LES_SOR_RESIDENT=0)
        probe.set_press_mode(1, outer=outer, inner=inner)
        probe.step(1, 3)
        h = probe.press_stats()["sor"]
        probe.close()
        assert h[3] < min(h[:3])
        base = dataclasses.replace(base, pjuge=float(np.sqrt(h[3] * min(h[:3]))))
    s = setup_gen.build(base, dense=False)
    print(f"\n[sor res dc] {dims} {outer}x{inner} omega {omega} mode {mode}", flush=True)
    ref, res = _domain(s, LES_SOR_RESIDENT=0), _domain(s, LES_SOR_RESIDENT=mode)
    for d in (ref, res):
        d.set_press_mode(1, outer=outer, inner=inner)
        d.set_press_omega(omega)
    res.set_graph(True)
    for n in range(1, 4):
        ref.step(n, 3)
        res.step(n, 3)
        st = _same(ref, res, n)
        assert outer != 6 or n > 1 or st["iters"] == 4, st["iters"]
    ref.close()
    res.close()


@pytest.mark.parametrize("dims", [(130, 50, 12), (121, 14, 17)], ids=["even", "odd im"])
def test_two_iterations_per_launch_on_either_grid(dims):
    """k_sor_pair with and without per-column coefficients against one
    iteration per launch."""
    s = setup_gen.build(setup_gen.small_workload(*dims, seed=9), dense=False)
    c = dict(s.coeffs, cn2l=s.coeffs["cn2l"].copy(), cn3s=s.coeffs["cn3s"].copy())
    c["cn2l"][5] *= np.float32(1.25)
    c["cn3s"][3] *= np.float32(0.75)
    for q, grid in enumerate((s, dataclasses.replace(s, coeffs=c))):
        print(f"\n[sor pair grid] {dims} {q}", flush=True)
        a, b = _domain(grid, LES_SOR_ROWS=2), _domain(grid, LES_SOR_ROWS=4)
        for n in (1, 2, 3):
            a.step(n, 3)
            b.step(n, 3)
            _same(a, b, n)
        a.close()
        b.close()
