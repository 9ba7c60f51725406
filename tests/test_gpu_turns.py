"""One-launch solves beside steps of other domains: a step that holds one runs
after the steps enqueued before it, on whatever stream, so its blocks find the
device free (no solve falls back to the slow form), and every domain gets the
results it has alone."""
import os
import threading

import numpy as np
import pytest

from lesamd import api, setup_gen

pytestmark = pytest.mark.gpu
FIELDS = ("u", "v", "w", "p")


def _domain(s, mode=1):
    os.environ["LES_SOR_RESIDENT"] = str(mode)
    try:
        d = api.Domain(s)
    finally:
        os.environ.pop("LES_SOR_RESIDENT")
    d.set_graph(True)
    return d


def _setup(dims, seed):
    return setup_gen.build(setup_gen.Workload("turns", *dims, dt=0.02, seed=seed), dense=False)


def _alone(s, n, mode=1):
    d = _domain(s, mode)
    d.run(1, n, n)
    out = {f: d.download(f) for f in FIELDS}
    d.close()
    return out


def _check(d, want, tag):
    for f in FIELDS:
        assert np.array_equal(d.download(f), want[f]), (tag, f)
    assert d.solve_fallbacks() == 0, tag


def test_steps_enqueued_before_the_first_one_launch_domain_exists():
    """A large domain without the one-launch solve has its steps enqueued when
    the first domain with one is created and steps: 504 boxes of 22 levels,
    two to a compute unit, which fit only where nothing else runs."""
    big, res = _setup((320, 320, 128), 3), _setup((320, 256, 128), 4)
    print("\n[turns] enqueued before", flush=True)
    want = _alone(res, 3)
    api.release_all()
    p = _domain(big, 0)
    p.run(1, 30, 60)
    q = _domain(res)
    for n in range(1, 4):
        q.step(n, 3)
        p.step(30 + n, 60)
    _check(q, want, "one-launch domain")
    p.synchronize()
    p.close()
    q.close()


def test_a_batch_beside_domains_on_their_own_streams():
    """As a server of mixed sizes steps them: a batch that solves in one launch,
    a domain that does and one that does not, bursts of steps of each in turn."""
    dims = [(96, 96, 64), (128, 96, 64), (60, 40, 20)]
    setups = [_setup(d, 5 + q) for q, d in enumerate(dims)]
    own = [(_setup((192, 160, 64), 8), 1), (_setup((200, 160, 64), 9), 0)]
    nsteps = 12
    print("\n[turns] batch and domains", flush=True)
    want = [_alone(s, nsteps) for s in setups]
    want_own = [_alone(s, nsteps, m) for s, m in own]
    doms, singles = [_domain(s) for s in setups], [_domain(s, m) for s, m in own]
    b = api.Batch(doms)
    for n0 in range(1, nsteps + 1, 4):
        for n in range(n0, n0 + 4):
            b.step([n] * len(doms), [nsteps] * len(doms))
        for d in singles:
            d.run(n0, n0 + 3, nsteps)
    b.synchronize()
    for q, (d, w) in enumerate(zip(doms + singles, want + want_own)):
        _check(d, w, q)
    b.close()
    for d in doms + singles:
        d.close()


def test_threads_step_tune_and_build_at_once():
    """Domains stepped by a thread each (with and without the one-launch solve)
    while another thread builds, tunes, steps and closes more of them."""
    shapes = [((96, 80, 32), 1), ((88, 72, 32), 0), ((61, 47, 20), 1)]
    setups = [_setup(d, 11 + q) for q, (d, _) in enumerate(shapes)]
    nsteps = 40
    print("\n[turns] threads", flush=True)
    want = [_alone(s, nsteps, m) for s, (_, m) in zip(setups, shapes)]
    extra = [_setup((40 + 4 * q, 30, 16), 21 + q) for q in range(4)]
    want_extra = [_alone(s, 4) for s in extra]
    doms = [_domain(s, m) for s, (_, m) in zip(setups, shapes)]
    made = [_domain(s) for s in extra]  # built here: the environment is read then
    errors = []

    def step(d):
        try:
            for n in range(1, nsteps + 1):
                d.step(n, nsteps)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    def tune():
        try:
            for d, w in zip(made, want_extra):
                d.autotune(reps=3)
                d.time_sor(10)
                d.run(1, 4, 4)
                _check(d, w, "tuned")
                d.close()
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    ts = [threading.Thread(target=step, args=(d,)) for d in doms] + [threading.Thread(target=tune)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors
    for q, (d, w) in enumerate(zip(doms, want)):
        _check(d, w, q)
        d.close()
