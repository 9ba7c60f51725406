"""The server builds its domains without touching the process environment
(other threads are inside calls that read it), and a run leaves nothing behind
that changes how a later run of the same server builds them."""
import os

import pytest

from lesamd import api, serving, setup_gen


class _Stub:
    seen = []

    def __init__(self, setup):
        _Stub.seen.append({k: v for k, v in os.environ.items() if k.startswith("LES_")})
        self.handle = self

    def set_graph(self, on):
        pass

    def autotune(self):
        pass

    def step(self, n, nmax):
        pass

    def done(self):
        return True

    def close(self):
        pass


@pytest.mark.parametrize("workers", [0, 1, 2])
@pytest.mark.parametrize("preset", [None, "0", "1"])
def test_domains_are_built_with_the_users_environment(workers, preset, monkeypatch):
    if preset is None:
        monkeypatch.delenv("LES_SOR_RESIDENT", raising=False)
    else:
        monkeypatch.setenv("LES_SOR_RESIDENT", preset)
    monkeypatch.setattr(api, "Domain", _Stub)
    monkeypatch.setattr(api, "bytes_needed", lambda im, jm, km: 1)
    monkeypatch.setattr(setup_gen, "build", lambda w, dense: w)
    before = dict(os.environ)
    want = {k: v for k, v in before.items() if k.startswith("LES_")}
    sizes = [(8, 8, 4), (32, 32, 8), (8, 8, 4), (40, 40, 8)]
    reqs = serving.sample_requests(4, 3, seed=1, sizes=sizes)

    class Batch(_Stub):
        def __init__(self, doms):
            pass

    srv = serving.Server(100, workers=workers, batch_factory=Batch)
    for run in (lambda: srv.run_batched(reqs, max_batch_cells=1000), lambda: srv.run(reqs),
                lambda: srv.warm(reqs), lambda: srv.run_batched(reqs)):
        _Stub.seen = []
        run()
        assert len(_Stub.seen) >= 3
        assert all(e == want for e in _Stub.seen), _Stub.seen
        assert dict(os.environ) == before
