"""Fields read back to pageable memory: those large enough to go through the
pinned slots (8 MiB and more) as well as small ones, from several threads at
once, hold what was uploaded."""
import threading

import numpy as np
import pytest

from lesamd import api, layout, setup_gen

pytestmark = pytest.mark.gpu


def _round_trips(dims, seed, out):
    try:
        d = api.Domain(setup_gen.build(setup_gen.small_workload(*dims, seed=3), dense=False))
        rng = np.random.default_rng(seed)
        for f in ("u", "p", "sm"):
            a = np.asfortranarray(rng.standard_normal(layout.new_field(f, *dims).shape).astype(np.float32))
            d.upload(f, a)
            for _ in range(2):
                assert np.array_equal(d.download(f), a), f
        d.close()
        out.append(None)
    except BaseException as e:  # noqa: BLE001 (reported by the main thread)
        out.append(e)


# 32 KiB; just below and above 8 MiB; more chunks than slots (2 MiB x 16)
SIZES = [(20, 18, 16), (125, 125, 127), (130, 129, 126), (250, 203, 200)]


@pytest.mark.parametrize("dims", SIZES, ids=lambda d: "x".join(map(str, d)))
def test_download_returns_the_upload(dims):
    print(f"\n[transfer] {dims}", flush=True)
    out = []
    _round_trips(dims, 1, out)
    assert out == [None]


def test_downloads_from_several_threads():
    print("\n[transfer] four threads, then the slots given back", flush=True)
    for _ in range(2):
        out = []
        th = [threading.Thread(target=_round_trips, args=((140, 130, 128), q, out)) for q in range(4)]
        for t in th:
            t.start()
        for t in th:
            t.join()
        assert out == [None] * 4
        api.release_all()
