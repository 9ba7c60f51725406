"""The order of the streams' work around whole-device work (csrc/turns.h), on
the CPU: the header is compiled into a small program that is told the calls
and answers with the waits each one places; those are followed here as
happens-before edges."""
import random
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "mpi-les_amd" / "csrc"
PROGRAM = """
#include <iostream>
#include "turns.h"
int main() {
  les::Turns<int> t;
  int s, what;  // stream; 0 other work, 1 whole-device work, 2 the stream goes away, 3 whole-device work whose first wait fails
  while (std::cin >> s >> what) {
    if (what == 2) {
      t.forget(s);
      std::cout << "\\n";
      continue;
    }
    int rc = t.take(s, what != 0, [&](int a, int) {
      if (what == 3) return 1;
      std::cout << a << " ";
      return 0;
    });
    std::cout << (rc ? "failed" : "") << std::endl;
  }
}
"""


@pytest.fixture(scope="module")
def turns(tmp_path_factory):
    d = tmp_path_factory.mktemp("turns")
    (d / "t.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", str(CSRC), str(d / "t.cpp"), "-o", str(d / "t")],
                   check=True)

    def run(calls):
        text = "".join(f"{s} {w}\n" for s, w in calls)
        out = subprocess.run([str(d / "t")], input=text, capture_output=True, text=True, check=True).stdout
        return [line.split() for line in out.split("\n")[:len(calls)]]

    return run


def _check(calls, waits):
    """before[q]: the works q runs after, by its stream's order and its waits."""
    last, before, works, gone = {}, [], [], set()
    whole_stream = None
    for (s, what), w in zip(calls, waits):
        if what == 2:  # its work is complete, and so is what that ran after
            q = last.pop(s, None)
            if q is not None:
                gone |= before[q] | {q}
            continue
        b = set()
        for t in [s] + [int(x) for x in w]:
            if t in last:
                b |= before[last[t]] | {last[t]}
        for p, (t, whole) in enumerate(works):
            if t == s or p in gone:
                continue
            if whole or what == 1:
                assert p in b, (calls, len(works), p)
            elif t != whole_stream and not any(x[1] for x in works[p:]):
                assert p not in b, ("other work was ordered", calls, len(works), p)
        last[s] = len(works)
        before.append(b)
        works.append((s, what == 1))
        if what == 1:
            whole_stream = s


def test_work_enqueued_before_any_whole_device_work_is_waited_for(turns):
    """Ten steps of one stream, then the first whole-device step of another."""
    calls = [(1, 0)] * 10 + [(2, 1)]
    assert turns(calls) == [[]] * 10 + [["1"]]


def test_one_stream_alone_places_no_waits(turns):
    calls = [(1, w) for w in (1, 1, 0, 1, 0, 0, 1)]
    assert turns(calls) == [[]] * len(calls)


def test_other_work_waits_once_for_the_last_whole_device_work(turns):
    assert turns([(1, 1), (2, 0), (2, 0), (3, 0), (2, 0), (1, 1), (2, 0)]) == [[], ["1"], [], ["1"], [], ["2", "3"],
                                                                              ["1"]]


def test_a_failed_wait_leaves_the_state(turns):
    assert turns([(1, 0), (2, 3), (3, 1)]) == [[], ["failed"], ["1"]]


@pytest.mark.parametrize("seed", range(40))
def test_random_calls(turns, seed):
    rng = random.Random(seed)
    kinds = rng.choice([[0, 1], [0, 0, 0, 1], [0, 1, 1, 1, 2], [0, 0, 1, 2]])
    calls = [(rng.randrange(1, 6), rng.choice(kinds)) for _ in range(60)]
    _check(calls, turns(calls))
