"""A workspace of the one-launch SOR is cleared before words left in it could
pass for those of a later solve (csrc/solve_age.h): their tags repeat after
2^19 solves of the domain, in which the workspace need not have been written.
On the CPU: the header in a small program that is told the solves."""
import random
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "mpi-les_amd" / "csrc"
PROGRAM = """
#include <iostream>
#include "solve_age.h"
int main() {
  les::SolveAge a;
  long long last, count;
  while (std::cin >> last >> count) std::cout << a.use(last, count) << "\\n";
}
"""
REPEAT = 1 << 19  # 32 tag bits, 8192 tags per solve


@pytest.fixture(scope="module")
def ages(tmp_path_factory):
    d = tmp_path_factory.mktemp("age")
    (d / "a.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", str(CSRC), str(d / "a.cpp"), "-o", str(d / "a")],
                   check=True)

    def run(uses):
        out = subprocess.run([str(d / "a")], input="".join(f"{x} {c}\n" for x, c in uses), capture_output=True,
                             text=True, check=True).stdout
        return [int(v) for v in out.split()]

    return run


def _check(uses, cleared):
    oldest = None  # the oldest solve with words in the workspace
    for (last, count), c in zip(uses, cleared):
        if c:
            oldest = None
        first = last - count + 1
        if oldest is not None:
            assert last - oldest < REPEAT, (last, oldest)
        oldest = first if oldest is None else oldest


def test_the_tags_repeat_as_the_kernel_makes_them():
    text = (CSRC / "k_sor_res.hip").read_text()
    assert "(unsigned)a0->ctrl->res_epoch * 8192u" in text and REPEAT * 8192 == 1 << 32


def test_a_solve_exactly_one_period_later_finds_a_cleared_workspace(ages):
    """One step of the domain itself, the next 2^19 - 1 in a batch, then one of
    its own again."""
    assert ages([(1, 1), (1 + REPEAT, 1)]) == [0, 1]


def test_steps_in_a_row_clear_once_per_quarter_million(ages):
    uses = [(n, 1) for n in range(1, 600_000)]
    c = ages(uses)
    _check(uses, c)
    assert sum(c) == 2


@pytest.mark.parametrize("seed", range(10))
def test_random_uses(ages, seed):
    rng = random.Random(seed)
    last, uses = 0, []
    for _ in range(2000):
        count = rng.choice([1, 1, 5, 65])
        last += count + rng.choice([0, 0, 0, 1, 100, 50_000, 262_143, 262_144, 524_287, 524_288, 10 ** 6])
        uses.append((last, count))
    _check(uses, ages(uses))
