"""The FP64 sum of the cell volumes (cell_sum in runtime.hip), whose runs of
equal products are added at once, against the chain of additions it stands
for: the same bits.  Its two functions are compiled here by themselves."""
import ctypes
import pathlib
import subprocess

import numpy as np
import pytest

SRC = pathlib.Path(__file__).resolve().parents[1] / "mpi-les_amd" / "csrc" / "runtime.hip"


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    text = SRC.read_text()
    body = text[text.index("double add_repeated("):text.index("float metric_at(const les_domain* D")]
    d = tmp_path_factory.mktemp("cell_sum")
    (d / "c.cpp").write_text("#include <algorithm>\n#include <cmath>\n#include <utility>\n#include <vector>\n"
                             'extern "C" {\n' + body + """
double chain(double s, double x, long n) { for (; n > 0; n--) s = s + x; return s; }
double chain_cells(const float* dx, const float* dy, const float* dz, int im, int jm, int km) {
  double s = 0.0;
  for (int k = 0; k < km; k++)
    for (int j = 0; j < jm; j++)
      for (int i = 0; i < im; i++) s = s + (double)(dx[i] * dy[j] * dz[k]);
  return s;
}
}
""")
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", str(d / "c.cpp"), "-o", str(d / "c.so")],
                   check=True)
    so = ctypes.CDLL(str(d / "c.so"))
    for f in (so.add_repeated, so.chain):
        f.restype, f.argtypes = ctypes.c_double, [ctypes.c_double, ctypes.c_double, ctypes.c_long]
    for f in (so.cell_sum, so.chain_cells):
        f.restype, f.argtypes = ctypes.c_double, [ctypes.c_void_p] * 3 + [ctypes.c_int] * 3
    return so


def _bits(x):
    return np.float64(x).tobytes()


def test_repeated_additions(lib):
    rng = np.random.default_rng(0)
    for _ in range(3000):
        s = float(np.ldexp(rng.random(), int(rng.integers(-30, 30)))) * int(rng.integers(0, 2))
        kind = rng.integers(0, 4)
        if kind == 0:  # halves of the last place of s, and powers of two
            x = float(np.spacing(s or 1.0)) * float(rng.choice([0.25, 0.5, 0.75, 1.0, 1.5, 2.5]))
        elif kind == 1:
            x = float(np.float32(rng.random() * 100.0))
        else:
            x = float(np.ldexp(rng.random(), int(rng.integers(-60, 10))))
        n = int(rng.integers(0, 20000))
        assert _bits(lib.add_repeated(s, x, n)) == _bits(lib.chain(s, x, n)), (s, x, n)


@pytest.mark.parametrize("x", [0.0, -0.0, -3.7, float("inf"), float("nan"), 5e-324, 1e308])
def test_other_values(lib, x):
    for s in (0.0, 1.0, 1e300):
        assert _bits(lib.add_repeated(s, x, 100)) == _bits(lib.chain(s, x, 100)), (s, x)


def test_cells(lib):
    rng = np.random.default_rng(1)
    for t in range(150):
        im, jm, km = (int(v) for v in rng.integers(1, 70, 3))
        dx = np.full(im, np.float32([4.0, 0.1 + rng.random()][t % 2]))
        dy = np.full(jm, np.float32([dx[0], 1.37 * dx[0]][t // 2 % 2]))
        dz = (2.5 * np.cumprod(np.full(km, [1.0, 1.05][t // 4 % 2]))).astype(np.float32)
        if t % 5 == 1:
            dx[im // 2:] *= np.float32(1.1)
        if t % 5 == 2:
            dy[jm // 3] *= np.float32(3.0)
        if t % 5 == 3:
            dx = rng.random(im).astype(np.float32)
        args = [a.ctypes.data for a in (dx, dy, dz)] + [im, jm, km]
        assert _bits(lib.cell_sum(*args)) == _bits(lib.chain_cells(*args)), t
