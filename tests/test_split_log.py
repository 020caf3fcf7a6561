"""The split correction's logarithm, compiled for the host, against extended
precision.

Bound: rounding of 1 / c's logarithm and of e log 2 plus it (half a unit each of
a value up to twice the result's size near the interval next to 1), of the
polynomial's sum and of the result: 3 units of the last place.
"""

import ctypes
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parents[1] / "volumential_amd" / "csrc"

SOURCE = """
#include "split_log.h"
extern "C" void split_logs(const double* x, long n, double* y) {
  vl1::SplitLog t[vl1::kSplitLogs];
  for (int i = 0; i < vl1::kSplitLogs; ++i) vl1::split_log_table(t, i);
  for (long k = 0; k < n; ++k) y[k] = vl1::split_log(x[k], t);
}
"""


@pytest.fixture(scope="module")
def split_logs(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("split_log")
    (d / "s.cc").write_text(SOURCE)
    subprocess.run([gxx, "-O2", "-mfma", "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}",
                    str(d / "s.cc"), "-o", str(d / "s.so")], check=True)
    fn = ctypes.CDLL(str(d / "s.so")).split_logs

    def run(x):
        x = np.ascontiguousarray(x, dtype=np.float64)
        y = np.empty_like(x)
        fn(ctypes.c_void_p(x.ctypes.data), ctypes.c_long(x.size), ctypes.c_void_p(y.ctypes.data))
        return y

    return run


@pytest.mark.parametrize("what", ["wide", "octaves", "near 1", "closest to 1", "intervals"])
def test_relative_error(split_logs, what):
    rng = np.random.default_rng(3)
    n = 200000
    if what == "wide":  # squared distances
        x = 10.0 ** rng.uniform(-300, 300, n)
    elif what == "octaves":
        x = rng.uniform(0.25, 4.0, n)
    elif what == "near 1":
        x = 1.0 + rng.uniform(-1 / 64, 1 / 64, n)
    elif what == "closest to 1":
        x = 1.0 + 10.0 ** rng.uniform(-15, -2, n) * rng.choice([-1, 1], n)
    else:  # ends of the table's intervals and of the octave
        ends = np.concatenate([0.5 + np.arange(129) / 256, 1 + np.arange(129) / 128, [np.sqrt(0.5)]])
        x = np.concatenate([ends * s for s in (1, 2, 4, 0.125)])
        x = np.concatenate([x, np.nextafter(x, 0), np.nextafter(x, 9)])
    y, ref = split_logs(x), np.log(x.astype(np.longdouble))
    ulp = np.spacing(np.abs(ref.astype(np.float64)))
    err = np.abs(y - ref) / ulp
    assert float(err.max()) <= 3.0
    assert np.all(split_logs(np.array([1.0])) == 0.0)
