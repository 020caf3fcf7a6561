"""Tables on a host without the native library: representatives by numpy."""

import numpy as np
import pytest

from volumential_amd import _capi, orbit


@pytest.mark.parametrize("load", ["missing", "unloadable"])
@pytest.mark.parametrize("dim,q,fixed", [(2, 1, ()), (2, 4, ()), (2, 5, (1,)), (3, 2, ()), (3, 3, (0,)),
                                         (3, 4, ()), (3, 4, (2,))])
def test_representatives_without_library(monkeypatch, dim, q, fixed, load):
    power = tuple(int(a in fixed) for a in range(dim))
    m = orbit.build_case_metadata(dim, q, fixed, power)
    want = orbit.enumerate_representatives(m)

    def lib():
        raise RuntimeError("missing") if load == "missing" else OSError("libamdhip64.so: not found")

    monkeypatch.setattr(_capi, "lib", lib)
    got = orbit.enumerate_representatives(m)
    assert got.dtype == want.dtype and np.array_equal(got, want)
