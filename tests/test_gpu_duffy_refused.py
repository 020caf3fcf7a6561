"""The 3D table build by sum factorization on inputs outside its contract: NaN
for the entries concerned, the others as before."""

import numpy as np
import pytest

from volumential_amd import _capi, duffy
from volumential_amd.kernels import HelmholtzKernel, LaplaceKernel
from volumential_amd.table import NearFieldInteractionTable

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", ["laplace", "helmholtz"])
@pytest.mark.parametrize("bad", ["range before", "range past", "mode", "max_entries"])
def test_refused_entries_are_nan(cuda, monkeypatch, bad, kernel):
    print(f"case: tensor build, {bad} {kernel}", flush=True)
    q = 11  # 1331 modes: entries of the first point past the first 1024
    t = NearFieldInteractionTable(q, 3, LaplaceKernel(3) if kernel == "laplace" else HelmholtzKernel(3, 5.0),
                                  source_box_extent=0.75)
    n = t.n_q_points
    per = [1200, 7, 5, 9]  # entries of four target points of case 0
    ids = np.concatenate([m * n + p for p, m in enumerate(np.arange(k) for k in per)])
    want = duffy.duffy_values(t, ids, 3, 3)
    refused = np.zeros(ids.size, bool)
    at = np.cumsum([0] + per)
    real = duffy._dev

    def dev(a):
        a = np.array(a)
        if a.dtype == np.int64 and bad == "range before":  # point 1 ends, point 2 begins there
            a[2] = -5
        elif a.dtype == np.int64 and bad == "range past":  # the last point's end
            a[4] = ids.size + 3
        elif a.dtype == np.int32 and bad == "mode":
            a[[3, 1202]] = [n, -1]
        return real(a)

    if bad == "range before":
        refused[at[1]:at[3]] = True
    elif bad == "range past":
        refused[at[3]:] = True
    elif bad == "mode":
        refused[[3, 1202]] = True
    else:
        refused[1024:at[1]] = True
        args = _capi.DuffyTensorArgs
        monkeypatch.setattr(_capi, "DuffyTensorArgs",
                            lambda **kw: args(**{**kw, "max_entries": 1024}))
    monkeypatch.setattr(duffy, "_dev", dev)
    got = duffy.duffy_values(t, ids, 3, 3)
    assert np.array_equal(np.isnan(got), refused)
    assert np.array_equal(got[~refused], want[~refused])
