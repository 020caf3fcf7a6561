"""The 3D node-sum table build (entries of a target point together), which rules
of more than 256 tail nodes take: against one lane per entry, |difference| <=
1e-13 max(1, |entry|) as in ``test_gpu_duffy``."""

import numpy as np
import pytest

from volumential_amd import duffy
from volumential_amd.kernels import (AxisSourceDerivative, AxisTargetDerivative, HelmholtzKernel,
                                     LaplaceKernel, RadialPowerLogKernel)
from volumential_amd.table import NearFieldInteractionTable

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q,kernel", [
    (1, LaplaceKernel(3)), (2, HelmholtzKernel(3, 5.0)), (3, AxisTargetDerivative(2, LaplaceKernel(3))),
    (4, LaplaceKernel(3)), (5, AxisSourceDerivative(0, HelmholtzKernel(3, 5.0))),
    (6, LaplaceKernel(3)), (7, RadialPowerLogKernel(3, 2)), (8, LaplaceKernel(3))])
def test_node_sum_matches_per_entry(cuda, monkeypatch, q, kernel):
    print(f"case: 3D node sum q={q} {kernel!r}", flush=True)
    t = NearFieldInteractionTable(q, 3, kernel, source_box_extent=0.75)
    ids = t.representative_entry_ids()
    ids = np.random.default_rng(q).permutation(ids)[:3000]

    def refuse(*args):
        raise AssertionError("the build by sum factorization ran")

    monkeypatch.setattr(duffy, "TENSOR_TAIL_NODES", 0)
    monkeypatch.setattr(duffy, "_tensor_values", refuse)
    a = duffy.duffy_values(t, ids, 6, 5)
    b = duffy.duffy_values(t, ids, 6, 5, segmented=False)
    assert np.all(np.isfinite(a))
    assert np.max(np.abs(a - b) / np.maximum(1.0, np.abs(b))) <= 1e-13
