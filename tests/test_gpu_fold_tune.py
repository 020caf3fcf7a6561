"""Tuning a folded plan: variants that are the same launch get one time."""

import pytest
import torch

from tests.gpu_helpers import adaptive, rel_errors, synthetic_table_levels
from tests.test_gpu_fold_symmetry import folded
from volumential_amd.wrangler import NearFieldWrangler

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form,S", [("f64", 0), ("split", 5), ("split_i8", 6)])
def test_folded_variants_share_times(cuda, form, S):
    print(f"case: tune a folded plan, {form}", flush=True)
    tr = adaptive(2, 6)
    w = NearFieldWrangler(tr, synthetic_table_levels(2, 6, n_tables=tr.nlevels, seed=8))
    plan = w.get_plan(w.target_kernels[0], tr.target_boxes, tr.neighbor_source_boxes_starts,
                      tr.neighbor_source_boxes_lists)
    assert folded(plan)
    f = torch.randn(4, tr.n_points, dtype=torch.float64, device="cuda")
    want = plan.eval(f, form=form, n_slices=S)
    ms = plan.tune(f, form=form, n_slices=S, reps=2)["times_ms"]
    # tile order: the only choice of the folded kernel (and of the int8 form)
    assert set(ms) == (set(range(8)) if form != "split_i8" else {0, 2})
    for v, t in ms.items():
        assert t == ms[v & 2]
    l2, linf = rel_errors(plan.eval(f, form=form, n_slices=S).cpu(), want.cpu())
    assert l2 <= 1e-12 and linf <= 1e-12
