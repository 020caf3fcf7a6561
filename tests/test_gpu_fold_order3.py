"""3D order 3 folds fewer axes on trees of 16384 target boxes and more (none
for real data, two for complex): parity with the oracle on sampled targets.

Values, sizes and tolerance as in ``test_gpu_fold``.
"""

import numpy as np
import pytest
import torch

from oracle import list1_ref, orbit_ref
from tests.gpu_helpers import rel_errors
from tests.test_gpu_fold import TOL, _table
from tests.test_gpu_plan import _sub_tree
from volumential_amd import tree as vtree
from volumential_amd.wrangler import NearFieldWrangler

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rhs", [1, 13])
@pytest.mark.parametrize("cplx", [False, True])
def test_large_trees(cuda, cplx, n_rhs):
    print(f"case: 3D q=3 32768 boxes R={n_rhs} {'complex' if cplx else 'real'}", flush=True)
    tr = vtree.uniform_tree(3, 3, 5)
    rng = np.random.default_rng(n_rhs)
    tr.local_ids = rng.permuted(np.tile(np.arange(27), (tr.nboxes, 1)), axis=1).ravel().astype(np.int32)
    t = _table(3, 3, cplx, tr.root_extent / 32 if cplx else 2.0)
    f = rng.standard_normal((n_rhs, tr.n_points))
    if cplx:
        f = f + 1j * rng.standard_normal(f.shape)
    w = NearFieldWrangler(tr, t)
    got = w.eval_direct_plan(tr.target_boxes, tr.neighbor_source_boxes_starts,
                             tr.neighbor_source_boxes_lists, torch.as_tensor(f, device="cuda"),
                             form="f64")[0][0].cpu().numpy()
    sel = np.sort(rng.choice(np.asarray(tr.target_boxes).size, 64, replace=False))
    nm = t.mode_normalizers[None]
    tsl = int(round(np.log2(tr.root_extent / t.source_box_extent)))
    ref = list1_ref.near_field_from_tree(
        _sub_tree(tr, sel), t.compact_values()[None], nm.astype(np.complex128) if cplx else nm,
        orbit_ref.case_metadata(3, 3), f, mode="fixed" if cplx else "canonical",
        scaling_power=0 if cplx else 2, log_displacement=False,
        table_root_extent=t.source_box_extent, table_starting_level=tsl)
    idx = np.concatenate([np.arange(tr.box_target_starts[b], tr.box_target_starts[b] + 27)
                          for b in np.asarray(tr.target_boxes)[sel]])
    l2, linf = rel_errors(got[:, idx], ref[:, idx])
    assert l2 <= TOL and linf <= TOL, (l2, linf)
