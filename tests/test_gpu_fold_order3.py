"""3D order 3: split calls of many columns (target boxes x densities, 49152 and
more) fold fewer axes (none for real data, two for complex), other calls all.
Parity with the oracle on sampled targets.

Values, sizes and tolerance as in ``test_gpu_fold``.
"""

import numpy as np
import pytest
import torch

from oracle import list1_ref, orbit_ref
from tests.gpu_helpers import rel_errors
from tests.test_gpu_fold import TOL, _table
from tests.test_gpu_plan import _sub_tree
from volumential_amd import _capi, tree as vtree
from volumential_amd.plan import FORMS
from volumential_amd.wrangler import NearFieldWrangler

pytestmark = pytest.mark.gpu


def _case(level, n_rhs, cplx):
    tr = vtree.uniform_tree(3, 3, level)
    rng = np.random.default_rng(n_rhs)
    tr.local_ids = rng.permuted(np.tile(np.arange(27), (tr.nboxes, 1)), axis=1).ravel().astype(np.int32)
    t = _table(3, 3, cplx, tr.root_extent / 2**level if cplx else 2.0)
    f = rng.standard_normal((n_rhs, tr.n_points))
    if cplx:
        f = f + 1j * rng.standard_normal(f.shape)
    return tr, t, f, NearFieldWrangler(tr, t)


@pytest.mark.parametrize("form,level,n_rhs", [("f64", 5, 2), ("split_i8", 5, 1), ("split_i8", 5, 2),
                                              ("split", 5, 13), ("split_i8", 4, 11),
                                              ("split_i8", 4, 12), ("split", 4, 64)])
@pytest.mark.parametrize("cplx", [False, True])
def test_large_trees(cuda, cplx, form, level, n_rhs):
    print(f"case: 3D q=3 level {level} R={n_rhs} {form} {'complex' if cplx else 'real'}", flush=True)
    tr, t, f, w = _case(level, n_rhs, cplx)
    rng = np.random.default_rng(n_rhs)
    got = w.eval_direct_plan(tr.target_boxes, tr.neighbor_source_boxes_starts,
                             tr.neighbor_source_boxes_lists, torch.as_tensor(f, device="cuda"),
                             form=form, n_slices=5)[0][0].cpu().numpy()
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


def test_allocation_free_bases(cuda):
    """A form and a density count prepared by different calls, whose product
    takes another basis than either."""
    print("case: 3D q=3 4096 boxes, allocation-free across bases", flush=True)
    tr, t, f, w = _case(4, 12, False)
    plan = w.get_plan(w.target_kernels[0], tr.target_boxes, tr.neighbor_source_boxes_starts,
                      tr.neighbor_source_boxes_lists)
    fd = torch.as_tensor(f, device="cuda")
    want = plan.eval(fd, form="f64")  # 12 densities, all axes
    plan.eval(fd[:1], form="split_i8", n_slices=5)  # one density, all axes
    y = torch.zeros_like(fd)
    _capi.check(_capi.lib().vl1_plan_eval_noalloc(
        plan.handle, FORMS["split_i8"], fd.data_ptr(), fd.shape[1], 12, y.data_ptr(), y.shape[1],
        _capi.SplitOpts(n_slices=5, n_products=0), _capi.stream_handle(None)),
        "vl1_plan_eval_noalloc")
    l2, linf = rel_errors(y.cpu().numpy(), want.cpu().numpy())
    assert not torch.equal(y, want) and l2 <= TOL and linf <= TOL
