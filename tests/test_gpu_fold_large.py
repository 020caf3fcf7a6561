"""Folded plans on trees whose boxes lie beyond 32-bit byte offsets at eight
densities per tile: few boxes are listed, the others are numbers only.

Tolerance as in ``test_gpu_fold``: FP64 sums of the same products in another
order.
"""

import types

import numpy as np
import pytest
import torch

from oracle import list1_ref, orbit_ref
from tests.gpu_helpers import rel_errors
from tests.test_gpu_fold import TOL, _table
from volumential_amd import _capi, tree as vtree
from volumential_amd.payload import DevicePayload
from volumential_amd.plan import List1Plan

pytestmark = pytest.mark.gpu


def _scattered(tr, nb, seed):
    """`tr` with its boxes renumbered among nb, the first and the last number
    among them; box numbers in between hold no points and are not listed."""
    rng = np.random.default_rng(seed)
    at = rng.choice(np.arange(1, nb - 1), tr.nboxes - 2, replace=False)
    at = np.concatenate([[nb - 1, 0], at])
    centers = np.zeros((tr.dim, nb))
    centers[:, at] = tr.box_centers
    levels = np.zeros(nb, np.uint8)
    levels[at] = tr.box_levels
    starts, counts = np.zeros((2, nb), np.int32)
    starts[at] = tr.box_target_starts
    counts[at] = tr.box_target_counts_nonchild
    return types.SimpleNamespace(
        dim=tr.dim, root_extent=tr.root_extent, box_centers=centers, box_levels=levels,
        box_target_starts=starts, box_target_counts_nonchild=counts, local_ids=tr.local_ids,
        target_boxes=at[np.asarray(tr.target_boxes)].astype(np.int32),
        neighbor_source_boxes_starts=tr.neighbor_source_boxes_starts,
        neighbor_source_boxes_lists=at[np.asarray(tr.neighbor_source_boxes_lists)].astype(np.int32))


@pytest.mark.parametrize("dim,q,level,nb", [(2, 8, 3, (1 << 20) + 5), (3, 6, 2, 299600)])
def test_boxes_beyond_offsets(cuda, dim, q, level, nb):
    print(f"case: folded {dim}D q={q} R=8, {nb} box numbers", flush=True)
    tr = vtree.uniform_tree(dim, q, level)
    t = _table(dim, q, False)
    f = np.random.default_rng(nb).standard_normal((8, tr.n_points))
    plan = List1Plan(_scattered(tr, nb, dim), DevicePayload(
        dim, q, t.compact_values()[None], t.mode_normalizers[None], t.case_indices,
        t.arithmetic_metadata()),
                     scaling_mode=_capi.SCALING_CANONICAL, log_displacement=dim == 2,
                     table_root_extent=2.0)
    got = plan.eval(torch.as_tensor(f, device="cuda"), form="f64").cpu().numpy()
    ref = list1_ref.near_field_from_tree(
        tr, t.compact_values()[None], t.mode_normalizers[None], orbit_ref.case_metadata(dim, q), f,
        mode="canonical", scaling_power=2, log_displacement=dim == 2, table_root_extent=2.0)
    l2, linf = rel_errors(got, ref)
    assert l2 <= TOL and linf <= TOL, (l2, linf)
