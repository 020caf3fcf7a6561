"""The plain route's FP64-MFMA kernel at the edges of its tiles: one to four
column tiles, chunks of 32 and 64 source particles, one to eight waves, more
list-1 pairs than are described at a time, ragged boxes.

Tolerance: rel-L2 and rel-Linf <= 1e-12 per density against the oracle, as for
every FP64 form (sums of at most 81 x 216 products: about 2e-14 expected).
"""

import numpy as np
import pytest
import torch

from oracle import list1_ref, orbit_ref
from tests.gpu_helpers import rel_errors, synthetic_table_levels
from volumential_amd import tree as vtree
from volumential_amd.wrangler import NearFieldWrangler

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rhs", [5, 16, 17, 33, 48, 64, 81])
@pytest.mark.parametrize("dim,q,level", [(2, 3, 3), (2, 5, 3), (3, 4, 1), (2, 9, 2), (3, 5, 1),
                                         (3, 6, 1)])
def test_column_tiles(cuda, dim, q, level, n_rhs):
    """Every list nine (2D) or ten (3D) times over: 80 pairs and more (the
    oracle takes the tree's lists, not its own)."""
    print(f"case: plain tiles {dim}D q={q} level {level} R={n_rhs}", flush=True)
    tr = vtree.uniform_tree(dim, q, level)
    st = np.asarray(tr.neighbor_source_boxes_starts)
    lists = np.asarray(tr.neighbor_source_boxes_lists)
    rep = [np.tile(lists[a:b], 9 if dim == 2 else 10) for a, b in zip(st[:-1], st[1:])]
    tr.neighbor_source_boxes_lists = np.concatenate(rep).astype(np.int32)
    tr.neighbor_source_boxes_starts = np.concatenate(
        [[0], np.cumsum([r.size for r in rep])]).astype(np.int32)
    assert max(r.size for r in rep) > 64
    rng = np.random.default_rng(q)
    tr.local_ids = np.concatenate(
        [rng.permutation(tr.n_q_points) for _ in range(tr.nboxes)]).astype(np.int32)
    table = synthetic_table_levels(dim, q, seed=q)[0]
    f = rng.standard_normal((n_rhs, tr.n_points))
    w = NearFieldWrangler(tr, table, direct_method="plain")
    pot, _ = w.eval_direct_batched(tr.target_boxes, tr.neighbor_source_boxes_starts,
                                   tr.neighbor_source_boxes_lists,
                                   torch.as_tensor(f, device="cuda"))
    pick = sorted({0, n_rhs // 2, n_rhs - 1})
    ref = list1_ref.near_field_from_tree(
        tr, np.stack([table.compact_values()]), np.stack([table.mode_normalizers]),
        orbit_ref.case_metadata(dim, q), f[pick], mode="canonical", log_displacement=dim == 2,
        table_root_extent=table.source_box_extent, table_starting_level=0, own_csr=False)
    l2, linf = rel_errors(pot[0].cpu().numpy()[pick], ref)
    assert l2 <= 1e-12 and linf <= 1e-12, (l2, linf)
