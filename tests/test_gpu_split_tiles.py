"""The split correction's staging at its edges: more source boxes than are
staged together and more sources than a chunk holds, 1 to 256 targets a box, one
to nine densities, empty lists; real, damped and Yukawa wave numbers.

Lists given several times over must give that multiple of the oracle's sum:
rel <= 1e-12 as for the single lists (sums of at most 81 x 256 products).
"""

import numpy as np
import pytest
import torch

from oracle import split_ref as S
from tests.gpu_helpers import rel_errors
from volumential_amd import tree as vtree
from volumential_amd.split import HelmholtzSplitCorrection

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,q,level,k,n_rhs,times", [
    (2, 1, 3, 9.0, 1, 9), (2, 3, 2, 9.0, 4, 9), (2, 6, 2, 4.0 + 1.0j, 9, 8), (2, 16, 1, 5.0, 1, 2),
    (2, 5, 2, 3.0j, 2, 8), (3, 2, 1, 5.0, 1, 9), (3, 4, 1, 2.0 + 0.5j, 5, 9)])
def test_repeated_lists(cuda, dim, q, level, k, n_rhs, times):
    print(f"case: split staging {dim}D q={q} k={k} R={n_rhs} x{times}", flush=True)
    tr = vtree.uniform_tree(dim, q, level)
    rng = np.random.default_rng(q)
    st = (rng.standard_normal((n_rhs, tr.n_points)) + 1j * rng.standard_normal((n_rhs, tr.n_points)))
    st *= np.asarray(tr.weights)[None, :]
    starts = np.asarray(tr.neighbor_source_boxes_starts)
    lists = np.asarray(tr.neighbor_source_boxes_lists)
    keep = np.arange(starts.size - 1) % 5 != 2  # the others' lists are empty
    rep = [np.tile(lists[a:b], times if on else 0)
           for a, b, on in zip(starts[:-1], starts[1:], keep)]
    nl = np.concatenate(rep).astype(np.int32)
    ns = np.concatenate([[0], np.cumsum([r.size for r in rep])]).astype(np.int32)
    corr = HelmholtzSplitCorrection(tr, k)
    got = corr(torch.as_tensor(st, device="cuda"), tr.target_boxes, ns, nl).cpu().numpy()
    ref = times * S.correction(tr, st, k, corr.nmax)
    for b, on in zip(np.asarray(tr.target_boxes), keep):
        s = int(tr.box_target_starts[b])
        ref[:, s:s + tr.n_q_points] *= on
    l2, linf = rel_errors(got, ref)
    assert l2 <= 1e-12 and linf <= 1e-12, (l2, linf)
