"""Infinities and NaN in densities of folded plans: every output is the sum
over sources, as the general form's, although the folded basis mixes mirror
nodes first."""

import numpy as np
import pytest
import torch

from oracle import list1_ref
from tests.gpu_helpers import adaptive
from tests.test_gpu_fold_symmetry import as_dict, folded, plan_of
from volumential_amd import orbit

pytestmark = pytest.mark.gpu


def _spoil(f, tr, q, rng):
    """Single infinities, two in mirror nodes of one box (equal and opposite
    signs), one in a middle node, a NaN; the last density stays finite."""
    n = tr.n_q_points
    box = rng.permutation(np.asarray(tr.target_boxes))
    at = tr.box_target_starts
    mid = (n - 1) // 2 if q % 2 else n // 2
    for r in range(f.shape[0] - 1):
        f[r, at[box[r]] + rng.integers(n)] = np.inf if r % 2 else -np.inf
    f[0, at[box[20]] + [1, n - 2]] = np.inf
    f[1, at[box[21]] + [0, n - 1]] = [np.inf, -np.inf]
    f[2, at[box[22]] + mid] = np.inf
    f[3, at[box[23]] + 1] = np.nan


@pytest.mark.parametrize("form", ["f64", "split_i8"])
@pytest.mark.parametrize("dim,q,cplx,signed", [(2, 4, False, False), (2, 5, False, False),
                                               (2, 6, True, False), (3, 3, False, False),
                                               (3, 4, False, True), (3, 5, False, False),
                                               (3, 4, True, False)])
def test_nonfinite_densities(cuda, dim, q, cplx, signed, form):
    print(f"case: non-finite densities {dim}D q={q} cplx={cplx} signed={signed} {form}", flush=True)
    tr = adaptive(dim, q, max_level=3)
    m = orbit.build_case_metadata(dim, q, *(((0,), (1,) + (0,) * (dim - 1)) if signed else ()))
    rng = np.random.default_rng(10 * dim + q)
    v = rng.standard_normal(m.n_compact_entries)
    if cplx:
        v = v + 1j * rng.standard_normal(v.size)
    plan, nm = plan_of(tr, dim, q, m, v)
    assert folded(plan)
    f = rng.standard_normal((5, tr.n_points))
    _spoil(f, tr, q, rng)
    # complex data: the spoiled values in the real parts (a complex product in
    # numpy multiplies the infinity with both parts, as the blocks do)
    fd = torch.as_tensor(f.astype(np.complex128) if cplx else f, device="cuda")
    est = torch.zeros((5, 2), dtype=torch.float64, device="cuda") if form == "split_i8" else None
    got = plan.eval(fd, form=form, error_est=est).cpu().numpy()
    # rows of [Re y; Im y] = the real sums with the tables' two parts
    parts = [v.real, v.imag] if cplx else [v]
    with np.errstate(invalid="ignore"):
        ref = [list1_ref.near_field_from_tree(tr, p[None], nm, as_dict(m, dim, q), f,
                                              mode="canonical", scaling_power=2, table_root_extent=2.0)
               for p in parts]
    got = [got.real, got.imag] if cplx else [got]
    for a, b in zip(got, ref):
        assert np.array_equal(np.isnan(a), np.isnan(b))
        inf = np.isinf(b)
        assert inf.any() and np.array_equal(a[inf], b[inf])
        ok = np.isfinite(b)
        # outputs of finite sums only: 27 x 125 products
        assert np.abs(a[ok] - b[ok]).max() <= 1e-12 * np.abs(b[ok]).max()
    if est is not None:
        e = est.cpu().numpy()
        assert np.isnan(e[:4]).all() and (e[4] > 0).all() and (e[4] <= 1e-15).all()
