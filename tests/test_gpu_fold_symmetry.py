"""Which plans fold: the folded form uses that every block is the reflection of
its class's representative and, along the axes on which a case vector is zero,
that a representative is its own reflection.  Tables without the latter keep
the general form; each is compared with the oracle.

Tolerance as in ``test_gpu_fold``: FP64 sums of the same products in another
order.
"""

import ctypes
import dataclasses

import numpy as np
import pytest
import torch

from oracle import list1_ref, orbit_ref
from tests.gpu_helpers import adaptive, rel_errors
from tests.test_gpu_fold import TOL
from volumential_amd import _capi, orbit, tree as vtree
from volumential_amd.kernels import AxisTargetDerivative, HelmholtzKernel, LaplaceKernel
from volumential_amd.payload import DevicePayload
from volumential_amd.plan import List1Plan
from volumential_amd.table import DuffyBuildConfig, NearFieldInteractionTable
from volumential_amd.wrangler import NearFieldWrangler

pytestmark = pytest.mark.gpu


def folded(plan):
    out = ctypes.c_int(-1)
    _capi.check(_capi.lib().vl1_plan_folded(plan.handle, ctypes.byref(out)), "vl1_plan_folded")
    return bool(out.value)


def unfolded_axes(dim, q):
    """Descriptors whose zero axes keep all q^2 node pairs (sign +1)."""
    m = orbit.build_case_metadata(dim, q)
    sign = np.where(m.case_axis_sign == 0, 1, m.case_axis_sign).astype(np.int8)
    counts = [orbit.case_value_count(sign[c], m.case_axis_group[c], q) for c in m.canonical_case_ids]
    return dataclasses.replace(m, case_axis_sign=sign,
                               case_value_offsets=np.cumsum([0] + counts).astype(np.int32))


def as_dict(m, dim, q):
    d = orbit_ref.case_metadata(dim, q)
    for k in ("case_axis_perm", "case_axis_sign", "case_axis_group", "case_value_offsets",
              "case_orbit_ranks", "axis_sign_power"):
        d[k] = getattr(m, k)
    d["n_compact_entries"] = int(m.case_value_offsets[-1])
    return d


def plan_of(tr, dim, q, m, v, **kw):
    nm = np.random.default_rng(5).standard_normal((1, q**dim)).astype(v.dtype)
    pay = DevicePayload(dim, q, v[None], nm, orbit_ref.case_metadata(dim, q)["case_indices"], m)
    return List1Plan(tr, pay, scaling_mode=_capi.SCALING_CANONICAL, scaling_power=2,
                     table_root_extent=2.0, **kw), nm


def check(plan, nm, tr, dim, q, m, v, f, scale=1.0):
    got = plan.eval(torch.as_tensor(f, device="cuda"), form="f64").cpu().numpy()
    ref = list1_ref.near_field_from_tree(tr, v[None], nm, as_dict(m, dim, q), f, mode="canonical",
                                         scaling_power=2, table_root_extent=2.0)
    l2, linf = rel_errors(got * scale, ref * scale)
    assert l2 <= TOL and linf <= TOL, (l2, linf)


@pytest.mark.parametrize("dim,q", [(2, 4), (2, 5), (3, 4), (3, 5)])
def test_unfolded_zero_axes(cuda, dim, q):
    print(f"case: zero axes not folded {dim}D q={q}", flush=True)
    tr = adaptive(dim, q, max_level=3)
    m = unfolded_axes(dim, q)
    rng = np.random.default_rng(q)
    v = rng.standard_normal(m.n_compact_entries)
    plan, nm = plan_of(tr, dim, q, m, v)
    assert not folded(plan)
    check(plan, nm, tr, dim, q, m, v, rng.standard_normal((3, tr.n_points)))


@pytest.mark.parametrize("dim,q", [(2, 3), (2, 5), (3, 3), (3, 5)])
def test_middle_node_derivative_values(cuda, dim, q):
    """Signed tables of odd order with a value where both nodes lie in the
    middle of a zero derivative axis: no odd function has one."""
    print(f"case: middle-node derivative values {dim}D q={q}", flush=True)
    tr = adaptive(dim, q, max_level=3)
    m = orbit.build_case_metadata(dim, q, (0,), (1,) + (0,) * (dim - 1))
    rng = np.random.default_rng(q)
    v = rng.standard_normal(m.n_compact_entries)
    plan, nm = plan_of(tr, dim, q, m, v)
    assert not folded(plan)
    check(plan, nm, tr, dim, q, m, v, rng.standard_normal((3, tr.n_points)))


@pytest.mark.parametrize("dim,q", [(2, 4), (3, 4)])
def test_entries_near_overflow(cuda, dim, q):
    """The folded blocks add up to 64 entries: tables whose sums leave the
    range keep the general form."""
    print(f"case: entries near overflow {dim}D q={q}", flush=True)
    tr = adaptive(dim, q, max_level=3)
    m = orbit.build_case_metadata(dim, q)
    rng = np.random.default_rng(q)
    v = 1e308 * rng.uniform(0.5, 1.0, m.n_compact_entries)
    plan, nm = plan_of(tr, dim, q, m, v)
    assert not folded(plan)
    # (the norms' squares stay in range at 2^-600)
    check(plan, nm, tr, dim, q, m, v, 1e-10 * rng.standard_normal((3, tr.n_points)), 2.0**-600)


@pytest.mark.parametrize("kernel", ["laplace", "gradient", "helmholtz", "helmholtz gradient"])
@pytest.mark.parametrize("dim,q", [(2, 4), (2, 5), (3, 3), (3, 4), (3, 5)])
def test_built_tables_fold(cuda, dim, q, kernel):
    """The library's own tables have the symmetry to rounding."""
    print(f"case: built {kernel} table folds {dim}D q={q}", flush=True)
    tr = vtree.uniform_tree(dim, q, 2)
    k = HelmholtzKernel(dim, 3.0) if "helmholtz" in kernel else LaplaceKernel(dim)
    if "gradient" in kernel:
        k = AxisTargetDerivative(dim - 1, k)
    t = NearFieldInteractionTable(q, dim, k,
                                  source_box_extent=tr.root_extent / (4 if k.is_complex_valued else 1))
    t.build_table(DuffyBuildConfig(regular_quad_order=12, radial_quad_order=21))
    w = NearFieldWrangler(tr, t)
    assert folded(w.get_plan(w.target_kernels[0], tr.target_boxes, tr.neighbor_source_boxes_starts,
                             tr.neighbor_source_boxes_lists))


@pytest.mark.parametrize("gradient", [False, True])
@pytest.mark.parametrize("dim,q", [(2, 6), (2, 5), (3, 4), (3, 5)])
def test_split_plans_fold(cuda, dim, q, gradient):
    print(f"case: fused split plan folds {dim}D q={q} gradient={gradient}", flush=True)
    tr = vtree.uniform_tree(dim, q, 3 if dim == 2 else 2)
    lap, hel = LaplaceKernel(dim), HelmholtzKernel(dim, 10.0 if dim == 2 else 3.0)
    if gradient:
        lap, hel = AxisTargetDerivative(0, lap), AxisTargetDerivative(0, hel)
    t = NearFieldInteractionTable(q, dim, lap, source_box_extent=tr.root_extent)
    t.build_table(DuffyBuildConfig(regular_quad_order=12, radial_quad_order=21))
    w = NearFieldWrangler(tr, {repr(hel): [t]}, target_kernels=[hel])
    assert folded(w.get_plan(hel, tr.target_boxes, tr.neighbor_source_boxes_starts,
                             tr.neighbor_source_boxes_lists, fused_split=True))
