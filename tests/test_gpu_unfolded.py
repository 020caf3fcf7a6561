"""Plans whose tables lack the reflection symmetry along zero axes: the general
FP64 kernel and the digit kernels at every slice count, in each tile variant,
with row groups, complex data, forests and the allocation-free entry.

Values are random.  Tolerances: FP64 and the BF16 split (whose sums within a
diagonal are FP32) as in ``test_gpu_plan``.  The int8 form, exact but for the
products of slices i + j >= S that it drops, is off by these: 2^-8S (S + 1) of a
row's and a column's largest entries, which against sums of K = 9 n or 27 n
products of random sign is about (S + 1) 2^-8S max^2 / rms^2 with max / rms <= 4.5
for normal values: 1.1e-10 at 5 slices and 5e-13 at 6, taken ten times for the
largest of all outputs.
"""

import numpy as np
import pytest
import torch

from oracle import list1_ref
from tests.gpu_helpers import adaptive, beam_forest, rel_errors
from tests.test_gpu_fold_symmetry import as_dict, folded, unfolded_axes
from tests.test_gpu_plan import TOL64, TOLSPLIT
from volumential_amd import _capi, tree as vtree
from volumential_amd.payload import DevicePayload
from volumential_amd.plan import FORMS, List1Plan

pytestmark = pytest.mark.gpu

TOL = {("f64", 0): TOL64, ("split", 5): TOLSPLIT, ("split", 6): TOLSPLIT, ("split_i8", 5): 1.1e-9,
       ("split_i8", 6): 5e-12}
RUNS = list(TOL)


class Case:
    """An unfolded plan with per-level tables, its densities and reference."""

    def __init__(self, tr, n_rhs, cplx=False, first_level=0, seed=0, reference=True):
        dim, q = tr.dim, tr.quad_order
        m = unfolded_axes(dim, q)
        rng = np.random.default_rng(seed)

        def normal(*shape):
            v = rng.standard_normal(shape)
            return v + 1j * rng.standard_normal(shape) if cplx else v

        n_tables = tr.nlevels - first_level
        data, nm = normal(n_tables, m.n_compact_entries), normal(n_tables, q**dim)
        meta = as_dict(m, dim, q)
        extent = tr.root_extent / 2**first_level
        pay = DevicePayload(dim, q, data, nm, meta["case_indices"], m)
        self.plan = List1Plan(tr, pay, scaling_mode=_capi.SCALING_PER_LEVEL,
                              table_root_extent=extent, table_starting_level=first_level)
        assert not folded(self.plan)
        self.f = torch.as_tensor(normal(n_rhs, tr.n_points), device="cuda")
        if reference:
            self.ref = list1_ref.near_field_from_tree(
                tr, data, nm, meta, self.f.cpu().numpy(), mode="per_level",
                table_root_extent=extent, table_starting_level=first_level)

    def check(self, form, S, what=""):
        i8 = form == "split_i8"
        est = torch.zeros((self.f.shape[0], 2), dtype=torch.float64, device="cuda") if i8 else None
        got = self.plan.eval(self.f, form=form, n_slices=S, error_est=est)
        a, b = got.cpu().numpy(), self.ref
        l2, linf = rel_errors(a, b)
        tol = TOL[form, S]
        print(f"{what} {form} S={S}: {l2:.2e} {linf:.2e}", flush=True)
        assert l2 <= tol and linf <= tol, (what, form, S, l2, linf)
        if S:  # a digit kernel's error, not FP64 rounding
            assert l2 > 1e-15
        if i8:  # (rounding of the FP64 recombination aside)
            e = est.cpu().numpy()
            err = np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1)
            assert np.all(e[:, 1] + 1e-14 >= err) and np.all(e <= 20 * tol)
        return got


@pytest.mark.parametrize("what", ["2D q=6", "2D q=6 complex", "3D q=4", "3D q=3 complex",
                                  "3D q=7 row groups", "3D q=5 complex row groups", "2D q=11"])
@pytest.mark.parametrize("n_rhs", [4, 64])
def test_forms_match_oracle(cuda, what, n_rhs):
    print(f"case: unfolded {what} R={n_rhs}", flush=True)
    dim, q = int(what[0]), int(what.split("=")[1].split()[0])
    large = q**dim * (2 if "complex" in what else 1) > 200  # (adaptive: beyond exact int32 sums)
    tr = vtree.uniform_tree(dim, q, 1) if large else adaptive(dim, q, max_level=3)
    c = Case(tr, n_rhs, cplx="complex" in what, seed=q + n_rhs)
    for form, S in RUNS:
        c.check(form, S)


def test_forest(cuda):
    print("case: unfolded complex forest", flush=True)
    fo = beam_forest([0, 1], q=4, tol=1e-4, min_level=4, max_level=6)
    c = Case(fo, 3, cplx=True, first_level=4, seed=1)
    for form, S in RUNS:
        c.check(form, S)


def test_variants(cuda):
    """Every tile variant (row tiles per wave, tile order, phase alignment)."""
    print("case: unfolded, all variants", flush=True)
    c = Case(adaptive(2, 6), 4, seed=3)
    for form, S in RUNS:
        for v in range(8) if form != "split_i8" else (0, 2):
            c.plan.set_variant(v, form=form, n_slices=S, n_rhs=4)
            c.check(form, S, f"variant {v}")
        c.plan.set_variant(None, form=form, n_slices=S, n_rhs=4)


@pytest.mark.parametrize("form", ["f64", "split"])
def test_autotune(cuda, form):
    print(f"case: unfolded, autotune {form}", flush=True)
    c = Case(adaptive(2, 6), 4, seed=4)
    S = 5 if form == "split" else 0
    info = c.plan.tune(c.f, form=form, n_slices=S, reps=2)
    assert set(info["times_ms"]) == set(range(8)) and info["variant"] in info["times_ms"]
    c.check(form, S)


def test_phase_aligned_variants_repeatable(cuda):
    """Repeated evaluations with phase alignment agree with the fixed step
    order to rounding (``test_gpu_plan``'s test, on the kernels that align)."""
    print("case: unfolded, phase-aligned variants, uniform 2D q=6 level 7, 16 RHS", flush=True)
    c = Case(vtree.uniform_tree(2, 6, 7), 16, seed=5, reference=False)
    for form, S in (("f64", 0), ("split", 5)):
        for v in (0, 1, 2, 3):
            c.plan.set_variant(4 | (v & 1), form=form, n_slices=S, n_rhs=16)
            base = c.plan.eval(c.f, form=form, n_slices=S)
            c.plan.set_variant(v, form=form, n_slices=S, n_rhs=16)
            for _ in range(12):
                got = c.plan.eval(c.f, form=form, n_slices=S)
                d = ((got - base).abs().amax(dim=1) / base.abs().amax(dim=1)).max()
                assert float(d) <= 1e-13, (form, v, float(d))


@pytest.mark.parametrize("cplx", [False, True])
def test_allocation_free(cuda, cplx):
    """vl1_plan_eval_noalloc: the results of vl1_plan_eval, bit for bit, for the
    forms whose steps keep their order."""
    print(f"case: unfolded, allocation-free cplx={cplx}", flush=True)
    c = Case(adaptive(3, 4, max_level=3), 5, cplx=cplx, seed=6)
    for form, S in RUNS:
        c.plan.set_variant(4, form=form, n_slices=max(S, 1), n_rhs=5)
        want = c.check(form, S)
        y = torch.zeros_like(c.f)
        k = 2 if cplx else 1
        opts = _capi.SplitOpts(n_slices=S, n_products=0)
        _capi.check(_capi.lib().vl1_plan_eval_noalloc(
            c.plan.handle, FORMS[form], c.f.data_ptr(), c.f.shape[1] * k, 5, y.data_ptr(),
            y.shape[1] * k, opts, _capi.stream_handle(None)), "vl1_plan_eval_noalloc")
        assert torch.equal(y, want)
