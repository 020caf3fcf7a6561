"""The 3D table build by sum factorization at the edges of its tiling: one tail
node and more than a chunk holds, one to sixteen nodes per axis, more entries
of a target point than a workgroup keeps, complex and derivative kernels.

Against the one-lane-per-entry form: |difference| <= 1e-13 max(1, |entry|), the
bound of the other builds (sums of at most 1e6 positive and negative terms of
size below 1 / nodes, about 1e-15 expected).  At 256 tail nodes that form's own
running sum is off by more (7e-13 at 2e7 nodes of one sign), and the reference
is the same sum in extended precision, axis by axis.
"""

import itertools

import numpy as np
import pytest

from volumential_amd import quadrature
from volumential_amd.duffy import duffy_values
from volumential_amd.kernels import (AxisSourceDerivative, AxisTargetDerivative, ConstantKernel,
                                     HelmholtzKernel, LaplaceKernel, RadialPowerLogKernel)
from volumential_amd.table import NearFieldInteractionTable

pytestmark = pytest.mark.gpu

KERNELS = {"laplace": LaplaceKernel(3), "constant": ConstantKernel(3),
           "helmholtz": HelmholtzKernel(3, 5.0), "dt": AxisTargetDerivative(2, LaplaceKernel(3)),
           "ds": AxisSourceDerivative(0, HelmholtzKernel(3, 5.0)), "log": RadialPowerLogKernel(3, 2)}


def _extended(t, entry_id, regular, radial):
    """Entry of the constant kernel in extended precision."""
    ld = np.longdouble
    case, pair = divmod(int(entry_id), t.n_pairs)
    mode, node = divmod(pair, t.n_q_points)
    x = t.case_target_points()[:, case, node].astype(ld)
    q, H, xi = t.quad_order, ld(t.source_box_extent), t.interp_nodes.astype(ld)
    m = (mode // (q * q), mode // q % q, mode % q)
    rho, w_rho = (a.astype(ld) for a in quadrature.tanh_sinh_fast(radial))
    eta, w_eta = (a.astype(ld) for a in quadrature.gauss_legendre_01(regular))
    v = np.clip(x, ld(0), H)

    def basis(y, i):
        out = np.ones_like(y)
        for j in range(q):
            if j != i:
                out *= (y - xi[j]) / (xi[i] - xi[j])
        return out

    u = (rho[:, None, None], rho[:, None, None] * eta[None, :, None],
         rho[:, None, None] * eta[None, :, None] * eta)
    jac = (rho**2 * w_rho)[:, None, None] * (eta * w_eta)[None, :, None] * w_eta
    total = ld(0)
    for sign in itertools.product((-1, 1), repeat=3):
        ln = np.array([v[a] if sign[a] < 0 else H - v[a] for a in range(3)])
        if np.any(ln <= 0):
            continue
        for axes in itertools.permutations(range(3)):
            g = jac
            for i, a in enumerate(axes):
                g = g * basis(v[a] + sign[a] * ln[a] * u[i], m[a])
            total += g.sum() * ln.prod()
    return float(total)


@pytest.mark.parametrize("q,kernel,regular,radial", [
    (1, "laplace", 5, 5), (2, "laplace", 1, 6), (2, "helmholtz", 70, 3), (3, "constant", 256, 3),
    (4, "ds", 7, 5), (5, "dt", 17, 6), (6, "helmholtz", 6, 4), (7, "log", 5, 4),
    (8, "laplace", 4, 4), (11, "laplace", 3, 3), (16, "ds", 2, 3)])
def test_tensor_build_matches_per_entry(cuda, q, kernel, regular, radial):
    print(f"case: tensor build q={q} {kernel} rule {regular}/{radial}", flush=True)
    t = NearFieldInteractionTable(q, 3, KERNELS[kernel], source_box_extent=0.75)
    ids = t.representative_entry_ids()
    # whole target points, those with the most entries first
    key = ids // t.n_pairs * t.n_q_points + ids % t.n_q_points
    points, count = np.unique(key, return_counts=True)
    some = points[np.argsort(-count, kind="stable")]
    some = np.concatenate([some[:3], np.random.default_rng(q).permutation(some)[:40]])
    ids = ids[np.isin(key, some)][:30000]
    if q == 16:
        assert count.max() > 1024
    a = duffy_values(t, ids, regular, radial)
    if kernel == "constant":  # 2e7 nodes
        pick = np.random.default_rng(q).choice(ids.size, 6, replace=False)
        for i in pick:
            ref = _extended(t, ids[i], regular, radial)
            assert abs(a[i] - ref) <= 1e-13 * max(1.0, abs(ref)), (ids[i], a[i], ref)
        return
    b = duffy_values(t, ids, regular, radial, segmented=False)
    assert np.all(np.isfinite(a))
    err = np.max(np.abs(a - b) / np.maximum(1.0, np.abs(b)))
    assert err <= 1e-13, err
