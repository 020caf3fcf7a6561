"""Device driver of the Duffy table build (``vl1_duffy_build``).

Host side of ``_batched_duffy_values_for_local_indices``
(volumential/nearfield_potential_table.py:2328-2463): gathers per-entry
geometry, uploads the node set once, launches one kernel over all entries.
"""

from __future__ import annotations

import ctypes

import numpy as np
import torch

from . import _capi, quadrature


def _dev(a: np.ndarray, dtype=None) -> torch.Tensor:
    t = torch.from_numpy(np.array(a, copy=True, order="C"))
    if dtype is not None:
        t = t.to(dtype)
    return t.to("cuda", non_blocking=False)


def target_point_chunks(table, entry_ids, max_chunk=64):
    """Sort entries by target point (case, target node) and cut each run
    into near-equal chunks of at most ``max_chunk``: ``(order, starts)``
    with ``entry_ids[order]`` the sorted entries and ``starts`` the chunk
    offsets (int64, ``n_chunks + 1``)."""
    entry_ids = np.asarray(entry_ids, dtype=np.int64)
    key = (entry_ids // table.n_pairs) * table.n_q_points + entry_ids % table.n_q_points
    order = np.argsort(key, kind="stable")
    ks = key[order]
    run = np.flatnonzero(np.r_[True, ks[1:] != ks[:-1], True])
    starts = [0]
    for a, b in zip(run[:-1], run[1:]):
        n = int(b - a)
        k = -(-n // max_chunk)
        cuts = a + (np.arange(1, k + 1) * n) // k
        starts.extend(int(c) for c in cuts)
    return order, np.asarray(starts, dtype=np.int64)


# tail nodes of a rule that the build by sum factorization takes (a thread each)
TENSOR_TAIL_NODES = 256


def _tensor_values(L, table, entry_ids, regular_order, radial_order, stream):
    """3D values by sum factorization over the rule's axes
    (``vl1_duffy_build_tensor``): entries grouped by target point, the rule as
    its one-dimensional parts."""
    entry_ids = np.ascontiguousarray(entry_ids, dtype=np.int64)
    n, count = table.n_q_points, entry_ids.size
    order, mode = np.empty(count, dtype=np.int64), np.empty(count, dtype=np.int32)
    start, key = np.empty((2, min(count, table.n_cases * n) + 1), dtype=np.int64)
    n_points = ctypes.c_int64()
    _capi.check(L.vl1_table_groups_host(
        table.n_cases, n, count, entry_ids.ctypes.data, order.ctypes.data, mode.ctypes.data,
        start.ctypes.data, key.ctypes.data, ctypes.byref(n_points)), "vl1_table_groups_host")
    start, key = start[:n_points.value + 1], key[:n_points.value]
    cases, case = np.unique(key // n, return_inverse=True)
    points = table.case_target_points(cases)[:, case, key % n]
    rho, w_rho = quadrature.tanh_sinh_fast(radial_order)
    eta, w_eta = quadrature.gauss_legendre_01(regular_order)
    cplx = bool(table.integral_knl.is_complex_valued)
    vw = 2 if cplx else 1
    # one upload: points, rule and nodes, then starts and modes
    d_f = _dev(np.concatenate([points.ravel(), rho, w_rho, eta, w_eta, table.interp_nodes]))
    d_start, d_mode = _dev(start), _dev(mode)
    at = [8 * int(k) for k in np.cumsum([0, points.size, rho.size, rho.size, eta.size, eta.size])]
    base = d_f.data_ptr()
    work = torch.empty(9 * vw * count, dtype=torch.float64, device="cuda")
    out = work[8 * vw * count:]
    args = _capi.DuffyTensorArgs(
        dim=3, quad_order=table.quad_order, kernel_kind=int(table.integral_knl.kind),
        deriv_axis=int(getattr(table.integral_knl, "axis", -1)),
        power=int(getattr(table.integral_knl.get_base_kernel(), "power", 0)),
        n_radial=rho.size, n_tail=eta.size,
        helmholtz_k=float(getattr(table.integral_knl.get_base_kernel(), "k", 0.0)),
        source_box_extent=table.source_box_extent, n_targets=key.size, n_entries=count,
        max_entries=int(np.diff(start).max()), target_points=base + at[0],
        entry_start=d_start.data_ptr(), modes=d_mode.data_ptr(), radial_x=base + at[1],
        radial_w=base + at[2], tail_x=base + at[3], tail_w=base + at[4],
        interp_nodes=base + at[5], work=work.data_ptr(), result=out.data_ptr())
    st = stream if stream is not None else torch.cuda.current_stream()
    ev0 = torch.cuda.Event(enable_timing=True)
    ev1 = torch.cuda.Event(enable_timing=True)
    ev0.record(st)
    _capi.check(L.vl1_duffy_build_tensor(args, _capi.stream_handle(st)), "vl1_duffy_build_tensor")
    ev1.record(st)
    torch.cuda.synchronize()
    n_nodes = 48 * rho.size * eta.size**2
    table.last_build_kernel_ms = ev0.elapsed_time(ev1)
    table.last_build_node_evals = count * n_nodes
    table.last_build_chunks = int(key.size)
    table.last_build_n_nodes = n_nodes
    got = out.cpu().numpy()
    if cplx:
        got = got[0::2] + 1j * got[1::2]
    res = np.empty_like(got)
    res[order] = got
    return res


def duffy_values(table, entry_ids, regular_order, radial_order, stream=None,
                 segmented=True) -> np.ndarray:
    """Duffy values of ``entry_ids`` (one launch).  ``segmented``: share each
    node's geometry and kernel value among the entries of one target point
    (the fast form; 3D: axis by axis, ``_tensor_values``); ``False`` runs one
    lane per entry."""
    if not torch.cuda.is_available():
        raise RuntimeError("the Duffy table build runs on the GPU; no GPU is visible")
    L = _capi.lib()
    if (segmented and table.dim == 3 and np.size(entry_ids)
            and int(regular_order) <= TENSOR_TAIL_NODES):
        return _tensor_values(L, table, entry_ids, int(regular_order), int(radial_order), stream)
    nodes = quadrature.duffy_node_set(table.dim, int(regular_order), int(radial_order))
    entry_ids = np.asarray(entry_ids, dtype=np.int64)
    order = None
    if segmented and entry_ids.size:
        order, starts = target_point_chunks(table, entry_ids)
        entry_ids = entry_ids[order]
        d_starts = _dev(starts)
    tp, dv, axes = table.duffy_inputs(entry_ids)
    xi = table.interp_nodes
    bw = quadrature.barycentric_weights(xi)
    n_entries = int(tp.shape[1])
    cplx = bool(table.integral_knl.is_complex_valued)
    d_tp, d_dv, d_ax = _dev(tp), _dev(dv), _dev(axes)
    d_u, d_s, d_j = _dev(nodes.node_u), _dev(nodes.node_sign), _dev(nodes.node_jac)
    d_xi, d_bw = _dev(xi), _dev(bw)
    out = torch.empty(n_entries * (2 if cplx else 1), dtype=torch.float64, device="cuda")
    import math

    nodes_per_sign = nodes.n_nodes // (2**table.dim)
    assert nodes_per_sign * 2**table.dim == nodes.n_nodes
    assert nodes_per_sign % math.factorial(table.dim) == 0
    args = _capi.DuffyArgs(
        dim=table.dim,
        quad_order=table.quad_order,
        kernel_kind=int(table.integral_knl.kind),
        helmholtz_k=float(getattr(table.integral_knl.get_base_kernel(), "k", 0.0)),
        n_entries=n_entries,
        n_nodes=nodes.n_nodes,
        nodes_per_sign=nodes_per_sign,
        source_box_extent=table.source_box_extent,
        target_points=d_tp.data_ptr(),
        decomposition=d_dv.data_ptr(),
        mode_axes=d_ax.data_ptr(),
        node_u=d_u.data_ptr(),
        node_sign=d_s.data_ptr(),
        node_jac=d_j.data_ptr(),
        interp_nodes=d_xi.data_ptr(),
        bary_w=d_bw.data_ptr(),
        result=out.data_ptr(),
        deriv_axis=int(getattr(table.integral_knl, "axis", -1)),
        chunk_start=d_starts.data_ptr() if order is not None else None,
        n_chunks=int(starts.size - 1) if order is not None else 0,
        power=int(getattr(table.integral_knl.get_base_kernel(), "power", 0)),
    )
    st = stream if stream is not None else torch.cuda.current_stream()
    ev0 = torch.cuda.Event(enable_timing=True)
    ev1 = torch.cuda.Event(enable_timing=True)
    ev0.record(st)
    _capi.check(L.vl1_duffy_build(args, _capi.stream_handle(st)), "vl1_duffy_build")
    ev1.record(st)
    torch.cuda.synchronize()
    table.last_build_kernel_ms = ev0.elapsed_time(ev1)
    table.last_build_node_evals = int(n_entries) * int(nodes.n_nodes)
    table.last_build_chunks = int(starts.size - 1) if order is not None else int(n_entries)
    table.last_build_n_nodes = int(nodes.n_nodes)
    res = out.cpu().numpy()
    if cplx:
        res = res[0::2] + 1j * res[1::2]
    if order is not None:
        unsorted = np.empty_like(res)
        unsorted[order] = res
        res = unsorted
    return res
