"""List-1 near-field evaluation benchmark (one MI355X).

Workload (default): 3D Laplace, domain [-1,1]^3, uniform octree level 5
(32768 leaves), q = 6 (216 nodes per box, 7,077,888 target points),
R = 64 densities, each a seeded sum of 8 Gaussians (seeds 1000..1063);
canonical FP64 table (140,496 orbit-reduced values) built on the GPU.
A "step" is one evaluation of all 64 densities on all targets.

Forms:
  plain_f64       vl1_near_field_f64: CSR target boxes, one workgroup per
                  target box, lanes over target nodes, FP64 VALU; table
                  values from the expanded per-(level, case) blocks.
  dense_f64_mfma  batched plan, FP64 MFMA (vl1_plan_*, VL1_FORM_F64).
  split           batched plan, Ozaki split slices on MFMA with FP64 sums
                  (the headline form).

Prints one JSON line: metric/value (target points x RHS per second, 1e9),
timing, dtype, the roofline of the dominant kernel (algorithmic flops over
its time from HIP events on the stream the kernel runs on), the error of
every form per RHS against the FP64 oracle on sampled target boxes, and the
CPU baseline (C/OpenMP oracle on bounded samples, R = 1 and 4).
"""

from __future__ import annotations

import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

PEAK_FP64_TFLOPS = 78.6
PEAK_BF16_TFLOPS = 2500.0
PEAK_INT8_TOPS = 5000.0
SPLIT_TOL = 1e-10
PEAK_HBM_GBS = 8000.0


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--level", type=int, default=5)
    ap.add_argument("--q", type=int, default=6)
    ap.add_argument("--rhs", type=int, default=64)
    ap.add_argument("--form", default="auto", choices=["auto", "f64", "split"])
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--cpu-seconds", type=float, default=20.0)
    ap.add_argument("--slices", type=int, default=5,
                    help="BF16 split slices (the int8 form picks its own from its error estimate)")
    ap.add_argument("--i8-slices", type=int, default=0,
                    help="int8 split slices (0 = the fewest, from 5, whose per-RHS estimate "
                         "is <= 1e-10)")
    ap.add_argument("--only-split", action="store_true",
                    help="time only the split form (profiling runs)")
    ap.add_argument("--skip-plain", action="store_true",
                    help="do not time the plain FP64 kernel (profiling runs)")
    ap.add_argument("--no-table-build", action="store_true",
                    help="skip the near-field table build record (3D Laplace q=6, all cases)")
    ap.add_argument("--workload", default="c3", choices=["c3", "c4", "c2", "c1", "c5", "hsplit"],
                    help="c3 (default): 3D Laplace uniform level 5 q=6, 64 RHS; "
                         "c4: 2D Helmholtz k=40, 8 adaptive trees depth 4..10, q=6, 16 complex "
                         "RHS in one plan; c2: 3D Laplace adaptive (interpolation error 1e-8, "
                         "depth 3..7), q=5, 1 RHS; c1: 2D Laplace uniform level 5, q=4, "
                         "exp(-|x|^2/0.01), 1 RHS; c5: 3D Laplace q=6 table build (all "
                         "cases, one launch); hsplit: 2D Helmholtz k=40 with the "
                         "split (Laplace table + remainder), uniform level 7, q=6, 16 RHS")
    ap.add_argument("--no-tune", action="store_true",
                    help="skip the plan autotuner (vl1_plan_tune) before timing")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="only run a 1 GiB device copy (byte-counter calibration)")
    return ap.parse_args()


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def gaussian_densities_gpu(points_dev, seeds):
    """Seeded 8-Gaussian sums evaluated on the device (same recipe as
    volumential_amd.densities.gaussian_mixture)."""
    import torch

    from volumential_amd.densities import gaussian_mixture_params

    dim = points_dev.shape[0]
    out = torch.empty((len(seeds), points_dev.shape[1]), dtype=torch.float64, device="cuda")
    for i, s in enumerate(seeds):
        c, w, a = gaussian_mixture_params(dim, s)
        acc = torch.zeros(points_dev.shape[1], dtype=torch.float64, device="cuda")
        for k in range(c.shape[0]):
            r2 = torch.zeros_like(acc)
            for d in range(dim):
                r2 += (points_dev[d] - float(c[k, d])) ** 2
            acc += float(a[k]) * torch.exp(-r2 / float(w[k]) ** 2)
        out[i] = acc
    return out


class F64Runner:
    """Direct C-ABI driver of vl1_near_field_f64 with device-resident inputs."""

    def __init__(self, tree, table, f_dev, y_dev):
        import torch

        from volumential_amd import _capi, gallery
        from volumential_amd.payload import DevicePayload, prepare_table_data_and_entry_map

        data, nmlz, _, _, _, info = prepare_table_data_and_entry_map([table])
        meta = table.arithmetic_metadata()
        self.payload = DevicePayload(tree.dim, tree.quad_order, data, nmlz, table.case_indices, meta)

        def dev(a, dt):
            return torch.as_tensor(np.ascontiguousarray(a)).to(dt).cuda().contiguous()

        self.keep = dict(
            centers=dev(tree.box_centers, torch.float64),
            levels=dev(tree.box_levels, torch.uint8),
            counts=dev(tree.box_target_counts_nonchild, torch.int32),
            starts=dev(tree.box_target_starts, torch.int32),
            nstarts=dev(tree.neighbor_source_boxes_starts, torch.int32),
            nlists=dev(tree.neighbor_source_boxes_lists, torch.int32),
            tboxes=dev(tree.target_boxes, torch.int32),
            ids=dev(tree.local_ids, torch.int32),
        )
        k = self.keep
        self.f, self.y = f_dev, y_dev
        self.args = _capi.NearFieldArgs(
            scaling_mode=_capi.SCALING_CANONICAL,
            scaling_power=2,
            log_displacement=int(tree.dim == 2),
            root_extent=tree.root_extent,
            table_root_extent=table.source_box_extent,
            table_starting_level=0,
            encoding_shift=float(gallery.ENCODING_SHIFT),
            encoding_base=gallery.ENCODING_BASE,
            case_encoding_bias=1e-10,
            n_tgt_boxes=int(tree.target_boxes.size),
            aligned_nboxes=int(tree.nboxes),
            n_rhs=int(f_dev.shape[0]),
            ld_coefs=int(f_dev.shape[1]),
            ld_result=int(y_dev.shape[1]),
            result=y_dev.data_ptr(),
            mode_coefs=f_dev.data_ptr(),
            box_centers=k["centers"].data_ptr(),
            box_levels=k["levels"].data_ptr(),
            box_source_counts_nonchild=k["counts"].data_ptr(),
            box_source_starts=k["starts"].data_ptr(),
            box_target_counts_nonchild=k["counts"].data_ptr(),
            box_target_starts=k["starts"].data_ptr(),
            neighbor_source_boxes_starts=k["nstarts"].data_ptr(),
            neighbor_source_boxes_lists=k["nlists"].data_ptr(),
            target_boxes=k["tboxes"].data_ptr(),
            source_mode_ids=k["ids"].data_ptr(),
            target_point_ids=k["ids"].data_ptr(),
            error_flags=0,
        )
        self.L = _capi.lib()
        self.capi = _capi

    def __call__(self, stream_handle):
        self.capi.check(self.L.vl1_near_field_f64(self.payload.handle, self.args, stream_handle))


# declared FP64 work of the table build, 3D Laplace q=6, per target point and
# node of its nonempty sign blocks: the node and 1/r (13 flop), the weight (2),
# six basis values by prefix/suffix products into six sums (28), and the outer
# axes' sums per node (5)
FLOP_PER_TARGET_NODE_3D = 48.0


def table_build_record(rules):
    """Near-field table build, 3D Laplace q=6: every canonical entry of all
    139 cases (140,496 entries) in one vl1_duffy_build_tensor per rule
    (GL tail order, tanh-sinh-fast order); kernel time from HIP events."""
    from volumential_amd.kernels import LaplaceKernel
    from volumential_amd.table import DuffyBuildConfig, NearFieldInteractionTable

    out = []
    for reg, rad in rules:
        t = NearFieldInteractionTable(6, 3, LaplaceKernel(3), source_box_extent=2.0)
        t.build_table(DuffyBuildConfig(regular_quad_order=reg, radial_quad_order=rad))
        ms = t.last_build_kernel_ms
        ne = t.last_build_node_evals
        rate = ne / (ms * 1e-3)
        ids = t.reduced_entry_ids
        key = np.unique(ids // t.n_pairs * t.n_q_points + ids % t.n_q_points)
        x = t.case_target_points()[:, key // t.n_q_points, key % t.n_q_points]
        blocks = np.prod((x > 0.0).astype(int) + (x < 2.0), axis=0).sum()  # nonempty
        flops = blocks * t.last_build_n_nodes / 8 * FLOP_PER_TARGET_NODE_3D
        tf = flops / (ms * 1e-3) / 1e12
        out.append({"rule": [reg, rad], "entries": int(t.reduced_entry_ids.size),
                    "target_point_chunks": int(t.last_build_chunks),
                    "kernel_ms": ms, "build_s": t.last_build_seconds,
                    "node_evals": ne, "node_evals_per_s": rate,
                    "fp64_tflops_declared": tf, "fp64_frac": tf / PEAK_FP64_TFLOPS})
        log(f"table build rule {reg}/{rad}: kernel {ms:.2f} ms, {rate:.3e} node-evals/s, "
            f"{tf:.1f} TFLOP/s = {out[-1]['fp64_frac'] * 100:.1f} % of FP64 peak (declared "
            f"{FLOP_PER_TARGET_NODE_3D:.0f} flop per target point and node)")
    return out


def split_rows_per_wave(form_record):
    """Template argument NRT of the split kernel that ran: 1 when the tuned
    (or default) variant has one row tile per wave, else 2."""
    tuned = form_record.get("autotune") or {}
    return 1 if (tuned.get("variant", 0) & 1) else 2


def measured_traffic(kernel, level, q, rhs):
    """HBM-side bytes per launch of `kernel` on the default workload, from the
    committed counter passes (profiles/c3_traffic.json: FETCH_SIZE and
    WRITE_SIZE in KiB per dispatch, scaled by a 1 GiB copy's readings).
    Counters cannot be read from inside this process, so other workloads
    report None."""
    if (level, q, rhs) != (5, 6, 64):
        return None, None
    path = os.path.join(ROOT, "profiles", "c3_traffic.json")
    try:
        with open(path) as fh:
            d = json.load(fh)
        return float(d["kernels"][kernel]["traffic_bytes"]), "profiles/c3_traffic.json"
    except (OSError, KeyError, ValueError):
        return None, None


def measured_counters(kernel, level, q, rhs):
    """MFMA busy fraction and related counters of `kernel` on the default
    workload from the committed counter passes (profiles/c3_traffic.json,
    key "counters"), or None."""
    if (level, q, rhs) != (5, 6, 64):
        return None
    path = os.path.join(ROOT, "profiles", "c3_traffic.json")
    try:
        with open(path) as fh:
            d = json.load(fh)
        return d["kernels"][kernel].get("counters")
    except (OSError, KeyError, ValueError):
        return None


def host_cpu():
    """The host's CPU model (/proc/cpuinfo) and logical CPU count."""
    model = "unknown"
    try:
        with open("/proc/cpuinfo") as fh:
            for line in fh:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    return {"cpu_model": model, "nproc": os.cpu_count()}


def host_threads():
    """Threads for the CPU baseline: OMP_NUM_THREADS when set (the CPU share
    of a GPU host), else every CPU this process may run on."""
    env = os.environ.get("OMP_NUM_THREADS", "")
    if env.isdigit() and int(env) > 0:
        return int(env)
    try:
        return len(os.sched_getaffinity(0))
    except (AttributeError, OSError):
        return os.cpu_count() or 1


def _sub_tree(tree, pos):
    """Shallow copy of `tree` whose target boxes are the entries `pos` of its
    target-box list (with their list-1 sources)."""
    import copy

    sub = copy.copy(tree)
    starts = np.zeros(pos.size + 1, np.int32)
    lists = []
    for i, b in enumerate(pos):
        seg = tree.neighbor_source_boxes_lists[
            tree.neighbor_source_boxes_starts[b] : tree.neighbor_source_boxes_starts[b + 1]
        ]
        lists.append(seg)
        starts[i + 1] = starts[i] + seg.size
    sub.target_boxes = np.asarray(tree.target_boxes, np.int32)[pos]
    sub.neighbor_source_boxes_starts = starts
    sub.neighbor_source_boxes_lists = np.concatenate(lists).astype(np.int32)
    return sub


def _oracle_eval(tree, table, f_rows, sel, cores, own_csr=True):
    """C/OpenMP oracle on the target-box list entries `sel` of `tree` for the densities
    `f_rows` [R, n_pts]; returns (output [R, n_pts], seconds).  With
    `own_csr` the oracle derives the list-1 sources of `sel` from the box
    geometry (not timed apart); the timed baseline samples take the tree's
    lists."""
    from oracle import cpu as ocpu
    from oracle import orbit_ref

    meta = orbit_ref.case_metadata(tree.dim, tree.quad_order)
    sub = _sub_tree(tree, sel)
    t0 = time.perf_counter()
    out = ocpu.near_field(sub, table.compact_values()[None], table.mode_normalizers[None], meta,
                          f_rows, mode="canonical", scaling_power=2,
                          log_displacement=(tree.dim == 2),
                          table_root_extent=table.source_box_extent, nthreads=cores,
                          own_csr=own_csr)
    return out, time.perf_counter() - t0


def cpu_baseline(tree, table, f_host_rows, seconds, rhs_counts=(1,)):
    """C/OpenMP oracle (reference semantics, one evaluation per RHS) on
    bounded samples of interior target boxes, one sample per RHS count in
    `rhs_counts` (each about seconds / len(rhs_counts) of CPU work); returns
    points x RHS / s at the largest RHS count, the rate of every count, and
    (key "_samples", not part of the JSON line) the sampled boxes with the
    oracle's outputs."""
    from oracle import cpu as ocpu

    counts = np.diff(tree.neighbor_source_boxes_starts)
    full = np.flatnonzero(counts == counts.max())
    if full.size < 1024:  # adaptive trees: a seeded sample of all target boxes
        full = np.random.default_rng(0).permutation(counts.size)
    cores = host_threads()
    ocpu.lib()
    rates, samples, notes = {}, [], []
    budget = seconds / len(rhs_counts)
    for R_ in rhs_counts:
        rows = f_host_rows[:R_]

        def pick(nb):
            return np.asarray(full[:: max(1, full.size // nb)][:nb], np.int32)

        sel = pick(max(cores, 8))
        _, t = _oracle_eval(tree, table, rows, sel, cores, own_csr=False)
        per_box = t / sel.size
        sel = pick(int(min(full.size, max(cores, budget / max(per_box, 1e-9)))))
        out, t = _oracle_eval(tree, table, rows, sel, cores, own_csr=False)
        rates[R_] = sel.size * tree.n_q_points * R_ / t / 1e9
        samples.append((np.asarray(tree.target_boxes, np.int32)[sel], out))
        notes.append(f"{sel.size} target boxes x {R_} RHS ({t:.1f} s)")
    top = max(rhs_counts)
    return {
        "value": rates[top],
        "unit": "Gpts*RHS/s",
        "cores": cores,
        "kind": "port",
        "sample": "; ".join(notes) + " of the same tree/table/densities; the oracle "
                  "evaluates each RHS separately, so the rate is linear in the RHS count",
        "value_by_rhs": {str(k): v for k, v in rates.items()},
        **host_cpu(),
        "_samples": samples,
    }


def oracle_check_sample(tree, table, f_host, n_boxes=48, seed=7):
    """The oracle (own list-1 CSR) on a seeded sample of `n_boxes` target
    boxes for every density of `f_host`; returns [(boxes, output)] for
    ``error_vs_oracle``."""
    t0 = time.perf_counter()
    rng = np.random.default_rng(seed)
    nt = tree.target_boxes.size
    pos = np.sort(rng.choice(nt, size=min(n_boxes, nt), replace=False)).astype(np.int32)
    out, _ = _oracle_eval(tree, table, f_host, pos, host_threads())
    log(f"oracle check sample: {pos.size} boxes x {f_host.shape[0]} RHS in "
        f"{time.perf_counter() - t0:.1f} s")
    return [(np.asarray(tree.target_boxes, np.int32)[pos], out)]


def oracle_check_sample_numpy(tree, tables, f_host, mode, n_boxes=16, seed=7, **kw):
    """The numpy oracle (complex data, per-level tables; own list-1 CSR) on
    a seeded sample of `n_boxes` target boxes; returns [(boxes, output)]
    like ``oracle_check_sample``."""
    from oracle import list1_ref, orbit_ref

    t0 = time.perf_counter()
    rng = np.random.default_rng(seed)
    tb_all = np.asarray(tree.target_boxes, np.int32)
    sel = np.sort(rng.choice(tb_all.size, size=min(n_boxes, tb_all.size), replace=False))
    boxes = tb_all[sel]
    st, ls = list1_ref.list1_csr_bruteforce(tree.box_centers, tree.box_levels, tree.root_extent,
                                            boxes, box_group=list1_ref.tree_groups(tree))
    out = list1_ref.near_field(
        dim=tree.dim, q=tree.quad_order, box_centers=tree.box_centers,
        box_levels=tree.box_levels, box_starts=tree.box_target_starts,
        box_counts=tree.box_target_counts_nonchild, target_boxes=boxes, nbr_starts=st,
        nbr_lists=ls, source_mode_ids=tree.local_ids, target_point_ids=tree.local_ids,
        table_data=np.stack([t.compact_values() for t in tables]),
        mode_nmlz=np.stack([t.mode_normalizers for t in tables]),
        meta=orbit_ref.case_metadata(tree.dim, tree.quad_order), mode=mode,
        root_extent=tree.root_extent, table_root_extent=tables[0].source_box_extent,
        mode_coefs=f_host, **kw)
    log(f"oracle check sample (numpy): {boxes.size} boxes x {f_host.shape[0]} RHS in "
        f"{time.perf_counter() - t0:.1f} s")
    return [(boxes, out)]


def sample_points(tree, sel):
    """Tree-order point indices of the target boxes `sel`."""
    return np.concatenate([np.arange(tree.box_target_starts[b],
                                     tree.box_target_starts[b] + tree.box_target_counts_nonchild[b])
                           for b in sel])


def error_vs_oracle(tree, samples, forms_out, full_ref=None):
    """Per-RHS relative error of each GPU form against the oracle on its
    sampled target points: {form: {rel_linf_per_rhs_max, rel_l2_per_rhs_max,
    rhs, points, ...}}.  `samples`: [(boxes, oracle output [R, n_pts])];
    `forms_out`: {form: device tensor [R_all, n_pts]}.

    The metric is relative to each RHS's whole result vector.  With
    `full_ref` (a device tensor [R, n_pts] over all targets, the FP64 form)
    the denominators are its max |y| and ||y||_2 over all targets and the
    sampled squared error is scaled by (all points / sampled points) for the
    L2 figure; the sample-relative figures (denominators over the sampled
    points only) are reported as `sample_relative`."""
    n_all = int(np.sum(np.asarray(tree.box_target_counts_nonchild)[np.asarray(tree.target_boxes)]))
    res = {}
    for name, y in forms_out.items():
        l2, li, sl2, sli, npt, nr = [], [], [], [], 0, 0
        for sel, ref in samples:
            idx = sample_points(tree, sel)
            R_ = ref.shape[0]
            got = y[:R_, idx].cpu().numpy()
            got = got.astype(np.complex128 if np.iscomplexobj(got) else np.float64)
            want = ref[:, idx]
            d = got - want
            sl2.extend(np.linalg.norm(d, axis=1) / np.linalg.norm(want, axis=1))
            sli.extend(np.abs(d).max(axis=1) / np.abs(want).max(axis=1))
            if full_ref is not None:
                fr = full_ref[:R_]
                ymax = fr.abs().amax(dim=1).cpu().numpy()
                ynorm = fr.norm(dim=1).cpu().numpy()
                li.extend(np.abs(d).max(axis=1) / ymax)
                l2.extend(np.sqrt((np.abs(d) ** 2).sum(axis=1) * n_all / idx.size) / ynorm)
            npt += idx.size
            nr = max(nr, R_)
        rec = {"rhs": nr, "points": int(npt)}
        if full_ref is not None:
            rec.update({"rel_linf_per_rhs_max": float(np.max(li)), "rel_l2_per_rhs_max": float(np.max(l2)),
                        "denominators": "max |y| and ||y||_2 of each RHS over all targets (FP64 form); "
                                        "L2 numerator from the sample scaled to all targets",
                        "sample_relative": {"rel_linf_per_rhs_max": float(np.max(sli)),
                                            "rel_l2_per_rhs_max": float(np.max(sl2))}})
        else:
            rec.update({"rel_linf_per_rhs_max": float(np.max(sli)), "rel_l2_per_rhs_max": float(np.max(sl2)),
                        "denominators": "the sampled points"})
        res[name] = rec
    return res


def _build_beam_tree(seed):
    from volumential_amd import densities
    from volumential_amd import tree as vtree

    f = (lambda P: densities.helmholtz_beams(P, seed, k=40.0))
    return vtree.adaptive_tree_batched(2, 6, vtree.interpolation_refiner(f, 2, 6, 1e-10, 4.0),
                                       min_level=4, max_level=10)


def _plan_forms(plan, f, R, n_pts, flops, steps, warmup, slices, complex_data):
    """Time stage + contract of the FP64 and split plan forms; per-RHS error
    of the split form against the FP64 form."""
    import torch

    from volumential_amd import _capi
    from volumential_amd.plan import FORMS

    L = _capi.lib()
    stream = torch.cuda.current_stream()
    sh = int(stream.cuda_stream)
    fr = torch.view_as_real(f).reshape(R, -1) if complex_data else f
    ldf = fr.shape[1]  # rows are contiguous (a one-row tensor may report stride 0)
    res = {}
    ys = {}
    for form, S in (("f64", 0), ("split", slices)):
        tuned = plan.tune(f, form=form, n_slices=S, reps=2)
        log(f"autotune {form}: variant {tuned['variant']} {tuned['flags']} times {tuned['times_ms']}")
        y = torch.zeros_like(f)
        yr = torch.view_as_real(y).reshape(R, -1) if complex_data else y
        opts = _capi.SplitOpts(n_slices=S, n_products=0)
        kern = []

        def step():
            _capi.check(L.vl1_plan_stage(plan.handle, FORMS[form], fr.data_ptr(), ldf, R, opts, sh))
            a = torch.cuda.Event(enable_timing=True)
            b = torch.cuda.Event(enable_timing=True)
            a.record(stream)
            _capi.check(L.vl1_plan_contract(plan.handle, FORMS[form], R, yr.data_ptr(), ldf, opts, sh))
            b.record(stream)
            kern.append((a, b))

        for _ in range(warmup):
            step()
        torch.cuda.synchronize()
        kern.clear()
        e0 = torch.cuda.Event(enable_timing=True)
        e1 = torch.cuda.Event(enable_timing=True)
        e0.record(stream)
        for _ in range(steps):
            step()
        e1.record(stream)
        torch.cuda.synchronize()
        ms = e0.elapsed_time(e1) / steps
        kms = sum(a.elapsed_time(b) for a, b in kern) / len(kern)
        res[form] = {"ms": ms, "kernel_ms": kms, "value": n_pts * R / (ms * 1e-3) / 1e9,
                     "tflops": flops / (kms * 1e-3) / 1e12, "autotune": tuned}
        ys[form] = y
        log(f"{form}: {ms:.3f} ms/step (contract {kms:.3f} ms), "
            f"{res[form]['value']:.3f} Gpts*RHS/s, {res[form]['tflops']:.2f} TFLOP/s")
    def vs_f64(y):
        d = y - ys["f64"]
        l2 = (d.abs().pow(2).sum(dim=1).sqrt() / ys["f64"].abs().pow(2).sum(dim=1).sqrt()).cpu().numpy()
        li = (d.abs().amax(dim=1) / ys["f64"].abs().amax(dim=1)).cpu().numpy()
        return l2, li

    l2, li = vs_f64(ys["split"])
    res["split"].update({"slices": slices, "rel_l2_max": float(l2.max()),
                         "rel_linf_max": float(li.max())})
    log(f"split vs f64: rel L2 max {l2.max():.2e}, Linf max {li.max():.2e}")

    # int8 split: slices from the per-RHS error estimate (5, else 6)
    est = torch.zeros((R, 2), dtype=torch.float64, device="cuda")
    y = torch.zeros_like(f)
    yr = torch.view_as_real(y).reshape(R, -1) if complex_data else y
    try:
        S8 = 5
        while True:
            plan.eval(f, out=y, form="split_i8", n_slices=S8, error_est=est)
            torch.cuda.synchronize()
            if float(est.max()) <= SPLIT_TOL or S8 == 6:
                break
            S8 += 1
    except RuntimeError as exc:  # e.g. a tile too long for exact int32 sums
        log(f"int8 split not available here: {exc}")
        return res, ys
    opts = _capi.SplitOpts(n_slices=S8, n_products=0, error_est=est.data_ptr())
    kern = []

    def step8():
        _capi.check(L.vl1_plan_stage(plan.handle, FORMS["split_i8"], fr.data_ptr(), ldf, R, opts, sh))
        a = torch.cuda.Event(enable_timing=True)
        b = torch.cuda.Event(enable_timing=True)
        a.record(stream)
        _capi.check(L.vl1_plan_contract(plan.handle, FORMS["split_i8"], R, yr.data_ptr(), ldf, opts, sh))
        b.record(stream)
        kern.append((a, b))

    for _ in range(warmup):
        step8()
    torch.cuda.synchronize()
    kern.clear()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record(stream)
    for _ in range(steps):
        step8()
    e1.record(stream)
    torch.cuda.synchronize()
    ms = e0.elapsed_time(e1) / steps
    kms = sum(a.elapsed_time(b) for a, b in kern) / len(kern)
    l2, li = vs_f64(y)
    e8 = est.cpu().numpy()
    res["split_i8"] = {"ms": ms, "kernel_ms": kms, "value": n_pts * R / (ms * 1e-3) / 1e9,
                       "tflops": flops / (kms * 1e-3) / 1e12, "slices": S8,
                       "rel_l2_max": float(l2.max()), "rel_linf_max": float(li.max()),
                       "estimate_rel_linf_max": float(e8[:, 0].max()),
                       "estimate_rel_l2_max": float(e8[:, 1].max()),
                       "estimate_covers_error": bool(np.all(e8[:, 0] >= li) and np.all(e8[:, 1] >= l2))}
    ys["split_i8"] = y
    log(f"split_i8 S={S8}: {ms:.3f} ms/step (contract {kms:.3f} ms), vs f64 rel L2 max "
        f"{l2.max():.2e}, Linf max {li.max():.2e}; estimate Linf {e8[:, 0].max():.2e}")
    return res, ys


def on_folded_kernel(rel_l2_vs_f64):
    """A split form at 5 and more slices of a plan with reflection-symmetric
    blocks runs on the FP64 form's kernel: the same result, bit for bit."""
    return float(rel_l2_vs_f64) == 0.0


def folded_roofline(flops, kernel_ms, dim):
    """Roofline of the folded FP64 kernel, which does 1 / 2^dim of the
    products of the sum over sources (`flops`) on FP64 MFMA."""
    done = flops / 2**dim
    achieved = done / (kernel_ms * 1e-3) / 1e12
    return {"bound": "mfma", "achieved": achieved, "peak": PEAK_FP64_TFLOPS, "unit": "TFLOP/s",
            "frac": achieved / PEAK_FP64_TFLOPS, "traffic": None, "kernel": "fold_f64_kernel",
            "kernel_ms": kernel_ms, "flops_per_launch": done,
            "flops_note": f"products done: 1/{2**dim} of 2 R sum_pairs n^2 (reflection folding)",
            "tflops_unfolded_equiv": flops / (kernel_ms * 1e-3) / 1e12}


def _split_line_parts(forms, key, flops, bf16_slices, dim):
    """(dtype, form label, roofline) of split form `key` for a bench line."""
    sp = forms[key]
    if on_folded_kernel(sp["rel_l2_max"]):
        return ("f64", f"{key} S={sp.get('slices', bf16_slices)} (on the folded FP64 kernel)",
                folded_roofline(flops, sp["kernel_ms"], dim))
    if key == "split_i8":
        S, peak = sp["slices"], PEAK_INT8_TOPS
        kname = f"split_i8_kernel<{S}>"
        dtype = "int8 digits (MFMA, exact int32 sums) + f64 recombination"
    else:
        S, peak = bf16_slices, PEAK_BF16_TFLOPS
        kname = f"split_bf16_kernel<{S}, {split_rows_per_wave(sp)}>"
        dtype = "bf16 slices (MFMA) + f64 sums"
    nprod = S * (S + 1) // 2
    achieved = flops / (sp["kernel_ms"] * 1e-3) / 1e12
    roof = {"bound": "mfma", "achieved": achieved, "peak": peak, "unit": "TFLOP/s",
            "frac": achieved / peak, "traffic": None, "kernel": kname,
            "kernel_ms": sp["kernel_ms"], "flops_per_launch": flops,
            "flops_note": "algorithmic (FP64-equivalent useful work)",
            "mfma_work": {"slice_products": nprod, "ops_per_launch": nprod * flops,
                          "frac": nprod * flops / (sp["kernel_ms"] * 1e-3) / 1e12 / peak}}
    return dtype, f"{key} S={S}", roof


def _headline_split(forms):
    """The fastest split form within 1e-10 of the FP64 form (per RHS, L2
    and Linf); the BF16 form if none is."""
    ok = [k for k in ("split_i8", "split") if k in forms and
          forms[k]["rel_l2_max"] <= SPLIT_TOL and forms[k]["rel_linf_max"] <= SPLIT_TOL]
    return min(ok, key=lambda k: forms[k]["ms"]) if ok else "split"


def _line(metric_value, ms, steps, warmup, dtype, data, config, roofline, forms, extra=None,
          metric="list-1 eval Gpts*RHS/s at <=1e-10 rel err; split-MFMA vs FP64 GPU kernel",
          unit="Gpts*RHS/s"):
    out = {
        "metric": metric,
        "value": metric_value, "unit": unit, "n_gpus": 1, "steps": steps,
        "warmup": warmup, "ms_per_step": ms, "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": dtype, "data": data, "config": config,
        "roofline": roofline, "forms": forms,
    }
    out.update(extra or {})
    return out


def run_c4(args):
    """2D Helmholtz k=40: eight adaptive quadtrees (seeds 0..7, depth 4..10,
    refined until the q=6 interpolant of each tree's beam density is within
    1e-10 x 4), per-level complex tables for levels 4..10 built on the GPU,
    16 complex beam densities (seeds 100..115) on every tree, one plan over
    the forest (one launch per eval)."""
    from concurrent.futures import ProcessPoolExecutor

    t0 = time.perf_counter()
    with ProcessPoolExecutor(max_workers=8) as ex:  # before any GPU call
        trees = list(ex.map(_build_beam_tree, range(8)))
    log(f"8 trees built in {time.perf_counter() - t0:.1f} s")
    import torch

    from volumential_amd import densities, tree as vtree
    from volumential_amd.kernels import HelmholtzKernel
    from volumential_amd.payload import DevicePayload, prepare_table_data_and_entry_map
    from volumential_amd.plan import List1Plan
    from volumential_amd.table import DuffyBuildConfig, NearFieldInteractionTable

    if not torch.cuda.is_available():
        print(json.dumps({"error": "no GPU visible"}))
        sys.exit(2)
    fo = vtree.Forest(trees)
    lv = np.bincount(fo.box_levels)
    log(f"forest: {fo.nboxes} boxes, {fo.n_points} points, {fo.n_list1_pairs} pairs, levels {lv.tolist()}")
    tables = []
    t0 = time.perf_counter()
    for lev in range(4, fo.nlevels):
        t = NearFieldInteractionTable(6, 2, HelmholtzKernel(2, 40.0), source_box_extent=2.0 / 2**lev)
        t.build_table(DuffyBuildConfig(regular_quad_order=20, radial_quad_order=41))
        tables.append(t)
    log(f"{len(tables)} complex tables built on the GPU in {time.perf_counter() - t0:.2f} s")
    data, nmlz, _, _, _, _ = prepare_table_data_and_entry_map(tables)
    t0_ = tables[0]
    payload = DevicePayload(2, 6, data, nmlz, t0_.case_indices, t0_.arithmetic_metadata())
    plan = List1Plan(fo, payload, scaling_mode=2, scaling_power=0, table_root_extent=t0_.source_box_extent,
                     table_starting_level=4)
    R = 16
    f = torch.as_tensor(np.stack([densities.helmholtz_beams(fo.points, 100 + r) for r in range(R)]),
                        device="cuda").contiguous()
    n = 36
    flops = 8.0 * R * fo.n_list1_pairs * n * n
    forms, ys = _plan_forms(plan, f, R, fo.n_points, flops, args.steps, args.warmup, args.slices,
                            True)
    outs = {"dense_f64_mfma": ys["f64"], "split_bf16": ys["split"]}
    if "split_i8" in ys:
        outs["split_i8"] = ys["split_i8"]
    errs = error_vs_oracle(fo, oracle_check_sample_numpy(
        fo, tables, f.cpu().numpy(), "per_level", table_starting_level=4), outs, full_ref=ys["f64"])
    for k_, v_ in errs.items():
        log(f"{k_} vs oracle: rel L2 {v_['rel_l2_per_rhs_max']:.2e}, rel Linf "
            f"{v_['rel_linf_per_rhs_max']:.2e} ({v_['rhs']} RHS, {v_['points']} points)")
    key = _headline_split(forms)
    sp = forms[key]
    dtype, label, roof = _split_line_parts(forms, key, flops, args.slices, 2)
    return _line(
        sp["value"], sp["ms"], args.steps, args.warmup, dtype + ", complex128 I/O",
        "synthetic (seeded Gaussian beams, GPU-built per-level Helmholtz tables)",
        {"workload": "2D Helmholtz k=40, 8 adaptive quadtrees depth 4..10, q=6, 16 complex RHS",
         "boxes": fo.nboxes, "target_points": fo.n_points, "rhs": R, "list1_pairs": fo.n_list1_pairs,
         "levels": lv.tolist(), "form": label, "parallelism": "single GPU"},
        roof,
        forms,
        {"error_vs_fp64": {"rel_l2_per_rhs_max": sp["rel_l2_max"],
                           "rel_linf_per_rhs_max": sp["rel_linf_max"]},
         "error_vs_oracle": errs,
         "speedup_vs_dense_f64_mfma": forms["f64"]["ms"] / sp["ms"]})


def run_c2(args):
    """3D Laplace, adaptive: refine while max|f - I_5 f| > 1e-8 on the 6^3
    check grid (f = the seed-0 8-Gaussian sum), depth 3..7, 2:1 balanced;
    q = 5; one Laplace table (H = 2, canonical scaling); one RHS."""
    from volumential_amd import densities, tree as vtree

    t0 = time.perf_counter()
    fden = (lambda P: densities.gaussian_mixture(P, 0))
    tr = vtree.adaptive_tree_batched(3, 5, vtree.interpolation_refiner(fden, 3, 5, 1e-8),
                                     min_level=3, max_level=7)
    log(f"tree: {tr.nboxes} leaves, {tr.n_points} points, {tr.n_list1_pairs} pairs, "
        f"levels {np.bincount(tr.box_levels).tolist()} ({time.perf_counter() - t0:.1f} s)")
    import torch

    from volumential_amd import _capi
    from volumential_amd.kernels import LaplaceKernel
    from volumential_amd.payload import DevicePayload, prepare_table_data_and_entry_map
    from volumential_amd.plan import List1Plan
    from volumential_amd.table import DuffyBuildConfig, NearFieldInteractionTable

    if not torch.cuda.is_available():
        print(json.dumps({"error": "no GPU visible"}))
        sys.exit(2)
    # list-1 CSR of the same leaves on the GPU (vl1_csr_builder_*) vs the host builder
    t0 = time.perf_counter()
    st_h, ls_h = vtree._list1_csr(3, tr.leaf_levels, tr.leaf_index)
    csr_host_s = time.perf_counter() - t0
    vtree.list1_csr_gpu(3, tr.leaf_levels, tr.leaf_index)  # warm
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    st_g, ls_g = vtree.list1_csr_gpu(3, tr.leaf_levels, tr.leaf_index)
    torch.cuda.synchronize()
    csr_gpu_s = time.perf_counter() - t0
    csr_same = bool(np.array_equal(st_g.cpu().numpy(), st_h) and np.array_equal(ls_g.cpu().numpy(), ls_h))
    log(f"list-1 CSR: host {csr_host_s:.2f} s, GPU {csr_gpu_s * 1e3:.1f} ms, identical {csr_same}")
    table = NearFieldInteractionTable(5, 3, LaplaceKernel(3), source_box_extent=2.0)
    table.build_table(DuffyBuildConfig(regular_quad_order=20, radial_quad_order=20))
    f = torch.as_tensor(densities.gaussian_mixture(tr.points, 0)[None, :], device="cuda").contiguous()
    y = torch.zeros_like(f)
    R = 1
    n = 125
    flops = 2.0 * R * tr.n_list1_pairs * n * n
    stream = torch.cuda.current_stream()
    sh = int(stream.cuda_stream)
    runner = F64Runner(tr, table, f, y)
    for _ in range(args.warmup):
        runner(sh)
    torch.cuda.synchronize()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record(stream)
    for _ in range(args.steps):
        runner(sh)
    e1.record(stream)
    torch.cuda.synchronize()
    ms_plain = e0.elapsed_time(e1) / args.steps
    log(f"plain f64: {ms_plain:.3f} ms/step, {flops / (ms_plain * 1e-3) / 1e12:.2f} TFLOP/s")
    data, nmlz, _, _, _, _ = prepare_table_data_and_entry_map([table])
    payload = DevicePayload(3, 5, data, nmlz, table.case_indices, table.arithmetic_metadata())
    plan = List1Plan(tr, payload, scaling_mode=_capi.SCALING_CANONICAL, scaling_power=2,
                     table_root_extent=2.0)
    forms, ys = _plan_forms(plan, f, R, tr.n_points, flops, args.steps, args.warmup, args.slices,
                            False)
    forms["plain_f64"] = {"ms": ms_plain, "value": tr.n_points * R / (ms_plain * 1e-3) / 1e9,
                          "tflops": flops / (ms_plain * 1e-3) / 1e12}
    key = _headline_split(forms)
    sp = forms[key]
    dtype, label, roof = _split_line_parts(forms, key, flops, args.slices, 3)
    extra = {"error_vs_fp64": {"rel_l2_per_rhs_max": sp["rel_l2_max"],
                               "rel_linf_per_rhs_max": sp["rel_linf_max"]},
             "speedup_vs_plain_f64": ms_plain / sp["ms"],
             "speedup_vs_dense_f64_mfma": forms["f64"]["ms"] / sp["ms"],
             "list1_csr": {"host_s": csr_host_s, "gpu_s": csr_gpu_s, "identical": csr_same}}
    if not args.no_cpu_baseline:
        cb = cpu_baseline(tr, table, f.cpu().numpy(), args.cpu_seconds)
        cb.pop("_samples")
        extra["cpu_baseline"] = cb
    outs = {"plain_f64": y, "dense_f64_mfma": ys["f64"], "split_bf16": ys["split"]}
    if "split_i8" in ys:
        outs["split_i8"] = ys["split_i8"]
    extra["error_vs_oracle"] = error_vs_oracle(
        tr, oracle_check_sample(tr, table, f.cpu().numpy()), outs, full_ref=ys["f64"])
    return _line(
        sp["value"], sp["ms"], args.steps, args.warmup, dtype,
        "synthetic (seed-0 8-Gaussian density, GPU-built Laplace table)",
        {"workload": "3D Laplace adaptive (interp. error 1e-8, depth 3..7), q=5, 1 RHS",
         "boxes": tr.nboxes, "target_points": tr.n_points, "rhs": R,
         "list1_pairs": tr.n_list1_pairs, "form": label, "parallelism": "single GPU"},
        roof, forms, extra)


def run_c1(args):
    """2D Laplace on [-1,1]^2, uniform level 5 (1,024 leaves), q=4 (16,384
    points), f = exp(-|x|^2/0.01), one canonical table with the 2D log term,
    one RHS.  Launch-latency bound (4.5 MFLOP); reported, not rooflined."""
    import torch

    from volumential_amd import _capi, tree as vtree
    from volumential_amd.kernels import LaplaceKernel
    from volumential_amd.payload import DevicePayload, prepare_table_data_and_entry_map
    from volumential_amd.plan import List1Plan
    from volumential_amd.table import DuffyBuildConfig, NearFieldInteractionTable

    if not torch.cuda.is_available():
        print(json.dumps({"error": "no GPU visible"}))
        sys.exit(2)
    tr = vtree.uniform_tree(2, 4, 5)
    table = NearFieldInteractionTable(4, 2, LaplaceKernel(2), source_box_extent=2.0)
    table.build_table(DuffyBuildConfig(regular_quad_order=20, radial_quad_order=41))
    f = torch.as_tensor(np.exp(-np.sum(tr.points**2, axis=0) / 0.01)[None, :], device="cuda").contiguous()
    y = torch.zeros_like(f)
    n = 16
    flops = 2.0 * tr.n_list1_pairs * n * n
    stream = torch.cuda.current_stream()
    sh = int(stream.cuda_stream)
    runner = F64Runner(tr, table, f, y)
    for _ in range(max(args.warmup, 1)):
        runner(sh)
    torch.cuda.synchronize()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    reps = max(args.steps, 20)
    e0.record(stream)
    for _ in range(reps):
        runner(sh)
    e1.record(stream)
    torch.cuda.synchronize()
    ms_plain = e0.elapsed_time(e1) / reps
    log(f"plain f64: {ms_plain * 1e3:.1f} us/eval, {flops / (ms_plain * 1e-3) / 1e9:.1f} GFLOP/s")
    data, nmlz, _, _, _, _ = prepare_table_data_and_entry_map([table])
    payload = DevicePayload(2, 4, data, nmlz, table.case_indices, table.arithmetic_metadata())
    plan = List1Plan(tr, payload, scaling_mode=_capi.SCALING_CANONICAL, scaling_power=2,
                     log_displacement=True, table_root_extent=2.0)
    forms, ys = _plan_forms(plan, f, 1, tr.n_points, flops, reps, max(args.warmup, 1), args.slices,
                            False)
    forms["plain_f64"] = {"ms": ms_plain, "value": tr.n_points / (ms_plain * 1e-3) / 1e9,
                          "gflops": flops / (ms_plain * 1e-3) / 1e9}
    extra = {"speedup_plain_vs_split": forms["split"]["ms"] / ms_plain}
    if not args.no_cpu_baseline:
        cb = cpu_baseline(tr, table, f.cpu().numpy(), min(args.cpu_seconds, 5.0))
        cb.pop("_samples")
        extra["cpu_baseline"] = cb
    extra["error_vs_oracle"] = error_vs_oracle(
        tr, oracle_check_sample(tr, table, f.cpu().numpy()),
        {"plain_f64": y, "dense_f64_mfma": ys["f64"], "split_bf16": ys["split"]}, full_ref=ys["f64"])
    return _line(
        forms["plain_f64"]["value"], ms_plain, reps, args.warmup, "f64",
        "synthetic (exp(-|x|^2/0.01) on the nodes, GPU-built Laplace 2D table)",
        {"workload": "2D Laplace uniform level 5, q=4, 1 RHS (plain FP64)", "boxes": tr.nboxes,
         "target_points": tr.n_points, "rhs": 1, "list1_pairs": tr.n_list1_pairs,
         "form": "plain_f64", "parallelism": "single GPU"},
        {"bound": "latency", "achieved": flops / (ms_plain * 1e-3) / 1e12, "peak": PEAK_FP64_TFLOPS,
         "unit": "TFLOP/s", "frac": flops / (ms_plain * 1e-3) / 1e12 / PEAK_FP64_TFLOPS,
         "traffic": None, "kernel": "near_field_f64_kernel<unsigned short, 1, false>",
         "kernel_ms": ms_plain, "flops_per_launch": flops},
        forms, extra)


def _hsplit_auto(args, tr, knl, lap, fd, args_csr):
    """``helmholtz_split_order="auto"`` on the same tree and densities: the
    order from |k| h and the smooth quadrature order by the reference's rule.
    Whole ``eval_direct_split`` calls (host work included, synchronized),
    the fused plan (one contraction: remainder, term tables and log parts in
    its blocks) against the two-launch route (table plans per term + the
    point-to-point sums); error of each fused form against the two-launch
    result."""
    import torch

    from volumential_amd.wrangler import NearFieldWrangler

    w = NearFieldWrangler(tr, {repr(knl): [lap]}, target_kernels=[knl],
                          helmholtz_split_order="auto")
    t0 = time.perf_counter()
    ref = w.eval_direct_split(*args_csr, fd, fused=False)[0][0]
    torch.cuda.synchronize()
    setup_two = time.perf_counter() - t0

    def timed(fn):
        for _ in range(args.warmup):
            fn()
        torch.cuda.synchronize()
        t1 = time.perf_counter()
        for _ in range(args.steps):
            fn()
        torch.cuda.synchronize()
        return (time.perf_counter() - t1) / args.steps * 1e3

    out = {"split_order": w.helmholtz_split_order,
           "smooth_quad_order": w.helmholtz_split_smooth_quad_order,
           "two_launch_ms": timed(lambda: w.eval_direct_split(*args_csr, fd, fused=False)),
           "two_launch_first_call_s": setup_two}
    for form in ("f64", "split_i8"):
        t0 = time.perf_counter()
        got = w.eval_direct_split(*args_csr, fd, form=form)[0][0]
        torch.cuda.synchronize()
        if form == "f64":
            out["fused_plan_build_s"] = time.perf_counter() - t0
        d = (got - ref).abs().pow(2).sum(dim=1).sqrt() / ref.abs().pow(2).sum(dim=1).sqrt()
        out[f"fused_{form}_ms"] = timed(lambda: w.eval_direct_split(*args_csr, fd, form=form))
        out[f"fused_{form}_rel_l2_vs_two_launch"] = float(d.max())
    out["speedup_fused_split_i8_vs_two_launch"] = out["two_launch_ms"] / out["fused_split_i8_ms"]
    log(f"auto split order {out['split_order']}, smooth order {out['smooth_quad_order']}: "
        f"two launches {out['two_launch_ms']:.3f} ms, fused f64 {out['fused_f64_ms']:.3f} ms "
        f"({out['fused_f64_rel_l2_vs_two_launch']:.2e}), fused int8 "
        f"{out['fused_split_i8_ms']:.3f} ms ({out['fused_split_i8_rel_l2_vs_two_launch']:.2e})")
    return out


def run_hsplit(args):
    """2D Helmholtz k=40 on [-1,1]^2 with the reference's default split:
    uniform level 7 (16,384 leaves), q=6 (589,824 points), 16 complex
    random-phase Gaussian-beam densities, one canonical Laplace table.  A
    step is the full list 1 (Laplace-table part + remainder G_k - G_0) of
    all 16 densities.  Forms: the fused split plan (one contraction, FP64 or
    Ozaki split) and the two-launch route (Laplace plan on Re/Im + the
    point-to-point correction kernel)."""
    import torch

    from oracle import cpu as ocpu
    from oracle import orbit_ref
    from oracle import split_ref as S
    from volumential_amd import densities, tree as vtree
    from volumential_amd.kernels import HelmholtzKernel, LaplaceKernel
    from volumential_amd.table import DuffyBuildConfig, NearFieldInteractionTable
    from volumential_amd.wrangler import NearFieldWrangler

    if not torch.cuda.is_available():
        print(json.dumps({"error": "no GPU visible"}))
        sys.exit(2)
    dim, q, level, k, R = 2, 6, 7, 40.0, 16
    tr = vtree.uniform_tree(dim, q, level)
    knl = HelmholtzKernel(dim, k)
    lap = NearFieldInteractionTable(q, dim, LaplaceKernel(dim), source_box_extent=2.0)
    lap.build_table(DuffyBuildConfig(regular_quad_order=20, radial_quad_order=61))
    w = NearFieldWrangler(tr, {repr(knl): [lap]}, target_kernels=[knl])
    f = np.stack([densities.helmholtz_beams(tr.points, 500 + r, k=k) for r in range(R)])
    fd = torch.as_tensor(f, device="cuda").contiguous()
    args_csr = (tr.target_boxes, tr.neighbor_source_boxes_starts, tr.neighbor_source_boxes_lists)
    n, pairs, n_pts = tr.n_q_points, tr.n_list1_pairs, tr.n_points
    log(f"tree: 2D q={q} level {level}, {tr.nboxes} boxes, {n_pts} points, {pairs} pairs")
    ref = w.eval_direct_split(*args_csr, fd, fused=False)[0][0]
    plan = w.get_plan(knl, *args_csr, fused_split=True)
    flops = 8.0 * R * pairs * n * n  # complex MACs, 8 real flops each
    forms, _ = _plan_forms(plan, fd, R, n_pts, flops, args.steps, args.warmup, args.slices, True)
    # the two-launch route: table part (Laplace plan, Re/Im as 2R real rows) + P2P
    stream = torch.cuda.current_stream()
    corr = w._correction(knl)
    wts = torch.as_tensor(np.asarray(tr.weights), device="cuda")
    st = (fd * wts[None, :]).contiguous()
    times = {"two_launch": [], "p2p": []}
    for it in range(args.warmup + args.steps):
        e0, e1, e2 = (torch.cuda.Event(enable_timing=True) for _ in range(3))
        e0.record(stream)
        w.eval_direct_plan(*args_csr, fd, form="f64")
        e1.record(stream)
        corr(st, *args_csr)
        e2.record(stream)
        torch.cuda.synchronize()
        if it >= args.warmup:
            times["two_launch"].append(e0.elapsed_time(e2))
            times["p2p"].append(e1.elapsed_time(e2))
    two_ms = float(np.mean(times["two_launch"]))
    p2p_ms = float(np.mean(times["p2p"]))
    fused = {}
    for form in ("f64", "split"):
        out = w.eval_direct_split(*args_csr, fd, form=form)[0][0]
        d = (out - ref).abs().pow(2).sum(dim=1).sqrt() / ref.abs().pow(2).sum(dim=1).sqrt()
        fused[form] = float(d.max())
    log(f"fused f64 {forms['f64']['ms']:.3f} ms, fused split {forms['split']['ms']:.3f} ms, "
        f"two launches {two_ms:.3f} ms (P2P kernel {p2p_ms:.3f} ms); "
        f"rel L2 vs two-launch: f64 {fused['f64']:.2e}, split {fused['split']:.2e}")
    auto = _hsplit_auto(args, tr, knl, lap, fd, args_csr)
    # P2P roofline: FP64 VALU, declared 8 N + 24 flop per (target, source)
    # point pair for the Horner series and log, plus 8 per complex MAC
    pt_pairs = pairs * n * n
    p2p_flops = pt_pairs * (8.0 * corr.nmax + 24.0 + 8.0 * R)
    # headline: the fastest fused form within 1e-10 of the fused FP64 form
    key = _headline_split(forms)
    ok = forms[key]["rel_l2_max"] <= SPLIT_TOL and forms[key]["rel_linf_max"] <= SPLIT_TOL
    best = key if ok and forms[key]["ms"] < forms["f64"]["ms"] else "f64"
    extra = {"two_launch_ms": two_ms, "p2p_kernel_ms": p2p_ms,
             "p2p_declared_fp64_tflops": p2p_flops / (p2p_ms * 1e-3) / 1e12,
             "p2p_fp64_frac": p2p_flops / (p2p_ms * 1e-3) / 1e12 / PEAK_FP64_TFLOPS,
             "series_terms": corr.nmax,
             "rel_l2_vs_two_launch": fused,
             "speedup_fused_vs_two_launch": two_ms / forms[best]["ms"],
             "auto_split_order": auto}
    if not args.no_cpu_baseline:
        # oracle on a sample of target boxes: C/OpenMP table part (Re, Im) +
        # numpy remainder sum; scaled to points x RHS per second
        import copy

        meta = orbit_ref.case_metadata(2, q)
        cores = host_threads()
        perm = np.random.default_rng(0).permutation(tr.nboxes)
        f1 = f[:1]

        def run(nb):
            sel = np.sort(perm[:nb]).astype(np.int32)
            starts = np.zeros(nb + 1, np.int32)
            lists = []
            for i, b in enumerate(sel):
                seg = tr.neighbor_source_boxes_lists[tr.neighbor_source_boxes_starts[b]:
                                                     tr.neighbor_source_boxes_starts[b + 1]]
                lists.append(seg)
                starts[i + 1] = starts[i] + seg.size
            lists = np.concatenate(lists).astype(np.int32)
            sub = copy.copy(tr)
            sub.target_boxes, sub.neighbor_source_boxes_starts = sel, starts
            sub.neighbor_source_boxes_lists = lists
            t0 = time.perf_counter()
            ocpu.near_field(sub, lap.compact_values()[None], lap.mode_normalizers[None], meta,
                            np.concatenate([f1.real, f1.imag]), mode="canonical",
                            scaling_power=2, log_displacement=True, table_root_extent=2.0,
                            nthreads=cores, own_csr=False)
            S.correction(tr, f1 * np.asarray(tr.weights)[None], k, corr.nmax,
                         target_boxes=sel, starts=starts, lists=lists)
            return time.perf_counter() - t0

        dt0 = run(128)
        nb = int(min(tr.nboxes, max(128, 128 * args.cpu_seconds / max(dt0, 1e-9))))
        dt = run(nb)
        extra["cpu_baseline"] = {
            "value": nb * n / dt / 1e9, "unit": "Gpts*RHS/s", "cores": cores, "kind": "port",
            "sample": f"{nb} target boxes x 1 RHS: C/OpenMP Laplace-table part (Re, Im) + "
                      f"numpy remainder sum ({dt:.1f} s)", **host_cpu()}
    note = ("a complex block runs as the real 2n x 2n block: 8 n^2 flops per RHS, "
            "the complex-MAC count")
    if best == "f64":
        dtype, label = "f64 (complex, fused)", "fused split plan f64"
        roof = {"bound": "mfma", "achieved": flops / (forms[best]["kernel_ms"] * 1e-3) / 1e12,
                "peak": PEAK_FP64_TFLOPS, "unit": "TFLOP/s",
                "frac": flops / (forms[best]["kernel_ms"] * 1e-3) / 1e12 / PEAK_FP64_TFLOPS,
                "traffic": None, "kernel": "dense_f64_kernel",
                "kernel_ms": forms[best]["kernel_ms"], "flops_per_launch": flops}
    else:
        dtype, label, roof = _split_line_parts(forms, best, flops, args.slices, dim)
        label = "fused split plan " + label
    roof["note"] = note
    return _line(
        forms[best]["value"], forms[best]["ms"], args.steps, args.warmup, dtype,
        "synthetic (16 seeded random-phase Gaussian beams, k=40; GPU-built Laplace 2D table)",
        {"workload": "2D Helmholtz k=40 split list 1, uniform level 7, q=6, 16 complex RHS",
         "boxes": tr.nboxes, "target_points": n_pts, "rhs": R, "list1_pairs": pairs,
         "form": label, "parallelism": "single GPU"},
        roof, forms, extra)


def run_c5(args):
    """Near-field table build, 3D Laplace q=6: all 140,496 canonical entries
    of the 139 list-1 cases in one launch (segmented Duffy kernel), rules
    (GL tail, tanh-sinh-fast) = (20, 20) and (40, 40).  value = node
    evaluations per second at rule (20, 20), counted as the reference counts
    them (entries x nodes)."""
    import torch

    from oracle import duffy_ref as D
    from volumential_amd.kernels import LaplaceKernel
    from volumential_amd.table import NearFieldInteractionTable

    if not torch.cuda.is_available():
        print(json.dumps({"error": "no GPU visible"}))
        sys.exit(2)
    recs = []
    for _ in range(max(1, args.steps)):
        recs.append(table_build_record([(20, 20), (40, 40)]))
    best = [min((r[i] for r in recs), key=lambda x: x["kernel_ms"]) for i in range(2)]
    r20 = best[0]
    extra = {"table_build": best}
    if not args.no_cpu_baseline:
        # the oracle's per-entry Duffy quadrature (numpy, one core) on a seeded
        # sample of canonical entries at the same rule
        t = NearFieldInteractionTable(6, 3, LaplaceKernel(3), source_box_extent=2.0)
        ids = t.representative_entry_ids()
        g = D.TableGeometry(3, 6, H=2.0)
        rng = np.random.default_rng(0)
        n_nodes = r20["node_evals"] / r20["entries"]
        done, t0 = 0, time.perf_counter()
        while time.perf_counter() - t0 < args.cpu_seconds:
            g.entry(int(rng.choice(ids)), D.laplace(3), 20, 20)
            done += 1
        dt = time.perf_counter() - t0
        extra["cpu_baseline"] = {
            "value": done * n_nodes / dt / 1e9, "unit": "Gnode-evals/s", "cores": 1,
            "kind": "port",
            "sample": f"{done} seeded canonical entries of the same table, rule (20, 20), "
                      f"numpy per-entry Duffy quadrature ({dt:.1f} s)", **host_cpu()}
    ms = r20["kernel_ms"]
    return _line(
        r20["node_evals_per_s"] / 1e9, ms, len(recs), 0, "f64",
        "table geometry only (no input data): all canonical entries of the 3D Laplace q=6 table",
        {"workload": "3D Laplace q=6 near-field table build, all 139 cases, rule (20, 20)",
         "entries": r20["entries"], "target_point_chunks": r20["target_point_chunks"],
         "node_evals": r20["node_evals"], "parallelism": "single GPU"},
        {"bound": "fp64 valu", "achieved": r20["fp64_tflops_declared"], "peak": PEAK_FP64_TFLOPS,
         "unit": "TFLOP/s", "frac": r20["fp64_frac"], "traffic": None,
         "kernel": "duffy_tensor_kernel<1, 6>", "kernel_ms": ms,
         "flops_per_launch": r20["fp64_tflops_declared"] * 1e12 * ms * 1e-3},
        {}, extra, metric="near-field table build Gnode-evals/s (3D Laplace q=6, all cases)",
        unit="Gnode-evals/s")


def main():
    args = parse()
    if args.gpus != 1:
        print(json.dumps({"error": "this benchmark runs on one GPU only; --gpus must be 1"}))
        sys.exit(2)
    if args.workload == "c4":
        print(json.dumps(run_c4(args)), flush=True)
        return
    if args.workload == "c2":
        print(json.dumps(run_c2(args)), flush=True)
        return
    if args.workload == "c1":
        print(json.dumps(run_c1(args)), flush=True)
        return
    if args.workload == "c5":
        print(json.dumps(run_c5(args)), flush=True)
        return
    if args.workload == "hsplit":
        print(json.dumps(run_hsplit(args)), flush=True)
        return
    import torch

    from volumential_amd import _capi, tree as vtree
    from volumential_amd.kernels import LaplaceKernel
    from volumential_amd.table import DuffyBuildConfig, NearFieldInteractionTable

    if not torch.cuda.is_available():
        print(json.dumps({"error": "no GPU visible"}))
        sys.exit(2)
    _capi.lib()
    if args.copy_calibration:
        x = torch.ones(2**27, dtype=torch.float64, device="cuda")
        z = torch.empty_like(x)
        torch.cuda.synchronize()
        z.copy_(x)
        torch.cuda.synchronize()
        print(json.dumps({"copy_bytes_read": x.numel() * 8, "copy_bytes_written": z.numel() * 8}))
        return
    dim, q, level, R = 3, args.q, args.level, args.rhs
    log(f"tree: {dim}D q={q} uniform level {level}")
    tr = vtree.uniform_tree(dim, q, level)
    n_pts = tr.n_points
    pairs = tr.n_list1_pairs
    log(f"points {n_pts}, boxes {tr.nboxes}, list-1 pairs {pairs}")
    t0 = time.perf_counter()
    table = NearFieldInteractionTable(q, dim, LaplaceKernel(dim), source_box_extent=2.0)
    table.build_table(DuffyBuildConfig(regular_quad_order=10, radial_quad_order=31))
    log(f"table built on GPU in {time.perf_counter() - t0:.2f} s ({table.reduced_entry_ids.size} values)")

    pts = torch.as_tensor(tr.points).cuda()
    seeds = list(range(1000, 1000 + R))
    f = gaussian_densities_gpu(pts, seeds).contiguous()
    y = torch.zeros_like(f)
    torch.cuda.synchronize()
    stream = torch.cuda.current_stream()
    sh = int(stream.cuda_stream)

    def timed(fn, steps, warmup, inner=None):
        """Average ms per step over `steps` (after `warmup`), events on the
        current stream; `inner` optionally returns (ev_a, ev_b) pairs
        bracketing the dominant kernel inside each step."""
        for _ in range(warmup):
            fn()
        torch.cuda.synchronize()
        e0 = torch.cuda.Event(enable_timing=True)
        e1 = torch.cuda.Event(enable_timing=True)
        pairs = []
        e0.record(stream)
        for _ in range(steps):
            r = fn()
            if r is not None:
                pairs.append(r)
        e1.record(stream)
        torch.cuda.synchronize()
        step_ms = e0.elapsed_time(e1) / steps
        kern_ms = sum(a.elapsed_time(b) for a, b in pairs) / len(pairs) if pairs else None
        return step_ms, kern_ms

    n = tr.n_q_points
    flops = 2.0 * R * pairs * n * n
    bytes_alg = 2.0 * 8 * n_pts * R + table.reduced_entry_ids.size * 8 + 4 * (pairs + tr.nboxes)
    forms = {}

    # plain FP64 kernel (reference semantics, CSR target boxes)
    ms_plain, y_plain = None, None
    if not args.skip_plain:
        runner = F64Runner(tr, table, f, y)
        ms_plain, _ = timed(lambda: runner(sh), args.steps, args.warmup)
        y_plain = y
        forms["plain_f64"] = {"ms": ms_plain, "value": n_pts * R / (ms_plain * 1e-3) / 1e9,
                              "tflops": flops / (ms_plain * 1e-3) / 1e12,
                              "fp64_frac": flops / (ms_plain * 1e-3) / 1e12 / PEAK_FP64_TFLOPS,
                              "hbm_gbs_alg": bytes_alg / (ms_plain * 1e-3) / 1e9}
        if R >= 16:  # the MFMA kernel of the plain route: its counter traffic
            kp = "near_field_mfma_kernel<8, 2>" if n > 128 else None
            tb, src = measured_traffic(kp, level, q, R) if kp else (None, None)
            if tb is not None:
                forms["plain_f64"].update({"kernel": kp, "traffic_bytes": tb,
                                           "hbm_gbs_measured": tb / (ms_plain * 1e-3) / 1e9,
                                           "hbm_frac": tb / (ms_plain * 1e-3) / 1e12 / 8.0,
                                           "traffic_source": src})
        log(f"plain f64: {ms_plain:.2f} ms/step, {forms['plain_f64']['value']:.3f} Gpts*RHS/s, "
            f"{forms['plain_f64']['tflops']:.2f} TFLOP/s")
        del runner

    # batched plan: dense FP64 MFMA and Ozaki split
    from volumential_amd.payload import DevicePayload, prepare_table_data_and_entry_map
    from volumential_amd.plan import FORMS, List1Plan

    data, nmlz, _, _, _, _ = prepare_table_data_and_entry_map([table])
    payload = DevicePayload(dim, q, data, nmlz, table.case_indices, table.arithmetic_metadata())
    t0 = time.perf_counter()
    plan = List1Plan(tr, payload, scaling_mode=_capi.SCALING_CANONICAL, scaling_power=2,
                     log_displacement=False, table_root_extent=table.source_box_extent)
    log(f"plan built in {time.perf_counter() - t0:.2f} s")
    L = _capi.lib()

    def plan_step(form, slices, y_out, est=None):
        opts = _capi.SplitOpts(n_slices=slices, n_products=0)
        if est is not None:
            opts.error_est = est.data_ptr()
        fm = FORMS[form]
        _capi.check(L.vl1_plan_stage(plan.handle, fm, f.data_ptr(), f.stride(0), R, opts, sh))
        a = torch.cuda.Event(enable_timing=True)
        b = torch.cuda.Event(enable_timing=True)
        a.record(stream)
        _capi.check(L.vl1_plan_contract(plan.handle, fm, R, y_out.data_ptr(), y_out.stride(0), opts, sh))
        b.record(stream)
        return a, b

    tuned = {}
    if not args.no_tune:
        for form, S_ in (("f64", 0), ("split", args.slices)):
            tuned[form] = plan.tune(f, form=form, n_slices=S_, reps=2)
            log(f"autotune {form}: variant {tuned[form]['variant']} {tuned[form]['flags']} "
                f"times {tuned[form]['times_ms']}")
    y64 = torch.zeros_like(f)
    if args.only_split:
        args.steps, args.warmup = max(1, args.steps), 0
    if not args.only_split:
        ms64, k64 = timed(lambda: plan_step("f64", 0, y64), args.steps, args.warmup)
    else:
        ms64, k64 = timed(lambda: plan_step("f64", 0, y64), 1, 0)
    forms["dense_f64_mfma"] = {"ms": ms64, "kernel_ms": k64, "value": n_pts * R / (ms64 * 1e-3) / 1e9,
                               "tflops": flops / (k64 * 1e-3) / 1e12,
                               "fp64_frac": flops / (k64 * 1e-3) / 1e12 / PEAK_FP64_TFLOPS}
    log(f"dense f64: {ms64:.2f} ms/step (contract {k64:.2f} ms, "
        f"{forms['dense_f64_mfma']['tflops']:.2f} TFLOP/s)")
    if y_plain is not None:
        d_plain = (y64 - y_plain).norm(dim=1) / y64.norm(dim=1)
        forms["plain_f64"]["rel_l2_vs_dense_f64"] = float(d_plain.max())
        log(f"plain vs dense f64 max rel L2 {float(d_plain.max()):.2e}")

    def vs_dense(y):
        l2 = ((y - y64).norm(dim=1) / y64.norm(dim=1)).cpu().numpy()
        li = ((y - y64).abs().amax(dim=1) / y64.abs().amax(dim=1)).cpu().numpy()
        return l2, li

    # BF16 split (the previous form), for comparison
    S = args.slices
    ysp = torch.zeros_like(f)
    if not args.only_split:
        mss, ks = timed(lambda: plan_step("split", S, ysp), args.steps, args.warmup)
        err_l2, err_inf = vs_dense(ysp)
        forms["split_bf16"] = {"ms": mss, "kernel_ms": ks, "value": n_pts * R / (mss * 1e-3) / 1e9,
                               "slices": S, "slice_products": S * (S + 1) // 2,
                               "tflops_fp64_equiv": flops / (ks * 1e-3) / 1e12,
                               "rel_l2_vs_dense_f64_max": float(err_l2.max()),
                               "rel_linf_vs_dense_f64_max": float(err_inf.max()),
                               "autotune": tuned.get("split")}
        log(f"bf16 split S={S}: {mss:.2f} ms/step (contract {ks:.2f} ms), vs dense f64: rel L2 "
            f"max {err_l2.max():.2e}, Linf max {err_inf.max():.2e}")

    # int8 split, the headline form: the slice count is the fewest (from 5)
    # whose per-RHS error estimate is within 1e-10 (the estimate comes with
    # every evaluation and is part of the timed step)
    yi8 = torch.zeros_like(f)
    est = torch.zeros((R, 2), dtype=torch.float64, device="cuda")
    if args.i8_slices:
        S8 = args.i8_slices
    else:
        S8 = 5
        while True:
            plan_step("split_i8", S8, yi8, est)
            torch.cuda.synchronize()
            if float(est.max()) <= SPLIT_TOL or S8 == 6:
                break
            S8 += 1
    msi, ki = timed(lambda: plan_step("split_i8", S8, yi8, est), args.steps, args.warmup)
    e8 = est.cpu().numpy()
    i8_l2, i8_li = vs_dense(yi8)
    nprod = S8 * (S8 + 1) // 2
    forms["split_i8"] = {"ms": msi, "kernel_ms": ki, "value": n_pts * R / (msi * 1e-3) / 1e9,
                         "slices": S8, "slice_products": nprod,
                         "tflops_fp64_equiv": flops / (ki * 1e-3) / 1e12,
                         "rel_l2_vs_dense_f64_max": float(i8_l2.max()),
                         "rel_linf_vs_dense_f64_max": float(i8_li.max()),
                         "estimate_rel_linf_max": float(e8[:, 0].max()),
                         "estimate_rel_l2_max": float(e8[:, 1].max()),
                         "estimate_covers_error": bool(np.all(e8[:, 0] >= i8_li) and
                                                       np.all(e8[:, 1] >= i8_l2))}
    log(f"int8 split S={S8}: {msi:.2f} ms/step (contract {ki:.2f} ms), vs dense f64: rel L2 max "
        f"{i8_l2.max():.2e}, Linf max {i8_li.max():.2e}; estimate max Linf {e8[:, 0].max():.2e} "
        f"L2 {e8[:, 1].max():.2e}")
    value = forms["split_i8"]["value"]
    ms = msi
    kname = f"split_i8_kernel<{S8}>"
    traffic, traffic_note = measured_traffic(kname, level, q, R)
    counters = measured_counters(kname, level, q, R)
    # roofline of the dominant kernel from the algorithmic work (flops_alg =
    # 2 R sum_pairs n^2) over its measured time, against the peak of the
    # unit it runs on (int8 MFMA); the digit products the split scheme
    # executes on that unit are reported beside it as mfma_work
    achieved = flops / (ki * 1e-3) / 1e12
    mfma_ops = nprod * flops

    roofline = {
        "bound": "mfma",
        "achieved": achieved,
        "peak": PEAK_INT8_TOPS,
        "unit": "TFLOP/s",
        "frac": achieved / PEAK_INT8_TOPS,
        "traffic": traffic,
        "traffic_source": traffic_note,
        "kernel": kname,
        "kernel_ms": ki,
        "flops_per_launch": flops,
        "flops_note": "algorithmic: 2 R sum_pairs n^2 (FP64-equivalent useful work)",
        "hbm_gbs_alg": bytes_alg / (ki * 1e-3) / 1e9,
        "mfma_work": {"slice_products": nprod, "ops_per_launch": mfma_ops,
                      "achieved": mfma_ops / (ki * 1e-3) / 1e12,
                      "frac": mfma_ops / (ki * 1e-3) / 1e12 / PEAK_INT8_TOPS,
                      "unit": "int8 TOP/s"},
        **({"counters": counters} if counters else {}),
    }
    dtype = "int8 digits (MFMA, exact int32 sums) + f64 recombination"
    form = f"split_i8 S={S8} (slices chosen by the per-RHS error estimate <= 1e-10)"
    if on_folded_kernel(i8_l2.max()):
        dtype, form = "f64", f"split_i8 S={S8} (on the folded FP64 kernel)"
        roofline = folded_roofline(flops, ki, 3)

    # error per RHS against the FP64 oracle (C/OpenMP restatement of the
    # reference kernel, its own list-1 CSR) on a seeded sample of target
    # boxes, all R densities
    f_host = f.cpu().numpy()
    samples = oracle_check_sample(tr, table, f_host)
    cb = None
    if not args.no_cpu_baseline:
        log("cpu baseline ...")
        cb = cpu_baseline(tr, table, f_host[:4], args.cpu_seconds, rhs_counts=(1, 4))
        cb.pop("_samples")  # timing samples (tree's own lists): not used as the check
        log(f"cpu: {cb}")
    outs = {"dense_f64_mfma": y64, "split_i8": yi8}
    if not args.only_split:
        outs["split_bf16"] = ysp
    if y_plain is not None:
        outs["plain_f64"] = y_plain
    errs = error_vs_oracle(tr, samples, outs, full_ref=y64)
    for k_, v_ in errs.items():
        log(f"{k_} vs oracle: rel L2 {v_['rel_l2_per_rhs_max']:.2e}, rel Linf "
            f"{v_['rel_linf_per_rhs_max']:.2e} ({v_['rhs']} RHS, {v_['points']} points)")

    res = {
        "metric": "list-1 eval Gpts*RHS/s at <=1e-10 rel err; split-MFMA vs FP64 GPU kernel",
        "value": value,
        "unit": "Gpts*RHS/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": dtype,
        "data": "synthetic (seeded 8-Gaussian densities, GPU-built Laplace table)",
        "config": {
            "workload": f"3D Laplace uniform level {level}, q={q}, {R} RHS",
            "boxes": int(tr.nboxes),
            "target_points": int(n_pts),
            "rhs": R,
            "list1_pairs": int(pairs),
            "form": form,
            "parallelism": "single GPU",
        },
        "roofline": roofline,
        "error_vs_oracle": errs,
        "error_vs_fp64": {"rel_l2_per_rhs_max": float(i8_l2.max()),
                          "rel_linf_per_rhs_max": float(i8_li.max()), "rhs": R,
                          "points": int(n_pts), "against": "dense FP64 MFMA form, all points"},
        "error_estimate": {"rel_linf_per_rhs_max": float(e8[:, 0].max()),
                           "rel_l2_per_rhs_max": float(e8[:, 1].max()),
                           "covers_error_vs_fp64": forms["split_i8"]["estimate_covers_error"]},
        "speedup_vs_plain_f64": (ms_plain / msi) if ms_plain else None,
        "speedup_vs_dense_f64_mfma": ms64 / msi,
        "speedup_vs_split_bf16": (forms["split_bf16"]["ms"] / msi) if "split_bf16" in forms else None,
        "autotune": tuned,
        "forms": forms,
    }
    if not args.no_table_build:
        res["table_build"] = table_build_record([(20, 20), (40, 40)])
    if cb is not None:
        res["cpu_baseline"] = cb
    print(json.dumps(res), flush=True)


if __name__ == "__main__":
    main()
