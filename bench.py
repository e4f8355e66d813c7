#!/usr/bin/env python3
"""Benchmark of the UNG cross-edge + mid-group kNN build stage on one MI355X.

Workload "cfg2" (the headline configuration): 1M x 128 fp32 vectors from a
1000-centroid Gaussian mixture, 40 labels (1-4 per vector, Zipf 1.2), k=6 cross
edges per vector and exact K=32 intra-group kNN for every mid-size group
(128 <= n <= 4096).  Synthetic, seeded data (no network).

A step = the whole device job with the base set already resident in HBM:
host work-list packing + descriptor upload + MFMA select + merge + exact
fallback for the cross edges, the additional edges of the groups whose
out-groups no cross edge reaches (edge lists returned to the host, as the
reference's materialized lists), and the intra-group kNN -- by default started on
the library's second stream with the cross edges (ung_hip_cross_intra_begin) and
collected after the additional edges (ung_hip_intra_end); --sequential runs the three
one after the other.  Cross and intra results stay in HBM.  value = (P_cross +
P_intra) / step time (distance evaluations/s, algorithmic pairs only).

After the timed steps (not part of `value`):
  * the drop-in calls with host output (ung_hip_cross_topk: FlatId rows, distances and
    sizes copied to host memory; ung_hip_group_knn likewise) are timed, D2H included;
  * the CPU baseline: the reference's own compiled distance + SearchQueue scan
    (oracle/_ref) on a bounded random sample of cross-edge rows and of mid groups;
  * parity of the same run: the GPU rows of those samples against the reference's rows.

Prints ONE JSON line.
"""
from __future__ import annotations

import argparse
import ctypes as C
import hashlib
import json
import math
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

MFMA_16BIT_PEAK_TFLOPS = 2500.0  # dense
MFMA_FP32_PEAK_TFLOPS = 157.3
HBM_PEAK_GBS = 8000.0
METRIC = "cross-edge build wall time + distance evals/s (MFMA util %), 1M×128 fp32, 1 GPU"
TIE_BAND = 1e-5  # relative distance gap of BASELINE.json's tie band


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def _sha256_files(paths, extra=b""):
    h = hashlib.sha256()
    for p in paths:
        with open(p, "rb") as f:
            h.update(f.read())
    h.update(extra)
    return h.hexdigest()


def kernel_source_digest():
    """Digest of what the select launches are built and planned from: ung_kernels.hip
    (every kernel), ung_runtime.hip (the work-list planning -- split sizes, item order,
    partial-row length -- and the launch choices, which change the kernels' traffic) and
    the HIP compile flags.  A traffic measurement holds while this is unchanged."""
    from filtervectorcode_refactor_amd import build as B
    return _sha256_files([os.path.join(B.CSRC, "ung_kernels.hip"), os.path.join(B.CSRC, "ung_runtime.hip")],
                         " ".join(B.HIP_FLAGS).encode())


def read_traffic(config_name):
    """HBM bytes per launch of the cross select kernel on this workload, measured offline
    with rocprofv3 --pmc (FETCH_SIZE, WRITE_SIZE), calibrated on a copy kernel, from
    profiles/traffic_select_cross_<config>.txt.  Returns (bytes or None, status): a file
    whose kernel_source_sha256 differs from the current source is stale and not used."""
    path = os.path.join(ROOT, "profiles", f"traffic_select_cross_{config_name}.txt")
    if not os.path.exists(path):
        return None, "not measured"
    fields = {}
    with open(path) as f:
        for line in f:
            if ":" in line and line.split(":", 1)[0] in ("traffic_bytes_per_launch", "kernel_source_sha256"):
                key, val = line.split(":", 1)
                fields[key] = val.strip()
    if fields.get("kernel_source_sha256") != kernel_source_digest():
        return None, f"stale ({os.path.basename(path)} was measured on another kernel source)"
    try:
        return float(fields["traffic_bytes_per_launch"]), f"measured ({os.path.basename(path)})"
    except (KeyError, ValueError):
        return None, "unreadable"


def calib_copy(nbytes):
    """One device-to-device hipMemcpy of nbytes (the runtime's blit kernel): the
    reference reading for FETCH_SIZE / WRITE_SIZE in a rocprofv3 --pmc pass."""
    hip = C.CDLL("libamdhip64.so")
    src, dst = C.c_void_p(), C.c_void_p()
    for p in (src, dst):
        if hip.hipMalloc(C.byref(p), C.c_size_t(nbytes)) != 0:
            raise RuntimeError("hipMalloc failed in calib_copy")
    try:
        if hip.hipMemcpy(dst, src, C.c_size_t(nbytes), 3) != 0 or hip.hipDeviceSynchronize() != 0:
            raise RuntimeError("hipMemcpy failed in calib_copy")
    finally:
        hip.hipFree(src)
        hip.hipFree(dst)
    log(f"calibration copy {nbytes} bytes done")


def cpu_model():
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_inventory():
    """What the host offers the CPU baseline: logical CPUs of the machine, the ones this
    process may run on (sched_getaffinity, what `nproc` prints), the OpenMP thread count
    the environment sets, and the CPU model line."""
    try:
        affinity = len(os.sched_getaffinity(0))
    except (AttributeError, OSError):
        affinity = None
    omp = os.environ.get("OMP_NUM_THREADS")
    return {"cpu_model": cpu_model(), "logical_cpus": os.cpu_count(), "nproc": affinity,
            "omp_num_threads_env": int(omp) if omp and omp.isdigit() else None}


def baseline_threads():
    """Threads of the CPU baseline: OMP_NUM_THREADS when the environment sets it (the GPU
    box sets the job's CPU share there), else every CPU this process may run on."""
    inv = cpu_inventory()
    return inv["omp_num_threads_env"] or inv["nproc"] or inv["logical_cpus"] or 1


def _rows_parity(g_ids, g_dist, r_ids, r_dist):
    """(rows, id-exact rows, distance-bit-exact rows) of GPU rows against reference rows."""
    ids_ok = (g_ids == r_ids).all(axis=1)
    dist_ok = (g_dist.view(np.uint32) == r_dist.view(np.uint32)).all(axis=1)
    return int(g_ids.shape[0]), int(ids_ok.sum()), int(dist_ok.sum())


def _tie_pairs(dist):
    """Adjacent entries of sorted rows whose fp32 distances differ by at most TIE_BAND
    relative (ties included); +inf padding ignored."""
    d0, d1 = dist[:, :-1].astype(np.float64), dist[:, 1:].astype(np.float64)
    ok = np.isfinite(d1)
    with np.errstate(invalid="ignore"):
        return int(((d1 - d0 <= TIE_BAND * d1) & ok).sum())


def cpu_leg_and_parity(st, cfg, gpu_cross, gpu_intra, p_cross, p_intra, seconds, timed=True):
    """The reference's compiled scan (oracle/_ref; else the plain-C oracle) on a bounded
    random sample of the workload -- cross-edge rows for about 2/3 of `seconds`, whole mid
    groups for the rest -- timed on all host threads, and the GPU rows of the same
    samples compared with its rows.  Returns (cpu_baseline or None, parity)."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    from oracle import Oracle, RefOracle, ref_available
    threads = baseline_threads()
    kind = "reference" if ref_available() else "port"
    ref = RefOracle() if kind == "reference" else Oracle()
    k, K = cfg.k_cross, cfg.k_intra
    sizes = np.diff(st.group_begin.astype(np.int64))[1:]
    cnt = np.diff(st.out_ptr.astype(np.int64))[1:]
    union = np.zeros(st.num_groups + 1, np.int64)
    np.add.at(union, np.repeat(np.arange(1, st.num_groups + 1), cnt), sizes[st.out_idx.astype(np.int64) - 1])
    pg = st.new_vec_id_to_group_id
    eligible = np.nonzero(union[pg] > 0)[0].astype(np.uint32)
    rng = np.random.default_rng(7)
    rng.shuffle(eligible)

    # cross leg: a calibration run, then one run sized to the budget; the reference scan
    # keeps k+1 entries so the k-th / (k+1)-th boundary can be checked for the tie band
    def cross_run(q):
        t0 = time.perf_counter()
        ri, rd = ref.cross_exact_points(st.base, st.group_begin, pg, st.out_ptr, st.out_idx, q, k + 1, threads)[:2]
        return ri, rd, time.perf_counter() - t0

    budget_x = seconds * 2 / 3 if timed else 0.0
    q1 = eligible[: min(eligible.size, 256 if timed else 3000)]
    ri, rd, dt1 = cross_run(q1)
    qs, ris, rds = [q1], [ri], [rd]
    pairs_x, dt_x = int(union[pg[q1]].sum()), dt1
    if timed and q1.size < eligible.size and dt1 < budget_x:
        rate = pairs_x / max(dt1, 1e-3)
        cum = np.cumsum(union[pg[eligible[q1.size:]]])
        n2 = int(np.searchsorted(cum, rate * (budget_x - dt1))) + 1
        q2 = eligible[q1.size: q1.size + n2]
        ri, rd, dt2 = cross_run(q2)
        qs.append(q2)
        ris.append(ri)
        rds.append(rd)
        pairs_x += int(union[pg[q2]].sum())
        dt_x += dt2
    q = np.concatenate(qs)
    r_ids, r_dist = np.concatenate(ris), np.concatenate(rds)
    g_ids, g_dist = gpu_cross
    n_x, ok_x, okd_x = _rows_parity(g_ids[q], g_dist[q], r_ids[:, :k], r_dist[:, :k])
    tie_x = _tie_pairs(r_dist)
    d_k, d_k1 = r_dist[:, k - 1].astype(np.float64), r_dist[:, k].astype(np.float64)
    with np.errstate(invalid="ignore"):
        boundary_x = int((np.isfinite(d_k1) & (d_k1 - d_k <= TIE_BAND * d_k1)).sum())

    # intra leg: whole mid groups in random order until the rest of the budget is spent
    gi_ids, gi_dist, gids, begins, gsz = gpu_intra
    starts = np.cumsum(gsz.astype(np.int64)) - gsz.astype(np.int64)
    order = rng.permutation(len(gids)) if len(gids) else np.zeros(0, np.int64)
    budget_i = seconds - dt_x if timed else 0.0
    pairs_i, dt_i, n_i, ok_i, okd_i, tie_i, groups_i = 0, 0.0, 0, 0, 0, 0, 0
    for j in order:
        b, n, r0 = int(begins[j]), int(gsz[j]), int(starts[j])
        t0 = time.perf_counter()
        oi, od = ref.intra_exact(st.base, b, n, K, threads)
        dt_i += time.perf_counter() - t0
        pairs_i += n * (n - 1)
        a, b2, c = _rows_parity(gi_ids[r0: r0 + n], gi_dist[r0: r0 + n], oi, od)
        n_i, ok_i, okd_i = n_i + a, ok_i + b2, okd_i + c
        tie_i += _tie_pairs(od)
        groups_i += 1
        if dt_i >= budget_i and groups_i >= (1 if timed else 5):
            break

    parity = {
        "cross_rows_checked": n_x, "cross_id_exact_rate": ok_x / max(n_x, 1),
        "cross_dist_bitexact_rate": okd_x / max(n_x, 1),
        "intra_rows_checked": n_i, "intra_groups_checked": groups_i, "intra_id_exact_rate": ok_i / max(n_i, 1),
        "intra_dist_bitexact_rate": okd_i / max(n_i, 1),
        "tie_band_pairs": tie_x + tie_i,
        "tie_band_kth_boundary_rows": boundary_x,
        "tie_band": f"adjacent entries of the reference's sorted rows (cross: top-{k + 1}, intra: top-{K}) within "
                    f"{TIE_BAND:g} relative; kth_boundary = cross rows whose {k}-th and {k + 1}-th differ by at most that",
        "checker": ("oracle/_ref (the reference's compiled distance.cpp + search_queue.cpp scan)" if kind == "reference"
                    else "the plain-C oracle's exact scan"),
    }
    if not timed:
        return None, parity
    r_x = pairs_x / dt_x
    r_i = pairs_i / dt_i if dt_i > 0 else None
    if r_i and p_intra:
        value = (p_cross + p_intra) / (p_cross / r_x + p_intra / r_i)  # the workload's mix
    else:
        value = r_x
    base = {
        "value": value, "unit": "distance evals/s", "cores": threads, "kind": kind, **cpu_inventory(),
        "threads_used": threads,
        "threads_rule": "OMP_NUM_THREADS when set (the GPU box's CPU share of the job), else nproc",
        "cross_evals_per_s": r_x, "intra_evals_per_s": r_i,
        "sample": f"{q.size} random cross-edge rows of {cfg.name} (exact scan of each row's minimum-superset union, "
                  f"{pairs_x} pairs, {dt_x:.1f} s) and {groups_i} random mid groups ({pairs_i} pairs, {dt_i:.1f} s), "
                  f"{threads} OpenMP threads; value = the workload's P_cross + P_intra over the time those two rates "
                  f"give for it",
    }
    return base, parity


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=0, help="timed steps (default: enough for about 2.5 s)")
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--config", default="cfg2")
    ap.add_argument("--n", type=int, default=0, help="override point count (smaller runs)")
    ap.add_argument("--no-cpu-baseline", action="store_true",
                    help="skip the timed CPU baseline (parity is still checked on a small sample)")
    ap.add_argument("--sequential", action="store_true",
                    help="cross edges, additional edges and the mid groups' kNN one after the other "
                         "(default: the kNN overlapped on the second stream)")
    ap.add_argument("--cpu-seconds", type=float, default=15.0)
    ap.add_argument("--calib-copy", action="store_true",
                    help="end with a 1 GiB device-to-device copy (counter calibration for --pmc runs)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(json.dumps({"error": "this build runs on exactly one GPU (one-GPU boxes); "
                                   "multi-GPU sharding is not built", "n_gpus": args.gpus}))
        sys.exit(2)

    import filtervectorcode_refactor_amd as F
    from filtervectorcode_refactor_amd import datasets as D

    cfg = D.CONFIGS[args.config]
    if args.n:
        cfg = D.scaled(cfg, args.n)
    t0 = time.perf_counter()
    X, lp, li = D.generate(cfg)
    log(f"generated {cfg.name} in {time.perf_counter() - t0:.1f}s")
    st = F.UngBuildStage(num_cross_edges=cfg.k_cross, max_degree=cfg.k_intra)
    t0 = time.perf_counter()
    st.prepare_inputs(X, lp, li)
    del X
    lng_s = time.perf_counter() - t0
    gids = st.mid_groups()
    begins = st.group_begin[gids].astype(np.uint32)
    sizes = (st.group_begin[gids + 1] - st.group_begin[gids]).astype(np.uint32)
    p_cross, _ = F.count_pairs(st.group_begin, st.out_ptr, st.out_idx)
    p_intra = int((sizes.astype(np.int64) * (sizes.astype(np.int64) - 1)).sum())
    log(f"groups={st.num_groups} lng_edges={len(st.out_idx)} mid_groups={len(gids)} "
        f"P_cross={p_cross:.3e} P_intra={p_intra:.3e} inputs {lng_s:.1f}s")

    ctx = st.ctx
    up = ctx.prepare_vectors(st.base)
    log(f"resident upload {up['h2d_ms']:.1f} ms ({st.base.nbytes / up['h2d_ms'] / 1e6:.1f} GB/s incl. PCIe)")

    def step():
        if args.sequential:
            s1 = ctx.cross_topk_device(st.group_begin, st.out_ptr, st.out_idx, cfg.k_cross)
        else:  # the mid groups' kNN runs on the second stream beside the cross tail
            s1 = ctx.cross_intra_begin(st.group_begin, st.out_ptr, st.out_idx, cfg.k_cross, begins, sizes,
                                       cfg.k_intra)
        t0 = time.perf_counter()
        _, ef, _, s3 = ctx.additional_edges(st.group_begin, st.out_ptr, st.out_idx, cfg.k_cross)
        s3["wall_ms"] = (time.perf_counter() - t0) * 1e3
        s3["edges"] = int(ef.size)
        s2 = ctx.group_knn_device(begins, sizes, cfg.k_intra) if args.sequential else ctx.intra_end()
        return s1, s2, s3

    warmup = max(args.warmup, 1 if args.steps <= 0 else 0)
    per = None
    for _ in range(warmup):
        t_w = time.perf_counter()
        step()
        ctx.synchronize()
        per = time.perf_counter() - t_w  # the last warmup step (the first one allocates)
    steps = args.steps
    if steps <= 0:  # enough timed steps for about 2.5 s at the last warmup step's pace
        steps = max(3, int(math.ceil(2.5 / max(per, 1e-4))))
    cross_stats, intra_stats, addl_stats = [], [], []
    ctx.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        s1, s2, s3 = step()
        cross_stats.append(s1)
        intra_stats.append(s2)
        addl_stats.append(s3)
    ctx.synchronize()
    wall = time.perf_counter() - t0
    ms_per_step = wall * 1e3 / steps
    log(f"{steps} timed steps: {ms_per_step:.3f} ms/step")
    # the timed cross calls' operands: fp16 (one product a coordinate pair), or bf16 pairs
    # (three) for a base set or a call that the fp16 ones cannot serve
    half = ctx.debug_error_bound()[3] and all(s["select_launches"] == 1 for s in cross_stats)

    # the drop-in calls with host output (D2H included), after the timed region: the cross
    # rows with distances and sizes, the FlatId rows alone (the reference's flat writeback,
    # src/gpu_cross_edge_output.cuh:87-103), the exact batch's packed rows [P x (K+1)]
    # (what build_fast_exact_cuda_batch hands to fill_tagore_batch_results,
    # src/tagore_graph_builder.cu:1354-1379) and the exact lists with distances
    dropin = [ctx.cross_topk(st.group_begin, st.out_ptr, st.out_idx, cfg.k_cross) for _ in range(3)]
    g_cross = (dropin[-1][0], dropin[-1][1])
    cross_rescanned = int(dropin[-1][3]["fallback_rows"])
    flat_dropin = [ctx.cross_topk(st.group_begin, st.out_ptr, st.out_idx, cfg.k_cross, with_dist=False,
                                  with_size=False)[3] for _ in range(3)]
    fd = cfg.k_intra
    tk, head_keep = max(st.tagore_k, fd + 1), (fd - 8 if fd > 8 else fd)

    def exact_batch():
        t0 = time.perf_counter()
        s_knn = ctx.group_knn_device(begins, sizes, fd)
        graph, _, s_pack = ctx.pack_anchor_rows(int(sizes.sum()), len(gids), tk, fd, head_keep, 1, 0, 0)
        return (time.perf_counter() - t0) * 1e3, s_knn, s_pack, graph

    packed_dropin = [exact_batch() for _ in range(3)]
    intra_dropin = [ctx.group_knn(begins, sizes, cfg.k_intra) for _ in range(2)]
    g_intra = (intra_dropin[-1][0], intra_dropin[-1][1], gids, begins, sizes)
    intra_rescanned = int(intra_dropin[-1][2]["fallback_rows"])

    def avg(lst, key):
        return float(np.mean([s[key] for s in lst]))

    sel_cross_ms = avg(cross_stats, "select_ms")
    sel_intra_ms = avg(intra_stats, "select_ms")
    d = cfg.dim
    dp = (d + 63) // 64 * 64 if half else (d + 31) // 32 * 32  # dimensions of an operand row
    # The cross select kernel's two floors: its MFMA work (one fp16 product, or three bf16
    # ones, per coordinate pair of 2 flops, against the dense 16-bit peak) and its
    # HBM traffic (measured with rocprofv3 on this kernel source, against 8 TB/s).  The
    # larger floor bounds it; without a valid traffic measurement the MFMA floor is used.
    sel_s = sel_cross_ms * 1e-3
    flops_cross = 2.0 * d * p_cross
    mfma_flops = (2.0 if half else 6.0) * dp * p_cross
    alg_bytes = float(cross_stats[-1]["select_bytes"])
    traffic, traffic_status = read_traffic(cfg.name) if not args.n else (None, "not measured (scaled run)")
    mfma_floor_ms = mfma_flops / (MFMA_16BIT_PEAK_TFLOPS * 1e12) * 1e3
    hbm_floor_ms = traffic / (HBM_PEAK_GBS * 1e9) * 1e3 if traffic else None
    mfma_tflops = mfma_flops / sel_s / 1e12
    if hbm_floor_ms is not None and hbm_floor_ms >= mfma_floor_ms:
        ach = traffic / sel_s / 1e9
        roofline = {"bound": "hbm", "achieved": round(ach, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                    "frac": round(ach / HBM_PEAK_GBS, 4), "traffic": traffic}
    else:
        roofline = {"bound": "mfma", "achieved": round(mfma_tflops, 3), "peak": MFMA_16BIT_PEAK_TFLOPS,
                    "unit": "TFLOP/s", "frac": round(mfma_tflops / MFMA_16BIT_PEAK_TFLOPS, 4), "traffic": traffic}
    roofline.update({
        "kernel": f"ung_select_kernel<8,*,false,2,{str(dp == 128).lower()},{str(half).lower()}> (cross edges, "
                  + ("register-query layout, " if dp == 128 else "") + "one launch per step)",
        "avg_launch_ms": round(sel_cross_ms, 4),
        "traffic_status": traffic_status,
        "streamed_operand_bytes_per_launch": alg_bytes,
        "hbm_floor_ms": round(hbm_floor_ms, 3) if hbm_floor_ms is not None else None,
        "mfma_flops_per_launch": mfma_flops, "mfma_floor_ms": round(mfma_floor_ms, 3),
        "mfma_tflops": round(mfma_tflops, 2), "mfma_frac": round(mfma_tflops / MFMA_16BIT_PEAK_TFLOPS, 4),
        "measured_hbm_gbs": round(traffic / sel_s / 1e9, 1) if traffic else None,
        "fp32_equiv_tflops": round(flops_cross / sel_s / 1e12, 2),
    })
    value = (p_cross + p_intra) / (ms_per_step * 1e-3)
    result = {
        "metric": METRIC, "value": value, "unit": "distance evals/s", "n_gpus": 1,
        "steps": steps, "warmup": warmup, "ms_per_step": round(ms_per_step, 3),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": f"f32 (certified {'fp16' if half else '3xbf16'} MFMA pre-select, exact f32 re-score)",
        "data": "synthetic",
        "config": {"workload": f"{cfg.name}: {cfg.n}x{cfg.dim} fp32 Gaussian mixture "
                               f"({cfg.n_centroids} centroids, sigma {cfg.sigma}), vocab {cfg.vocab}, "
                               f"{cfg.m_min}-{cfg.m_max} labels Zipf({cfg.zipf_s}); cross k={cfg.k_cross} + "
                               f"intra exact K={cfg.k_intra} for 128<=n<=4096",
                   "groups": st.num_groups, "lng_edges": int(len(st.out_idx)), "mid_groups": int(len(gids)),
                   "P_cross": int(p_cross), "P_intra": int(p_intra),
                   "intra_overlapped": not args.sequential},
        "roofline": roofline,
        "breakdown": {
            "cross_wall_ms": round(avg(cross_stats, "wall_ms"), 3),
            "cross_plan_ms": round(avg(cross_stats, "plan_ms"), 3),
            "cross_h2d_ms": round(avg(cross_stats, "h2d_ms"), 3),
            "cross_select_ms": round(sel_cross_ms, 3),
            "cross_merge_ms": round(avg(cross_stats, "merge_ms"), 3),
            "cross_fallback_ms": round(avg(cross_stats, "fallback_ms"), 3),
            "cross_fallback_rows": int(cross_stats[-1]["fallback_rows"]),
            "cross_padded_pairs": int(cross_stats[-1]["padded_pairs"]),
            "additional_wall_ms": round(avg(addl_stats, "wall_ms"), 3),
            "additional_kernel_ms": round(avg(addl_stats, "kernel_ms"), 3),
            "additional_edges": int(addl_stats[-1]["edges"]),
            "additional_query_rows": int(addl_stats[-1]["rows"]),
            "intra_wall_ms": round(avg(intra_stats, "wall_ms"), 3),
            "intra_select_ms": round(sel_intra_ms, 3),
            "intra_merge_ms": round(avg(intra_stats, "merge_ms"), 3),
            "intra_fallback_rows": int(intra_stats[-1]["fallback_rows"]),
            "intra_select_tflops": round(2.0 * d * p_intra / (sel_intra_ms * 1e-3) / 1e12, 3) if p_intra else None,
            "cross_evals_per_s": p_cross / (avg(cross_stats, "wall_ms") * 1e-3),
            "resident_upload_ms": round(up["h2d_ms"], 3),
            "cross_dropin_wall_ms": round(float(np.mean([s[3]["wall_ms"] for s in dropin])), 3),
            "cross_dropin_d2h_ms": round(float(np.mean([s[3]["d2h_ms"] for s in dropin])), 3),
            "cross_flat_dropin_wall_ms": round(float(np.mean([s["wall_ms"] for s in flat_dropin])), 3),
            "cross_flat_dropin_d2h_ms": round(float(np.mean([s["d2h_ms"] for s in flat_dropin])), 3),
            "exact_batch_packed_dropin_wall_ms": round(float(np.mean([x[0] for x in packed_dropin])), 3),
            "exact_batch_packed_d2h_ms": round(float(np.mean([x[2]["d2h_ms"] for x in packed_dropin])), 3),
            "exact_batch_packed_bytes": int(packed_dropin[-1][3].nbytes),
            "intra_dropin_wall_ms": round(float(np.mean([s[2]["wall_ms"] for s in intra_dropin])), 3),
            "intra_dropin_d2h_ms": round(float(np.mean([s[2]["d2h_ms"] for s in intra_dropin])), 3),
            "dropin_note": "host-output calls after the timed steps, D2H included (pinned staging, pieces copied "
                           "to the caller's memory on the host threads while the next ones transfer): "
                           "cross_dropin = ung_hip_cross_topk with FlatId rows + distances + sizes; "
                           "cross_flat_dropin = the FlatId rows alone; exact_batch_packed_dropin = "
                           "ung_hip_group_knn_device + ung_hip_pack_anchor_rows with the packed rows "
                           f"[P x {fd + 1}] u32 on the host; intra_dropin = ung_hip_group_knn lists + distances; "
                           "the one-time upload of X is resident_upload_ms",
        },
    }
    log("cpu baseline + parity ..." if not args.no_cpu_baseline else "parity ...")
    base, parity = cpu_leg_and_parity(st, cfg, g_cross, g_intra, p_cross, p_intra, args.cpu_seconds,
                                      timed=not args.no_cpu_baseline)
    parity["cross_rescanned_rows"] = cross_rescanned
    parity["intra_rescanned_rows"] = intra_rescanned
    result["parity"] = parity
    if base is not None:
        result["cpu_baseline"] = base
    st.close()
    if args.calib_copy:
        calib_copy(1 << 30)
    print(json.dumps(result), flush=True)


if __name__ == "__main__":
    main()
