#!/usr/bin/env python3
"""Benchmark of the neighbor-partitioned aggregation path on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--workload gcn2|share|gin|big|copy|convert|gather|vendor] [--no-cpu]

Default workload (`gcn2`): 2-layer GCN forward on the whole graph -- seeded RMAT
power-law graph (a=.57 b=.19 c=.19), 233,000 nodes, ~114 M undirected edges,
self loops, D^-1/2 (A+I) D^-1/2 weighting; fp32 features 602 -> 16 -> 41, Glorot
weights; ps=16, the other knobs from the library's search (run before timing).
One step = dense, aggregate, dense, aggregate, softmax, all inputs resident in
HBM.  Prints ONE JSON line: `value` = median forward ms over the timed steps (HIP
events; the host-clock median and the wall mean are beside it), what the set-up
of that setting cost, the same forward with the configuration's literal knobs and
with the library's rules alone, and the CPU oracle timed on this host's cores.
The metric's second half -- aggregation GB/s against HBM peak -- is quoted on
the HBM-resident workload, rank 0's 1/8 share, which the default
run times in the same process: that kernel is the `roofline` object.  The GCN
graph's tables live in cache; its aggregation gets ceilings it can be below
(compulsory HBM bytes, gather rates of the L2 and the LDS) under `detail`.
A result outside its tolerance against the CPU oracle makes the run fail.

`share` times the aggregation alone on rank 0's 1/8 share of a 4.2 M-node RMAT
graph with the remote rows pre-staged in a second HBM table; `gin` the 5-layer
GIN forward; `big` the bf16 large-share aggregation and update; `copy` the
stream-copy yardstick; `convert` the 2:1 read/write yardstick of the dense update (a bare fp32 -> bf16 conversion, by
the order in which the workgroups walk through memory); `gather` the random-gather yardstick (what the memory system sustains for row gathers from
tables of the benchmark sizes); `vendor` the library's kernels beside torch.mm and
torch.sparse.mm on the benchmark shapes.
"""
from __future__ import annotations

import argparse
import json
import re
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBPS = 8000.0  # MI355X HBM3E, published
COLD_COPIES = 6           # disjoint copies of the share's working set the cold-cache leg rotates over


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def hbm_roofline(kernel, nbytes, ms, traffic):
    """Roofline object of an aggregation kernel against the HBM peak.  achieved = algorithmic bytes / time.  Where hub
    rows are served from the caches that ratio can pass the peak and bounds nothing: `frac` is then taken from the measured
    HBM-side traffic of the same kernel (committed counter runs), and the algorithmic ratio is given under its own name."""
    achieved = nbytes / (ms * 1e-3) / 1e9
    r = {"bound": "hbm", "kernel": kernel, "achieved": round(achieved, 1), "peak": HBM_PEAK_GBPS, "unit": "GB/s",
         "algorithmic_bytes": nbytes, "avg_launch_ms": round(ms, 4), **traffic}
    ratio = achieved / HBM_PEAK_GBPS
    if ratio <= 1.0:
        r["frac"] = round(ratio, 4)
    else:
        r["algorithmic_gbps_over_hbm_peak"] = round(ratio, 4)
        t = traffic.get("traffic")
        r["frac"] = round(t / (ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4) if t else None
        r["frac_is"] = "measured HBM-side traffic / time / peak: the algorithmic ratio exceeds 1 because hub rows are served from L2"
    return r


def agg_bytes(nnz, rows, dim, s_in=4, ptr_arrays=1, gin=False):
    """Algorithmic bytes of one aggregation call: per edge one index and one feature row, per row one output
    row and the row pointers; no cache credit."""
    b = nnz * (4 + dim * s_in) + rows * dim * 4 + (rows + 1) * 4 * ptr_arrays
    if gin:
        b += rows * dim * s_in
    return b


class StageTimer:
    """HIP events (torch wrappers on the stream the library launches on) around each stage of every step; the events
    are created before the timed region starts."""

    def __init__(self, torch, names, steps=64):
        self.torch = torch
        self.names = names
        self.pool = [[torch.cuda.Event(enable_timing=True) for _ in range(len(names) + 1)] for _ in range(steps)]
        self.events = []

    def step(self, stages):
        ev = self.pool.pop() if self.pool else [self.torch.cuda.Event(enable_timing=True) for _ in range(len(self.names) + 1)]
        ev[0].record()
        for i, fn in enumerate(stages):
            fn()
            ev[i + 1].record()
        self.events.append(ev)

    def per_stage(self):
        """-> {name: [ms of each step]}"""
        self.torch.cuda.synchronize()
        return {k: [ev[i].elapsed_time(ev[i + 1]) for ev in self.events] for i, k in enumerate(self.names)}

    def per_step(self):
        self.torch.cuda.synchronize()
        return [ev[0].elapsed_time(ev[-1]) for ev in self.events]

    def averages(self):
        return {k: sum(v) / max(1, len(v)) for k, v in self.per_stage().items()}

    def medians(self):
        return {k: float(np.median(v)) for k, v in self.per_stage().items()}


def time_steps(torch, stages, names, steps, warmup):
    """W untimed steps, then exactly K steps between two device synchronisations.  -> dict(wall_ms = host clock over the
    K steps / K, event_median_ms = median over steps of the HIP-event time of a step, host_median_ms = median host-clock
    time of a step measured in a second pass with a synchronisation after every step, stage_avg / stage_median)."""
    for _ in range(warmup):
        for fn in stages:
            fn()
    timer = StageTimer(torch, names, steps)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        timer.step(stages)
    torch.cuda.synchronize()
    wall_ms = (time.perf_counter() - t0) * 1e3 / steps
    host = []
    for _ in range(steps):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for fn in stages:
            fn()
        torch.cuda.synchronize()
        host.append((time.perf_counter() - t0) * 1e3)
    return {"wall_ms": wall_ms, "event_median_ms": float(np.median(timer.per_step())), "host_median_ms": float(np.median(host)),
            "stage_avg": timer.averages(), "stage_median": timer.medians()}


def fail_on_parity(res, checks):
    """checks: [(name, error, tolerance)].  A result outside its tolerance voids the measurement: the line is still
    printed (value null) and the process exits non-zero."""
    bad = [(n, e, t) for n, e, t in checks if not (e <= t)]
    if bad:
        res["value"] = None
        res["parity_failed"] = ["%s: %.3e > %.1e" % b for b in bad]
        print(json.dumps(res), flush=True)
        log("PARITY FAILED:", res["parity_failed"])
        sys.exit(4)


# A dense cell's products for 16 columns: 512 x 256 positions in 384 sparse matrix instructions, each as long as a dense bf16 one of
# 16 x 16 x 32 (16,384 operations), at the 2.5 PFLOP/s of dense bf16.
CELL_NS_PER_16_COLUMNS = 384 * 16384 / 2.5e15 * 1e9


def gather_ceiling(torch, host, ld_bytes, row_bytes, table_rows, edges, ms, core_edges=0, cell_edges=0, cells=0, dim=0):
    """Where the feature table is cache resident the HBM peak does not bound the kernel; the L2 and, for the dense core,
    the LDS do.  Measured live with the library's yardsticks (random row reads of the kernel's geometry, no index
    stream, no reduction): from a 3 MB table (every load hits the L2), from a table of the kernel's size, and from an
    LDS tile.  The ceiling of a call is the longer of its two halves at those rates -- the core block's edges at the LDS
    rate, the remaining edges at the all-hit L2 rate -- because the two kernels run side by side on different units.  Dense
    cells are not gathered and run before the rest: what the matrix cores need for their products at full rate is added."""
    sink = torch.empty(262144, device="cuda")
    small = max(1, (3 << 20) // ld_bytes)
    table = torch.zeros(max(small, table_rows) * ld_bytes, dtype=torch.uint8, device="cuda")

    def rate(fn):
        fn(1)
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        done = sum(fn(i + 2) for i in range(3))
        e1.record()
        torch.cuda.synchronize()
        return done / (e0.elapsed_time(e1) * 1e-3) / 1e9

    out = {}
    for key, rows in (("all_l2_hits", small), ("uniform_random_whole_table", table_rows)):
        out[key + "_G_rows_per_s"] = round(rate(lambda sd: host.gather_probe(sink, table, rows, ld_bytes, row_bytes, 100_000_000, seed=sd)), 1)
    out["lds_G_rows_per_s"] = round(rate(lambda sd: host.lds_probe(sink, (row_bytes + 15) // 16 * 16, 400_000_000, seed=sd)), 1)
    out["kernel_G_rows_per_s"] = round(edges / (ms * 1e-3) / 1e9, 1)
    t_l2 = (edges - core_edges - cell_edges) / (out["all_l2_hits_G_rows_per_s"] * 1e9) * 1e3
    t_lds = core_edges / (out["lds_G_rows_per_s"] * 1e9) * 1e3
    out["edges_from_lds"], out["edges_through_l2"] = int(core_edges), int(edges - core_edges - cell_edges)
    out["edges_in_dense_cells"] = int(cell_edges)
    t_cells = cells * ((dim + 15) // 16) * CELL_NS_PER_16_COLUMNS * 1e-6
    ceiling = t_cells + max(t_l2, t_lds)
    out["ceiling_ms"] = round(ceiling, 4)
    out["ceiling_is"] = ("cells' products at the matrix cores' rate = %.4f ms + " % t_cells if cells else "") + \
        "max(edges through the L2 / all-hit rate = %.4f ms, edges from LDS / LDS rate = %.4f ms)" % (t_l2, t_lds)
    out["frac_of_gather_ceiling"] = round(ceiling / ms, 3)
    return out


# HBM-side bytes per aggregation call (kernel + fix-up), from rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE runs scaled by
# what the same counters read for a 1 GiB copy (x2.000 / x1.000), and the (wpb, dist) of those runs.  The figure moves
# by well under 1 % with (wpb, dist): the gathers are the same, only the carries differ.  Default graphs only.
MEASURED_TRAFFIC = {
    "gcn2_agg2": (28_216_496_128, (4, 16)),
    "gcn2_agg1": (6_481_731_891, (4, 16)),
    "gcn2_agg2_blocked": (7_519_810_150, (4, 16)),   # column blocks of 49152 ids: partial rows and their reduction included
    "gcn2_agg1_blocked": (1_746_502_963, (4, 16)),
    "gcn2_agg2_core36864_blocked": (5_892_428_288, (4, 16)),   # what the cost model picks at width 41: dense core of 36864 rows, workgroups of equal work
    "gcn2_agg1_core61440_blocked": (1_786_640_486, (4, 8)),    # ... and at width 16: 61440 rows
    "gcn2_agg2_cells_blocked": (5_560_100_045, (4, 16)),   # dense cells instead of the core, by rule: staging, cells, their reduction, rest, finish
    "gcn2_agg1_cells_blocked": (1_431_298_355, (4, 8)),
    "share_agg": (1_213_309_056, (4, 4)),
    "share_agg_compact": (1_028_547_520, (4, 4)),   # remote rows staged compactly (one row per distinct remote id)
    "gin_agg": (25_550_513_561, (16, 1)),
    "gin_agg_core98304": (15_702_715_472, (8, 8)),   # the size the cost model picks (row groups of 512 rows), the knobs the rules pick
    "big_agg": (60_511_998_361, (4, 16)),
}


def load_traffic(kernel_key, args, blk=-1, core=-1, cells=0):
    """{"traffic": bytes or None, "traffic_measured_at": knobs} for the roofline object."""
    if core > 0:
        kernel_key += "_core%d" % core
    if cells > 0:
        kernel_key += "_cells"
    if blk > 0:
        if blk != 49152:
            return {"traffic": None}
        kernel_key += "_blocked"
    if args.small or args.ps != 16 or (kernel_key.startswith("share_agg") and args.share_density != 1) or \
            (kernel_key == "big_agg" and args.big_scale != 0) or kernel_key not in MEASURED_TRAFFIC:
        return {"traffic": None}
    nbytes, (w, d) = MEASURED_TRAFFIC[kernel_key]
    return {"traffic": nbytes, "traffic_measured_at": "ps=16 wpb=%d dist=%d%s%s" % (w, d, ", column blocks of 49152 ids" if blk > 0 else "",
                                                                                 ", dense core of %d rows" % core if core > 0 else
                                                                                 ", %d dense cells" % cells if cells else "")}


class Knobs:
    """(ps, wpb, dist, column blocking, dense core) of one aggregation shape.  Default: the command line's values, where 0
    leaves the choice to the library's rules and its cost model for the dense core (no measurement).  With `search`
    (a callable) the library's search measures the settings on this input instead -- the reference fixes its setting per
    dataset from the same kind of sweep, bench_MGG_DSE_*.py."""

    def __init__(self, args, search=None):
        self.ps, self.wpb, self.dist, self.blk, self.core = args.ps, args.wpb, args.dist, args.col_block_rows, args.core_rows
        self.cells = 0  # dense cells the library chose (their plan has no size to pass: core_rows stays 0)
        self.searched_ms = None
        if search is not None:
            k, ms = search(args.ps, args.col_block_rows, args.core_rows)
            self.ps, self.wpb, self.dist, self.blk, self.core = k["ps"], k["wpb"], k["dist"], k["col_block_rows"], k["core_rows"]
            self.searched_ms = ms
            log("search: %s (%.4f ms)" % (self, ms))

    def tuple(self):
        return (self.ps, self.wpb, self.dist, self.blk, self.core)

    def saw_cells(self, kernel):
        m = re.search(r" cells=(\d+)", kernel)
        self.cells = int(m.group(1)) if m else 0

    def observe(self, host, call):
        """Where choices were left to the library: run the call once and read back what it used."""
        call()
        k = host.last_agg_kernel()
        m = re.search(r"blocks=(\d+)", k)
        if self.blk == 0:
            self.blk = 49152 if m and int(m.group(1)) > 1 else -1
        if self.core == 0:
            self.saw_cells(k)
            m = re.search(r"core=(\d+)", k)
            self.core = 0 if self.cells else int(m.group(1)) if m else -1
        m = re.search(r"wpb=(\d+) dist=(\d+)", k)
        if m:
            self.wpb, self.dist = (self.wpb or int(m.group(1))), (self.dist or int(m.group(2)))
        return k

    def __str__(self):
        return "ps=%d wpb=%d dist=%d %s%s" % (self.ps, self.wpb, self.dist,
                                              "column blocks of %d ids" % self.blk if self.blk > 0 else
                                              ("plain order" if self.blk < 0 else "order by rule"),
                                              ", dense core of %d rows from LDS" % self.core if self.core > 0 else
                                              ", %d dense cells on the matrix cores" % self.cells if self.cells else "")


def bench_gcn2(args, torch, host):
    V, scale, draws = 233_000, 18, 216_000_000
    in_dim, hidden, out_dim = 602, 16, 41
    if args.small:
        V, scale, draws = 20_000, 15, 2_000_000
    t0 = time.time()
    ptr, col = host.gen_rmat(scale, V, draws, seed=42)
    nnz = int(len(col))
    log("graph: V=%d nnz=%d (undirected %d) in %.1fs" % (V, nnz, (nnz - V) // 2, time.time() - t0))
    X = host.fill_normal((V, in_dim), seed=1)
    W1 = host.glorot(in_dim, hidden, seed=2)
    W2 = host.glorot(hidden, out_dim, seed=3)
    deg = np.diff(ptr).astype(np.float64)
    s = (1.0 / np.sqrt(np.maximum(deg, 1.0))).astype(np.float32)

    # Device layout: the 41-wide layer is computed at width 44 (zero padding columns) in tables with a row pitch of 48
    # floats, so its rows move as whole dwordx4 loads and start on 64-byte boundaries (a 192-byte row then touches two
    # 128-byte lines, never three); bytes and flops are still counted at width 41.
    ldo = (out_dim + 3) & ~3
    W2p = np.zeros((hidden, ldo), np.float32)
    W2p[:, :out_dim] = W2
    dev = "cuda"
    d_ptr = torch.from_numpy(ptr).to(dev)
    d_col = torch.from_numpy(col).to(dev)
    d_zero_ptr = torch.zeros(V + 1, dtype=torch.int32, device=dev)
    d_zero_col = torch.zeros(1, dtype=torch.int32, device=dev)
    d_X = torch.from_numpy(X).to(dev)
    d_W1 = torch.from_numpy(W1).to(dev)
    d_W2 = torch.from_numpy(W2p).to(dev)
    d_s = torch.from_numpy(s).to(dev)
    d_Y1 = torch.empty(V, hidden, device=dev)
    d_H1 = torch.empty(V, hidden, device=dev)
    pitch = max(ldo, args.pitch41 or 48)  # row pitch of the 41-wide tables in floats
    d_Y2 = torch.zeros(V, pitch, device=dev)
    d_H2 = torch.zeros(V, pitch, device=dev)
    d_P = torch.zeros(V, pitch, device=dev)  # class probabilities, in rows of the same pitch
    names = ["dense1", "agg1", "dense2", "agg2"]

    def forward_stages(k1, k2):
        """The stages of one forward with the given (ps, wpb, dist, order, core) per aggregation width: dense, aggregate,
        dense, aggregate with the row softmax as its epilogue (the reference's last two calls, src/mgg_np_div_mem.cu:221-225,
        in one).  The last aggregation sums 41 columns; its rows are read in 16-byte pieces out of a pitch of 48."""
        return [
            lambda: host.dense_forward(d_Y1, d_X, d_W1, V, in_dim, hidden, row_scale=d_s),
            lambda: host.mgg_SAG_np_div(d_H1, d_Y1, d_ptr, d_col, d_zero_ptr, d_zero_col, 0, V, hidden, V, 0, k1[0], k1[1], k1[2],
                                        row_scale_out=d_s, col_block_rows=k1[3], core_rows=k1[4]),
            lambda: host.dense_forward(d_Y2, d_H1, d_W2, V, hidden, ldo, row_scale=d_s, ld_out=pitch),
            lambda: host.mgg_SAG_np_div(d_P, d_Y2, d_ptr, d_col, d_zero_ptr, d_zero_col, 0, V, out_dim, V, 0, k2[0], k2[1], k2[2],
                                        row_scale_out=d_s, col_block_rows=k2[3], core_rows=k2[4], ld_in=pitch, ld_out=pitch, softmax=True),
        ]

    d_Y1.zero_()
    d_Y2.zero_()
    extra = {}
    # (1) The configuration's literal knobs (ps 16, wpb 8, the reference's default interleaved_dist 1, the reference's
    # row-major order, no dense core) and (2) the library's rules alone (no search): both timed in this run, so the
    # price of the searched setting below can be set against what it buys.
    lit = (16, 8, 1, -1, -1)
    if args.only_headline:
        return gcn2_headline_only(args, torch, host, forward_stages, names)
    t0 = time.perf_counter()
    for fn in forward_stages(lit, lit):
        fn()
    torch.cuda.synchronize()
    first_call_ms = (time.perf_counter() - t0) * 1e3
    r = time_steps(torch, forward_stages(lit, lit), names, max(3, args.steps // 2), 1)
    extra["literal_knobs"] = {"ps": 16, "wpb": 8, "dist": 1, "col_block_rows": -1, "core": -1, "fwd_ms": round(r["event_median_ms"], 4),
                              "stage_ms": {k: round(v, 4) for k, v in r["stage_median"].items()},
                              "first_forward_ms_with_plan_build": round(first_call_ms, 2)}
    rule = (args.ps, 0, 0, 0, -1)
    for fn in forward_stages(rule, rule):
        fn()
    torch.cuda.synchronize()
    r = time_steps(torch, forward_stages(rule, rule), names, max(3, args.steps // 2), 1)
    extra["rules_without_dense_core"] = {"fwd_ms": round(r["event_median_ms"], 4),
                                         "knobs": "ps=%d, wpb / dist / order by the library's rules, dense core off" % args.ps,
                                         "stage_ms": {k: round(v, 4) for k, v in r["stage_median"].items()}}
    log("literal knobs %.4f ms, rules without the dense core %.4f ms" % (extra["literal_knobs"]["fwd_ms"], r["event_median_ms"]))

    # (3) the headline: knobs as the command line gives them; by default everything is left to the library -- its rules
    # for ps / wpb / dist / order and its cost model (degree histogram x row width) for the dense core.  No search, no
    # measurement; the first forward builds the plans (on the GPU) and is timed as the set-up.  With --tune the
    # library's search picks the knobs instead, as it does in (4) for comparison.
    search1 = lambda ps, blk, core: host.tune_np_div(d_H1, d_Y1, d_ptr, d_col, d_zero_ptr, d_zero_col, 0, V, hidden, V, ps,
                                                     row_scale_out=d_s, col_block_rows=blk, core_rows=core)
    search2 = lambda ps, blk, core: host.tune_np_div(d_P, d_Y2, d_ptr, d_col, d_zero_ptr, d_zero_col, 0, V, out_dim, V, ps,
                                                     row_scale_out=d_s, col_block_rows=blk, core_rows=core, ld_in=pitch, ld_out=pitch, softmax=True)
    host.release_cached()   # the plans of (1) and (2) are gone: the set-up below is what a first call costs
    setup = {}
    mark = host.cache_stats()
    t0 = time.perf_counter()
    k1 = Knobs(args, search1 if args.tune else None)
    k2 = Knobs(args, search2 if args.tune else None)
    stages = forward_stages(k1.tuple(), k2.tuple())
    k1.observe(host, stages[1])
    mid = host.cache_stats()
    kstr = k2.observe(host, stages[3])
    torch.cuda.synchronize()
    setup["first_use_of_both_aggregations"] = (time.perf_counter() - t0) * 1e3
    now = host.cache_stats()
    # the core plan the last aggregation uses: its own when the two widths got different core sizes, else the shared one
    agg2_core_plan_bytes = now["core_plan_bytes"] - mid["core_plan_bytes"] or now["core_plan_bytes"] - mark["core_plan_bytes"]
    setup["core_plan_build"] = now["core_plan_build_ms"] - mark["core_plan_build_ms"]
    setup["plan_build"] = now["plan_build_ms"] - mark["plan_build_ms"]
    setup["search"] = now["search_ms"] - mark["search_ms"]
    setup = {k: round(v, 2) for k, v in setup.items()}
    setup["note"] = ("host clock; first_use_of_both_aggregations is everything between cold caches and two finished aggregation calls and includes "
                     "the builds listed beside it" + ("" if args.tune else "; no search ran for the headline"))
    stages = forward_stages(k1.tuple(), k2.tuple())
    m = re.search(r"core_nnz=(\d+)", kstr)
    core_edges = int(m.group(1)) if m else 0

    r = time_steps(torch, stages, names, args.steps, args.warmup)
    avg, med = r["stage_avg"], r["stage_median"]
    held = host.cache_stats()
    extra["setup_ms"] = setup
    extra["rule_only_fwd_ms"] = None if args.tune else round(r["event_median_ms"], 4)  # the headline itself: rules and cost model, no search
    extra["device_bytes_held_by_library"] = {k: int(held[k]) for k in ("plan_bytes", "core_plan_bytes", "workspace_bytes", "core_scratch_bytes")}
    log("stage ms (median):", {k: round(v, 4) for k, v in med.items()}, "per forward: events median %.4f, host median %.4f, wall mean %.4f"
        % (r["event_median_ms"], r["host_median_ms"], r["wall_ms"]))

    b1 = agg_bytes(nnz, V, hidden)
    b2 = agg_bytes(nnz, V, out_dim)
    # The GCN graph's feature tables (15 / 45 MB) live in cache: algorithmic bytes / time exceeds the HBM peak and
    # bounds nothing.  What the aggregation must move through HBM at least (index lists and ids actually streamed, the
    # table once, the output once) and what the L2 / LDS sustain for its gathers are the ceilings it can be below.
    agg2 = {"kernel": "%sk_agg (agg2 with the softmax epilogue, dim %d)" % ("k_core_sell + " if k2.core > 0 else "k_cells + " if k2.cells else "", out_dim), "knobs": str(k2),
            "avg_launch_ms": round(avg["agg2"], 4), "median_launch_ms": round(med["agg2"], 4),
            "algorithmic_bytes": b2, "algorithmic_gbps": round(b2 / (avg["agg2"] * 1e-3) / 1e9, 1),
            "algorithmic_gbps_over_hbm_peak": round(b2 / (avg["agg2"] * 1e-3) / 1e9 / HBM_PEAK_GBPS, 3),
            **load_traffic("gcn2_agg2", args, k2.blk, k2.core, k2.cells)}
    comp = agg2_core_plan_bytes if k2.core > 0 or k2.cells else nnz * 4   # lists or cells + remaining ids, or the plain id stream
    comp += V * pitch * 4 + V * out_dim * 4 + (V + 1) * 4           # the table once, the output once, the row pointers
    agg2["compulsory_hbm_bytes"] = int(comp)
    agg2["frac_compulsory"] = round(comp / (avg["agg2"] * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4)
    if agg2.get("traffic"):
        agg2["frac_traffic"] = round(agg2["traffic"] / (avg["agg2"] * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4)
    agg2["gather_ceiling"] = gather_ceiling(torch, host, pitch * 4, ldo * 4, V, nnz, avg["agg2"], core_edges if k2.core > 0 else 0,
                                            core_edges if k2.cells else 0, k2.cells, out_dim)
    extra["launches_per_forward"] = ("dense 1 + aggregation %d + dense 1 + aggregation %d (softmax inside)" %
                                     ((5, 5) if (k2.core > 0 or k2.cells) and k2.blk > 0 else ((6, 6) if k2.core > 0 or k2.cells else (2, 2))))
    extra["agg2_cache_resident"] = agg2
    extra.update({
        "stage_ms": {k: round(v, 4) for k, v in med.items()},
        "stage_ms_mean": {k: round(v, 4) for k, v in avg.items()},
        "fwd_ms": {"hip_events_median": round(r["event_median_ms"], 4), "host_clock_median": round(r["host_median_ms"], 4),
                   "host_clock_mean_over_the_timed_region": round(r["wall_ms"], 4)},
        "agg1_gbps": round(b1 / (avg["agg1"] * 1e-3) / 1e9, 1),
        "dense1_gflops": round(2.0 * V * in_dim * hidden / (avg["dense1"] * 1e-3) / 1e9, 1),
        "dense1_gbps": round((V * in_dim * 4 + V * hidden * 4) / (avg["dense1"] * 1e-3) / 1e9, 1),
    })

    # The same forward with the second layer re-associated, (A H1) W2 instead of A (H1 W2): the aggregation then runs
    # at width 16 instead of 41.  Mathematically identical; reported beside the reference's order, not instead of it.
    d_s2 = d_s * d_s
    d_G = torch.empty(V, hidden, device=dev)
    d_P2 = torch.empty(V, out_dim, device=dev)
    d_Y2b = torch.empty(V, out_dim, device=dev)
    d_W2u = torch.from_numpy(W2).to(dev)
    alt = [
        lambda: host.dense_forward(d_Y1, d_X, d_W1, V, in_dim, hidden, row_scale=d_s),
        lambda: host.mgg_SAG_np_div(d_H1, d_Y1, d_ptr, d_col, d_zero_ptr, d_zero_col, 0, V, hidden, V, 0, k1.ps, k1.wpb, k1.dist,
                                    row_scale_out=d_s2, col_block_rows=k1.blk, core_rows=k1.core),
        lambda: host.mgg_SAG_np_div(d_G, d_H1, d_ptr, d_col, d_zero_ptr, d_zero_col, 0, V, hidden, V, 0, k1.ps, k1.wpb, k1.dist,
                                    row_scale_out=d_s, col_block_rows=k1.blk, core_rows=k1.core),
        lambda: host.dense_forward(d_Y2b, d_G, d_W2u, V, hidden, out_dim),
        lambda: host.softmax_forward(d_P2, d_Y2b, V, out_dim),
    ]
    P_main = d_P[:, :out_dim].clone()
    ra = time_steps(torch, alt, ["dense1", "agg1", "aggA", "dense2", "softmax"], max(3, args.steps // 2), 1)
    extra["aggregate_first_order"] = {"fwd_ms": round(ra["event_median_ms"], 4),
                                      "softmax_max_abs_diff_vs_reference_order": float((d_P2 - P_main).abs().max())}
    # leave the reference-order results in the buffers the parity check reads
    for fn in stages:
        fn()
    torch.cuda.synchronize()
    H1_gpu, P_gpu, Y1_gpu = d_H1.cpu().numpy(), d_P[:, :out_dim].cpu().numpy(), d_Y1.cpu().numpy()
    agg1_ms = avg["agg1"]
    # (4) the library's search on the same inputs (ps x order x core size x wpb x dist measured on the device), timed in the
    # same run: what the rules and the cost model leave on the table, and what finding out costs.
    if not args.tune and not args.no_search:
        mark = host.cache_stats()
        t0 = time.perf_counter()
        s1 = Knobs(args, search1)
        s1.saw_cells(host.last_agg_kernel())
        s2 = Knobs(args, search2)
        s2.saw_cells(host.last_agg_kernel())
        torch.cuda.synchronize()
        search_wall = (time.perf_counter() - t0) * 1e3
        now = host.cache_stats()
        rs_ = time_steps(torch, forward_stages(s1.tuple(), s2.tuple()), names, max(3, args.steps // 2), 1)
        extra["searched"] = {"fwd_ms": round(rs_["event_median_ms"], 4), "width16": str(s1), "width41": str(s2),
                             "stage_ms": {k: round(v, 4) for k, v in rs_["stage_median"].items()},
                             "search_wall_ms": round(search_wall, 1),
                             "of_which_plan_builds_ms": round(now["plan_build_ms"] + now["core_plan_build_ms"] - mark["plan_build_ms"] - mark["core_plan_build_ms"], 1),
                             "headline_over_searched": round(r["event_median_ms"] / rs_["event_median_ms"], 4)}
        log("searched: %.4f ms per forward (headline / searched = %.3f), search took %.0f ms" % (rs_["event_median_ms"], extra["searched"]["headline_over_searched"], search_wall))
    host.release_cached()

    # The HBM-resident workload of the same run: rank 0's 1/8 share, the kernel the roofline is quoted on.
    share = share_record(args, torch, host, with_cpu=not args.no_cpu)
    extra["share"] = share

    checks = list(share.pop("_checks"))
    if not args.small and not args.no_extra:
        more, more_checks = other_configs(args, torch, host)
        extra.update(more)
        checks += more_checks

    cpu = None
    parity = None
    if not args.no_cpu:
        from oracle import orc
        th = orc.max_threads()
        t0 = time.perf_counter()
        P_ref, H2_ref, H1_ref = orc.gcn2_forward(X, W1, W2, ptr, col, None, None, 0, V, V, rs=s, f64=False, threads=th)
        cpu_s = time.perf_counter() - t0
        cpu = {"value": round(cpu_s * 1e3, 1), "unit": "ms", "cores": th, "kind": "port",
               "sample": "1 full forward of the same workload (OpenMP over rows, fp32)"}
        parity = {"softmax_max_abs_err": float(np.abs(P_gpu - P_ref).max()), "softmax_tolerance": 1e-5,
                  "h1_max_rel_err": float(np.abs(H1_gpu - H1_ref).max() / np.abs(H1_ref).max()), "h1_tolerance": 1e-5,
                  "share_max_err_over_abs_sum": share["parity"]["max_err_over_abs_sum"] if share.get("parity") else None}
        checks += [("softmax |gpu - cpu|", parity["softmax_max_abs_err"], 1e-5), ("h1 relative error", parity["h1_max_rel_err"], 1e-5)]
        log("cpu forward %.1f ms on %d threads; parity %s" % (cpu_s * 1e3, th, parity))
        if orc.have_ref():
            # The reference's own CPU aggregation (SAG_ref, serial), compiled from its source: first rows of agg1
            # worth about 20 M edges, on the first layer's output.
            k = int(np.searchsorted(ptr, 20_000_000))
            k = max(1, min(k, V))
            t0 = time.perf_counter()
            got = orc.ref_sag_ref(Y1_gpu, ptr[: k + 1], col[: ptr[k]])
            ref_s = time.perf_counter() - t0
            mine = H1_gpu[:k] / s[:k, None]
            cpu["reference_sag_ref"] = {"m_edges_per_s": round(int(ptr[k]) / ref_s / 1e6, 1), "cores": 1,
                                        "sample": "rows 0..%d of agg1 (%d edges), width 16" % (k - 1, int(ptr[k])),
                                        "gpu_m_edges_per_s": round(nnz / (agg1_ms * 1e-3) / 1e6, 1),
                                        "max_rel_diff_vs_gpu": float(np.abs(got - mine).max() / np.abs(got).max())}

    res = {
        "metric": "gcn_2layer_fwd_ms", "value": round(r["event_median_ms"], 4), "unit": "ms", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(r["wall_ms"], 4), "higher_is_better": False, "scaling": "weak",
        "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"workload": "configs[1]: 2-layer GCN forward, RMAT(a=.57,b=.19,c=.19) V=%d nnz=%d (self loops, sym-norm), "
                               "602->16->41 fp32; width 16: %s; width 41: %s.  value = median over the timed steps (HIP events); "
                               "aggregation GB/s vs HBM peak (roofline) on %s" % (V, nnz, k1, k2, share["workload"])},
        "roofline": share["roofline"], "cpu_baseline": cpu, "parity": parity, "detail": extra,
    }
    fail_on_parity(res, checks)
    return res


def other_configs(args, torch, host):
    """configs[4] (large bf16 share: aggregation + 128x128 update) and configs[2] (5-layer GIN forward) at their full sizes, in
    the same process as the default run, knobs by the library's rules, fewer timed steps; each with its parity figure from the
    same run (the large share on sampled rows as a sub-problem of their own, the GIN forward whole).  -> ({"big": ..., "gin":
    ...}, parity checks)"""
    import copy
    out, checks = {}, []
    a = copy.copy(args)
    a.no_tune, a.no_compact, a.big_scale = True, True, 0
    a.steps, a.warmup = max(3, min(args.steps, 10)), 3
    host.release_cached()
    t0 = time.perf_counter()
    r = bench_big(a, torch, host)
    rf = r["roofline"]
    out["big"] = {"workload": r["config"]["workload"], "ms": r["detail"]["stage_ms"]["agg"], "update_ms": r["detail"]["stage_ms"]["update"],
                  "algorithmic_bytes": rf["algorithmic_bytes"], "achieved": rf["achieved"], "frac": rf["frac"], "traffic": rf.get("traffic"),
                  "traffic_measured_at": rf.get("traffic_measured_at"), "update_gbps": r["detail"]["update_gbps"],
                  "update_tflops": r["detail"]["update_tflops"], "steps": a.steps, "parity": r["parity"], "cpu_baseline": r["cpu_baseline"],
                  "leg_wall_s": round(time.perf_counter() - t0, 1)}
    checks += r["_checks"]
    host.release_cached()
    torch.cuda.empty_cache()
    a.warmup = 10
    t0 = time.perf_counter()
    r = bench_gin(a, torch, host)
    rf = r["roofline"]
    agg_ms = rf["avg_launch_ms"]
    out["gin"] = {"workload": r["config"]["workload"], "fwd_ms": r["value"], "agg_ms": agg_ms, "mlp_total_ms": r["detail"]["mlp_total_ms"],
                  "algorithmic_bytes": rf["algorithmic_bytes"], "algorithmic_gbps_over_hbm_peak": rf.get("algorithmic_gbps_over_hbm_peak"),
                  "traffic": rf.get("traffic"), "traffic_measured_at": rf.get("traffic_measured_at"),
                  "frac_traffic": round(rf["traffic"] / (agg_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4) if rf.get("traffic") else None,
                  "steps": a.steps, "parity": r["parity"], "cpu_baseline": r["cpu_baseline"], "leg_wall_s": round(time.perf_counter() - t0, 1)}
    checks += r["_checks"]
    host.release_cached()
    torch.cuda.empty_cache()
    return out, checks


def gcn2_headline_only(args, torch, host, forward_stages, names):
    """--only-headline: the timed forward of the default run and nothing around it (no literal-knob / rule / search /
    share / CPU legs), so that a profiler run sees one setting per kernel."""
    k = (args.ps, args.wpb, args.dist, args.col_block_rows, args.core_rows)
    stages = forward_stages(k, k)
    r = time_steps(torch, stages, names, args.steps, args.warmup)
    return {"metric": "gcn_2layer_fwd_ms", "value": round(r["event_median_ms"], 4), "unit": "ms", "n_gpus": 1, "steps": args.steps,
            "warmup": args.warmup, "ms_per_step": round(r["wall_ms"], 4), "higher_is_better": False, "scaling": "weak", "vs_baseline": None,
            "dtype": "f32", "data": "synthetic",
            "config": {"workload": "configs[1], the headline forward only; last aggregation: %s" % host.last_agg_kernel()},
            "detail": {"stage_ms": {n: round(v, 4) for n, v in r["stage_median"].items()}}}


def paired_tables(torch, local, remote):
    """The local and the remote feature table of an aggregation call as views into ONE device allocation (the remote table
    256-byte aligned behind the local one).  How the library forms gather addresses -- 32-bit buffer offsets when both
    tables lie inside one window of under 2 GiB, 64-bit addresses otherwise -- then follows from the table sizes and not
    from where the allocator put two separate blocks: the same kernel variant in every run, under the profiler too.
    `local` / `remote`: host arrays or device tensors.  -> (d_local, d_remote, block)"""
    as_dev = lambda a: a if torch.is_tensor(a) else torch.from_numpy(np.ascontiguousarray(a))
    local, remote = as_dev(local), as_dev(remote)
    nl = local.numel() * local.element_size()
    first = (nl + 255) & ~255
    block = torch.empty(first + remote.numel() * remote.element_size(), dtype=torch.uint8, device="cuda")
    d_l = block[:nl].view(local.dtype).view(local.shape)
    d_r = block[first:].view(remote.dtype).view(remote.shape)
    d_l.copy_(local)
    d_r.copy_(remote)
    return d_l, d_r, block


def share_inputs(args, torch, host):
    """Rank 0's share of an 8-way partitioned RMAT graph (ids scrambled) with the remote rows pre-staged: host arrays,
    device tensors and the compactly staged remote table (one row per distinct remote id, most referenced first)."""
    scale, V, draws, dim, num_gpus = 22, 4_194_304, 52_000_000 * args.share_density, 16, 8
    npp, lb, ub = host.range_partition(V, num_gpus, 0)
    t0 = time.time()
    ptr, col = host.gen_rmat(scale, V, draws, seed=7, scramble=True, row_lo=lb, row_hi=ub)
    lp, rp, lc, rc = host.split_CSR(np.concatenate([np.zeros(lb, np.int32), ptr]) if lb else ptr, col, lb, ub)
    R, nnz = ub - lb, len(col)
    log("share: rows=%d nnz=%d local=%d remote=%d in %.1fs" % (R, nnz, len(lc), len(rc), time.time() - t0))
    dev = "cuda"
    x_remote = host.fill_normal((num_gpus * npp, dim), seed=11)
    sh = dict(V=V, dim=dim, npp=npp, lb=lb, ub=ub, R=R, nnz=nnz, lp=lp, rp=rp, lc=lc, rc=rc, x_remote=x_remote)
    sh["d_xl"], sh["d_xr"], sh["tables"] = paired_tables(torch, x_remote[lb:ub], x_remote)  # the local rows are a table of their own
    sh["d"] = [torch.from_numpy(a).to(dev) if len(a) else torch.zeros(1, dtype=torch.int32, device=dev) for a in (lp, lc, rp, rc)]
    sh["d_out"] = torch.empty(R, dim, device=dev)
    return sh


def share_record(args, torch, host, with_cpu):
    """configs[3] timed two ways: the remote table indexed by global id (the reference's addressing: row u of PE
    u / nodesPerPE) and staged compactly (what a pre-exchange of the remote rows delivers).  Same sums, same algorithmic
    bytes.  The compact staging is the setting a multi-GPU run would use and is the headline of this record; the
    global-id figure stands beside it.  Each result is checked against the CPU oracle."""
    sh = share_inputs(args, torch, host)
    d, d_out, d_xl, d_xr = sh["d"], sh["d_out"], sh["d_xl"], sh["d_xr"]
    lb, ub, dim, npp, R, nnz = sh["lb"], sh["ub"], sh["dim"], sh["npp"], sh["R"], sh["nnz"]
    nbytes = agg_bytes(nnz, R, dim, ptr_arrays=2)

    def cold_leg(kn, col_r, xl, table, want):
        """The same call with nothing of it left in the caches: each launch goes to the next of COLD_COPIES disjoint
        copies of everything the call touches (row pointers, column ids, both feature tables, the output, and -- a plan
        is keyed by its CSR's addresses -- its own descriptors and row offsets), so between two uses of a copy the others
        move several times the 256 MB of the last-level cache.  HIP events around each launch only; the mean over all."""
        n = COLD_COPIES
        sets = []
        for _ in range(n):
            c = [t.clone() for t in (d[0], d[1], d[2], col_r)]
            c += list(paired_tables(torch, xl, table)[:2])
            c.append(torch.empty_like(d_out))
            sets.append(c)
        calls = [lambda c=c: host.mgg_SAG_np_div(c[6], c[4], c[0], c[1], c[2], c[3], lb, ub, dim, npp, 0, kn.ps, kn.wpb, kn.dist,
                                                 input_remote=c[5], col_block_rows=kn.blk, core_rows=kn.core) for c in sets]
        mark = host.cache_stats()["plan_bytes"]
        calls[0]()
        plan_bytes = host.cache_stats()["plan_bytes"] - mark
        for fn in calls:   # plans built, code loaded
            fn()
            fn()
        torch.cuda.synchronize()
        ev = [[(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(n)] for _ in range(args.steps)]
        for step in ev:
            for (e0, e1), fn in zip(step, calls):
                e0.record()
                fn()
                e1.record()
        torch.cuda.synchronize()
        ms = [e0.elapsed_time(e1) for step in ev for e0, e1 in step]
        slowest = sorted(range(len(ms)), key=lambda i: -ms[i])[:4]
        same = all(bool((c[6] == sets[0][6]).all()) for c in sets) and bool(np.array_equal(sets[0][6].cpu().numpy(), want))
        per_copy = sum(t.numel() * t.element_size() for t in sets[0]) + plan_bytes
        # the median launch: with events around single launches a stall of the launching thread (the stream runs empty
        # between the first event and the kernel) lands inside one interval; the mean is given beside it
        mean, med = float(np.mean(ms)), float(np.median(ms))
        out = {"copies": n, "launches": len(ms), "avg_launch_ms": round(mean, 4), "median_launch_ms": round(med, 4),
               "achieved": round(nbytes / (med * 1e-3) / 1e9, 1), "frac": round(nbytes / (med * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4),
               "frac_by_mean_launch": round(nbytes / (mean * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4),
               "bytes_allocated_per_copy": int(per_copy), "bytes_of_other_copies_between_two_uses": int(per_copy * (n - 1)),
               "results_identical_to_the_warm_call": same,
               "slowest_launches": [{"step": i // n, "copy": i % n, "ms": round(ms[i], 4)} for i in slowest]}
        for c in sets:
            for t in c[:4]:
                host.forget(t)
        del sets, calls
        return out

    def measure(col_r, xl, table, key):
        search = lambda ps, blk, core: host.tune_np_div(d_out, xl, d[0], d[1], d[2], col_r, lb, ub, dim, npp, ps, input_remote=table,
                                                        col_block_rows=blk, core_rows=core)

        def timed(kn):
            call = lambda: host.mgg_SAG_np_div(d_out, xl, d[0], d[1], d[2], col_r, lb, ub, dim, npp, 0, kn.ps, kn.wpb, kn.dist, input_remote=table,
                                               col_block_rows=kn.blk, core_rows=kn.core)
            kn.observe(host, call)
            r = time_steps(torch, [call], ["agg"], args.steps, args.warmup)
            return call, r["stage_avg"]["agg"], r["stage_median"]["agg"]

        kn = Knobs(args, search if args.tune else None)
        call, ms, med = timed(kn)
        gbps = nbytes / (ms * 1e-3) / 1e9
        rec = {"avg_launch_ms": round(ms, 4), "median_launch_ms": round(med, 4), "achieved": round(gbps, 1),
               "frac": round(gbps / HBM_PEAK_GBPS, 4), "knobs": str(kn) + (" (searched)" if args.tune else " (library rules, no search)"),
               "kernel": host.last_agg_kernel().split(" grid")[0] + (" (%s gather addressing)" % re.search(r"addr=(\w+)", host.last_agg_kernel()).group(1)),
               **load_traffic(key, args, kn.blk, kn.core)}
        call()
        torch.cuda.synchronize()
        result = d_out.cpu().numpy()
        rec["cold"] = cold_leg(kn, col_r, xl, table, result)
        rec["frac_cold"] = rec["cold"]["frac"]
        if not args.tune and not args.no_search:
            t0 = time.perf_counter()
            ks = Knobs(args, search)
            torch.cuda.synchronize()
            search_ms = (time.perf_counter() - t0) * 1e3
            _, ms_s, _ = timed(ks)
            rec["searched"] = {"avg_launch_ms": round(ms_s, 4), "knobs": str(ks), "search_wall_ms": round(search_ms, 2),
                               "frac": round(nbytes / (ms_s * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4), "rules_over_searched": round(ms / ms_s, 4)}
        return rec, result

    glob, out_glob = measure(d[3], d_xl, d_xr, "share_agg")
    # compact staging: distinct remote ids most referenced first, column array rewritten, rows gathered into a small table
    host.compact_remote_device(d[3], len(sh["rc"]))  # first use: scratch allocation
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    d_rcc, d_ids = host.compact_remote_device(d[3], len(sh["rc"]))
    torch.cuda.synchronize()
    compaction_ms = (time.perf_counter() - t0) * 1e3
    d_xl2, d_xc, _block = paired_tables(torch, d_xl, torch.empty(len(d_ids), dim, device="cuda", dtype=d_xr.dtype))
    stage = lambda: host.gather_rows(d_xc, d_xr, d_ids, len(d_ids), dim * 4)
    rs = time_steps(torch, [stage], ["stage"], args.steps, 2)
    comp, out_comp = measure(d_rcc, d_xl2, d_xc, "share_agg_compact")
    comp.update({"distinct_remote_rows": int(len(d_ids)), "table_bytes": int(len(d_ids)) * dim * 4,
                 "setup_ms": {"compaction_on_gpu_once_per_graph": round(compaction_ms, 2),
                              "staging_gather_per_layer": round(rs["stage_median"]["stage"], 4)},
                 "max_abs_diff_vs_global_id_table": float(np.abs(out_comp - out_glob).max())})
    checks = []
    cpu = None
    parity = None
    if with_cpu:
        from oracle import orc
        th = orc.max_threads()
        x_remote = sh["x_remote"]
        t0 = time.perf_counter()
        ref = orc.sag_np_div(x_remote[lb:ub], x_remote, sh["lp"], sh["lc"], sh["rp"], sh["rc"], lb, ub, dim, npp, f64=False, threads=th)
        cpu_s = time.perf_counter() - t0
        ref64 = orc.sag_np_div(x_remote[lb:ub], x_remote, sh["lp"], sh["lc"], sh["rp"], sh["rc"], lb, ub, dim, npp, f64=True, threads=th)
        mag = orc.sag_np_div_rows(np.arange(R, dtype=np.int32), x_remote[lb:ub], x_remote, sh["lp"], sh["lc"], sh["rp"], sh["rc"], lb, ub, dim,
                                  npp, abs_sum=True, threads=th)
        e1 = float(np.max(np.abs(out_glob - ref64) / (mag + 1e-30)))
        e2 = float(np.max(np.abs(out_comp - ref64) / (mag + 1e-30)))
        parity = {"max_err_over_abs_sum": max(e1, e2), "tolerance": 1e-5, "global_id_table": e1, "compact_staging": e2,
                  "against": "the CPU oracle in double precision, whole share, every element"}
        cpu = {"value": round(cpu_s * 1e3, 1), "unit": "ms", "cores": th, "kind": "port", "sample": "the same aggregation call, whole share (fp32, OpenMP over rows)",
               "max_abs_diff_vs_gpu": float(np.abs(out_glob - ref).max())}
        checks = [("share, global-id table", e1, 1e-5), ("share, compact staging", e2, 1e-5)]
    for rec_, name in ((glob, "global-id table"), (comp, "compact staging")):
        checks.append(("share, %s: cold-cache copies differ from the warm call" % name, 0.0 if rec_["cold"]["results_identical_to_the_warm_call"] else 1.0, 0.5))
    workload = ("configs[3]: rank-0 1/8 share of RMAT V=%d (ids scrambled), rows=%d nnz=%d (local %d, remote %d), fp32 dim %d, remote rows "
                "pre-staged in a second HBM table" % (sh["V"], R, nnz, len(sh["lc"]), len(sh["rc"]), dim))
    roofline = {"bound": "hbm", "kernel": "%s on %s, remote rows staged compactly (%s)" % (comp["kernel"], "configs[3]", comp["knobs"]),
                "achieved": comp["achieved"], "peak": HBM_PEAK_GBPS, "unit": "GB/s", "frac": comp["frac"], "traffic": comp.get("traffic"),
                "algorithmic_bytes": nbytes, "avg_launch_ms": comp["avg_launch_ms"],
                "frac_cold": comp["frac_cold"], "median_launch_ms_cold": comp["cold"]["median_launch_ms"], "avg_launch_ms_cold": comp["cold"]["avg_launch_ms"],
                "cold_is": "every launch on the next of %d disjoint copies of all arrays of the call (%.0f MB of other copies between two uses of "
                           "one; the last-level cache holds 256 MB)" % (COLD_COPIES, comp["cold"]["bytes_of_other_copies_between_two_uses"] / 1e6),
                "frac_global_id_table": glob["frac"], "frac_cold_global_id_table": glob["frac_cold"],
                "achieved_global_id_table": glob["achieved"], "traffic_global_id_table": glob.get("traffic")}
    if comp.get("traffic_measured_at"):
        roofline["traffic_measured_at"] = comp["traffic_measured_at"]
    return {"workload": workload, "ms": comp["avg_launch_ms"], "algorithmic_bytes": nbytes, "frac": comp["frac"], "traffic": comp.get("traffic"),
            "compact_staging": comp, "global_id_table": glob, "cpu_baseline": cpu, "parity": parity, "roofline": roofline, "_checks": checks}


def bench_share(args, torch, host):
    """Aggregation alone on rank 0's share of an 8-way partitioned RMAT graph, remote rows pre-staged."""
    share = share_record(args, torch, host, with_cpu=not args.no_cpu)
    checks = share.pop("_checks")
    roofline = share.pop("roofline")
    res = {
        "metric": "np_aggregation_ms", "value": share["compact_staging"]["median_launch_ms"], "unit": "ms", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": share["ms"], "higher_is_better": False, "scaling": "weak",
        "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"workload": share["workload"] + "; value = compact staging, median over the timed steps"},
        "roofline": roofline, "cpu_baseline": share["cpu_baseline"], "parity": share["parity"], "detail": share,
    }
    fail_on_parity(res, checks)
    return res


def compact_variant(args, torch, host, d_out, d_xl, d_xr, d, rc, lb, ub, dim, npp, nbytes, esize):
    """The same aggregation with the remote rows staged compactly: one row per distinct remote id, most referenced
    first, remote_col rewritten to match (what a pre-exchange of remote rows would deliver).  Reported beside the
    table indexed by global id (the reference's addressing); same algorithmic bytes."""
    dev = d_out.device
    host.compact_remote_device(d[3], len(rc))  # first use: scratch allocation
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    d_rcc, d_ids = host.compact_remote_device(d[3], len(rc))
    prep_s = time.perf_counter() - t0
    ids = d_ids
    d_xc = torch.empty(len(ids), dim, device=dev, dtype=d_xr.dtype)
    stage = lambda: host.gather_rows(d_xc, d_xr, d_ids, len(ids), dim * esize)
    stage()
    want = d_out.clone()  # produced from the global-id table by the caller
    kn = Knobs(args, None if args.no_tune else lambda ps, blk, core: host.tune_np_div(d_out, d_xl, d[0], d[1], d[2], d_rcc, lb, ub, dim, npp, ps,
                                                                                         input_remote=d_xc, col_block_rows=blk, core_rows=core))
    call = lambda: host.mgg_SAG_np_div(d_out, d_xl, d[0], d[1], d[2], d_rcc, lb, ub, dim, npp, 0, kn.ps, kn.wpb, kn.dist,
                                       input_remote=d_xc, col_block_rows=kn.blk, core_rows=kn.core)
    for _ in range(args.warmup):
        call()
    timer = StageTimer(torch, ["agg", "stage"], args.steps)
    for _ in range(args.steps):
        timer.step([call, stage])
    avg = timer.averages()
    gbps = nbytes / (avg["agg"] * 1e-3) / 1e9
    return {"distinct_remote_rows": int(len(ids)), "table_bytes": int(len(ids)) * dim * esize, "agg_ms": round(avg["agg"], 4),
            "achieved_gbps": round(gbps, 1), "frac_of_hbm_peak": round(gbps / HBM_PEAK_GBPS, 4), "knobs": str(kn),
            "staging_gather_ms": round(avg["stage"], 4), "compaction_on_gpu_ms": round(prep_s * 1e3, 2),
            "max_abs_diff_vs_global_id_table": float((d_out - want).abs().max())}


def bench_gin(args, torch, host):
    """5-layer GIN forward on the whole graph: dense(100->64); 5 x [GIN aggregate (1+eps) x_v + sum, eps = 0,
    then a 2-layer MLP 64->64->64 with ReLU between, the last MLP ending at 47 classes]; softmax.  (The reference's main
    has one dense per GIN layer and eps = 0.5; the benchmark configuration asks for the 2-layer MLP and eps = 0.)"""
    V, scale, draws = 2_450_000, 22, 64_000_000
    in_dim, hidden, out_dim, L, eps = 100, 64, 47, 5, 0.0
    ps = args.ps
    if args.small:
        V, scale, draws = 50_000, 16, 1_300_000
    t0 = time.time()
    ptr, col = host.gen_rmat(scale, V, draws, seed=3)
    nnz = int(len(col))
    log("graph: V=%d nnz=%d in %.1fs" % (V, nnz, time.time() - t0))
    X = host.fill_normal((V, in_dim), seed=1)
    W0 = host.glorot(in_dim, hidden, seed=2)
    Wa = [host.glorot(hidden, hidden, seed=10 + l) * 0.2 for l in range(L)]
    Wb = [host.glorot(hidden, out_dim if l == L - 1 else hidden, seed=30 + l) * 0.2 for l in range(L)]
    dev = "cuda"
    d_ptr, d_col = torch.from_numpy(ptr).to(dev), torch.from_numpy(col).to(dev)
    zp, zc = torch.zeros(V + 1, dtype=torch.int32, device=dev), torch.zeros(1, dtype=torch.int32, device=dev)
    d_X, d_W0 = torch.from_numpy(X).to(dev), torch.from_numpy(W0).to(dev)
    d_Wa = [torch.from_numpy(w).to(dev) for w in Wa]
    ldo = (out_dim + 3) & ~3
    d_Wb = [torch.from_numpy(w).to(dev) for w in Wb]
    d_Y = torch.empty(V, hidden, device=dev)
    d_H = torch.empty(V, hidden, device=dev)
    d_T = torch.empty(V, hidden, device=dev)
    d_logits = torch.empty(V, out_dim, device=dev)
    d_P = torch.empty(V, out_dim, device=dev)

    d_Y.zero_()
    kn = Knobs(args, None if args.no_tune else lambda ps, blk, core: host.tune_np_div(d_H, d_Y, d_ptr, d_col, zp, zc, 0, V, hidden, V, ps, gin_eps=eps,
                                                                                         col_block_rows=blk, core_rows=core))
    stages, names = [lambda: host.dense_forward(d_Y, d_X, d_W0, V, in_dim, hidden)], ["dense0"]
    for l in range(L):
        last = l == L - 1
        stages.append(lambda: host.mgg_GIN_np_div(d_H, d_Y, d_ptr, d_col, zp, zc, 0, V, hidden, V, 0, kn.ps, kn.wpb, kn.dist, eps,
                                                  col_block_rows=kn.blk, core_rows=kn.core))
        if args.unfused_mlp:
            stages.append(lambda l=l: host.dense_forward(d_T, d_H, d_Wa[l], V, hidden, hidden, relu=True))
            if last:
                stages.append(lambda l=l: host.dense_forward(d_logits, d_T, d_Wb[l], V, hidden, out_dim))
            else:
                stages.append(lambda l=l: host.dense_forward(d_Y, d_T, d_Wb[l], V, hidden, hidden))
            names += ["agg%d" % l, "mlp%da" % l, "mlp%db" % l]
        else:  # both updates of the MLP in one pass; the 64-wide intermediate stays in registers, and the last one ends in
            # the row softmax: the logits never make a round trip through memory
            stages.append(lambda l=l, o=(d_P if last else d_Y), w=(out_dim if last else hidden), last=last:
                          host.mlp2_forward(o, d_H, d_Wa[l], d_Wb[l], V, hidden, hidden, w, relu_mid=True, softmax_out=last))
            names += ["agg%d" % l, "mlp%d" % l]
    if args.unfused_mlp:
        stages.append(lambda: host.softmax_forward(d_P, d_logits, V, out_dim))
        names.append("softmax")
    kn.observe(host, stages[1])  # what the library chose where the knobs were left to it

    for _ in range(args.warmup):
        for fn in stages:
            fn()
    torch.cuda.synchronize()
    timer = StageTimer(torch, names)
    t0 = time.perf_counter()
    for _ in range(args.steps):
        timer.step(stages)
    torch.cuda.synchronize()
    wall_ms = (time.perf_counter() - t0) * 1e3 / args.steps
    avg = timer.averages()
    agg_ms = sum(avg["agg%d" % l] for l in range(L)) / L
    mlp_ms = sum(v for k, v in avg.items() if k.startswith("mlp"))
    log("ms: agg avg %.4f, all MLPs %.4f, dense0 %.4f, softmax %s, wall %.4f" %
        (agg_ms, mlp_ms, avg["dense0"], "%.4f" % avg["softmax"] if "softmax" in avg else "inside the last MLP", wall_ms))
    nbytes = agg_bytes(nnz, V, hidden, gin=True)
    achieved = nbytes / (agg_ms * 1e-3) / 1e9

    cpu = None
    parity = None
    if not args.no_cpu:
        from oracle import orc
        th = orc.max_threads()
        t0 = time.perf_counter()
        Y = orc.dense(X, W0, f64=False, threads=th)
        for l in range(L):
            H = orc.sag_np_div(Y, Y, ptr, col, None, None, 0, V, hidden, V, flags=orc.GIN, eps=eps, f64=False, threads=th)
            T = np.maximum(orc.dense(H, Wa[l], f64=False, threads=th), 0)
            Y = orc.dense(T, Wb[l], f64=False, threads=th)
        P_ref = orc.softmax_rows(Y, threads=th)
        cpu_s = time.perf_counter() - t0
        cpu = {"value": round(cpu_s * 1e3, 1), "unit": "ms", "cores": th, "kind": "port",
               "sample": "1 full forward of the same workload (OpenMP over rows, fp32)"}
        if not args.unfused_mlp:  # the timed forward does not write the logits: one more call of the last update without the softmax
            host.mlp2_forward(d_logits, d_H, d_Wa[L - 1], d_Wb[L - 1], V, hidden, hidden, out_dim, relu_mid=True)
            torch.cuda.synchronize()
        lg = d_logits.cpu().numpy()
        parity = {"logits_max_rel_err": float(np.abs(lg - Y).max() / np.abs(Y).max()),
                  "softmax_max_abs_err": float(np.abs(d_P.cpu().numpy() - P_ref).max())}
        log("cpu forward %.1f ms on %d threads; parity %s" % (cpu_s * 1e3, th, parity))
    return {
        "metric": "gin_5layer_fwd_ms", "value": round(wall_ms, 4), "unit": "ms", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(wall_ms, 4), "higher_is_better": False, "scaling": "weak",
        "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"workload": "configs[2]: 5-layer GIN forward, RMAT V=%d nnz=%d, 100->64->47, 2-layer MLP per layer (%s), eps=0, "
                               "%s" % (V, nnz, "two kernels" if args.unfused_mlp else "one fused kernel, the last one with the softmax inside", kn)},
        "roofline": hbm_roofline("%sk_agg (GIN, dim 64)" % ("k_core_sell + " if kn.core > 0 else ""), nbytes, agg_ms,
                                 load_traffic("gin_agg", args, kn.blk, kn.core)),
        "cpu_baseline": cpu, "parity": parity,
        "detail": {"stage_ms": {k: round(v, 4) for k, v in avg.items()}, "mlp_total_ms": round(mlp_ms, 4)},
        "_checks": [("configs[2] logits, relative", parity["logits_max_rel_err"], 1e-5),
                    ("configs[2] softmax", parity["softmax_max_abs_err"], 1e-5)] if parity else [],
    }


def bench_big(args, torch, host):
    """large-share stress.  One rank's 1/8 share of a 111 M-node RMAT graph (ids scrambled): ~13.9 M rows,
    ~200 M neighbors, bf16 width-128 tables (local + a separate remote table indexed by global id), fp32 accumulation,
    then the 128x128 update on the bf16 matrix cores.  --big-scale shrinks every size by 2^k for a quicker run."""
    k = args.big_scale
    scale, V, draws, dim, num_gpus = 27 - k, 111_000_000 >> k, 790_000_000 >> k, 128, 8
    ps = args.ps
    npp, lb, ub = host.range_partition(V, num_gpus, 0)
    t0 = time.time()
    ptr, col = host.gen_rmat(scale, V, draws, seed=5, scramble=True, row_lo=lb, row_hi=ub)
    lp, rp, lc, rc = host.split_CSR(ptr, col, lb, ub)
    R, nnz = ub - lb, len(col)
    log("share: rows=%d nnz=%d local=%d remote=%d in %.1fs" % (R, nnz, len(lc), len(rc), time.time() - t0))
    dev = "cuda"
    gen = torch.Generator(device=dev)
    gen.manual_seed(5)
    d_xr = torch.randn(num_gpus * npp, dim, device=dev, dtype=torch.bfloat16, generator=gen)
    d_xl = d_xr[lb:ub].clone()
    d = [torch.from_numpy(a).to(dev) if len(a) else torch.zeros(1, dtype=torch.int32, device=dev) for a in (lp, lc, rp, rc)]
    d_out = torch.empty(R, dim, device=dev)
    W = host.glorot(dim, dim, seed=6)
    d_W = torch.from_numpy(W).to(dev).to(torch.bfloat16)
    d_next = torch.empty(R, dim, device=dev, dtype=torch.bfloat16)
    kn = Knobs(args, None if args.no_tune else lambda ps, blk, core: host.tune_np_div(d_out, d_xl, d[0], d[1], d[2], d[3], lb, ub, dim, npp, ps,
                                                                                         input_remote=d_xr, col_block_rows=blk, core_rows=core))
    stages = [
        lambda: host.mgg_SAG_np_div(d_out, d_xl, d[0], d[1], d[2], d[3], lb, ub, dim, npp, 0, kn.ps, kn.wpb, kn.dist, input_remote=d_xr,
                                    col_block_rows=kn.blk, core_rows=kn.core),
        lambda: host.dense_forward_bf16(d_next, d_out, d_W, R, dim, dim),
    ]
    for _ in range(args.warmup):
        for fn in stages:
            fn()
    torch.cuda.synchronize()
    timer = StageTimer(torch, ["agg", "update"])
    t0 = time.perf_counter()
    for _ in range(args.steps):
        timer.step(stages)
    torch.cuda.synchronize()
    wall_ms = (time.perf_counter() - t0) * 1e3 / args.steps
    avg = timer.averages()
    nbytes = agg_bytes(nnz, R, dim, s_in=2, ptr_arrays=2)
    achieved = nbytes / (avg["agg"] * 1e-3) / 1e9
    gflop = 2.0 * R * dim * dim / 1e9
    gemm_bytes = R * dim * 4 + R * dim * 2 + dim * dim * 2
    parity = None
    cpu = None
    if not args.no_cpu:
        from oracle import orc
        th = orc.max_threads()
        deg = np.diff(lp) + np.diff(rp)
        rng = np.random.default_rng(0)
        rows = np.unique(np.concatenate([np.argsort(deg)[-20:], rng.integers(0, R, 2000)])).astype(np.int32)
        # The sampled rows as a small problem of their own: a compact table with just the feature rows they touch
        # (the local table holds the same values as rows lb..ub of the global one), ids renumbered into it.
        nbrs = [np.concatenate([lc[lp[r]:lp[r + 1]], rc[rp[r]:rp[r + 1]]]) for r in rows]
        need = np.unique(np.concatenate(nbrs))
        x_small = d_xr[torch.from_numpy(need.astype(np.int64)).to(dev)].float().cpu().numpy()
        sp = np.zeros(len(rows) + 1, np.int32)
        sp[1:] = np.cumsum([len(x) for x in nbrs])
        cc = np.searchsorted(need, np.concatenate(nbrs)).astype(np.int32)
        zp_ = np.zeros(len(rows) + 1, np.int32)
        n_small = len(rows)
        dummy_local = np.zeros((n_small, dim), np.float32)
        t0 = time.perf_counter()
        want = orc.sag_np_div(dummy_local, x_small, zp_, np.zeros(0, np.int32), sp, cc, 0, n_small, dim, n_small, f64=True, threads=th)
        cpu_s = time.perf_counter() - t0
        mag = orc.sag_np_div_rows(np.arange(n_small, dtype=np.int32), dummy_local, x_small, zp_, np.zeros(0, np.int32), sp, cc, 0,
                                  n_small, dim, n_small, abs_sum=True, threads=th)
        got = d_out[torch.from_numpy(rows.astype(np.int64)).to(dev)].cpu().numpy()
        err = float(np.max(np.abs(got - want) / (mag + 1e-30)))
        parity = {"rows_checked": int(len(rows)), "agg_max_err_over_abs_sum": err}
        edges = int(sp[-1])
        cpu = {"value": round(edges / cpu_s / 1e6, 2), "unit": "M edges/s", "cores": th, "kind": "port",
               "sample": "%d sampled rows (%d neighbors) of the same share, double accumulation" % (len(rows), edges),
               "gpu_same_unit": round(nnz / (avg["agg"] * 1e-3) / 1e6, 1)}
        log("parity %s; cpu %s" % (parity, cpu))
    compact = None if getattr(args, "no_compact", False) else compact_variant(args, torch, host, d_out, d_xl, d_xr, d, rc, lb, ub, dim, npp, nbytes, 2)
    return {
        "metric": "np_aggregation_plus_update_ms", "value": round(wall_ms, 4), "unit": "ms", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(wall_ms, 4), "higher_is_better": False, "scaling": "weak",
        "vs_baseline": None, "dtype": "bf16", "data": "synthetic",
        "config": {"workload": "configs[4] / 2^%d: rank-0 1/8 share of RMAT V=%d (scrambled), rows=%d nnz=%d (local %d, remote %d), "
                               "bf16 dim %d, fp32 accumulate, then %dx%d bf16 MFMA update; %s"
                               % (k, V, R, nnz, len(lc), len(rc), dim, dim, dim, kn)},
        "roofline": hbm_roofline("k_agg (bf16 dim 128, local+remote)", nbytes, avg["agg"], load_traffic("big_agg", args, kn.blk, kn.core)),
        "cpu_baseline": cpu, "parity": parity,
        "detail": {"stage_ms": {k2: round(v, 4) for k2, v in avg.items()},
                   "update_tflops": round(gflop / avg["update"], 2), "update_gbps": round(gemm_bytes / (avg["update"] * 1e-3) / 1e9, 1),
                   "compact_remote_staging": compact},
        "_checks": [("configs[4] sampled rows", parity["agg_max_err_over_abs_sum"], 1e-5)] if parity else [],
    }


def bench_vendor(args, torch, host):
    """The library's kernels beside the vendor libraries torch dispatches to (GEMM behind torch.mm, CSR x dense SpMM
    behind torch.sparse.mm) on the benchmark shapes.  A yardstick, not a target; nothing of torch's is on the product path."""
    def timeit(fn, it):
        fn(); fn()
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(it):
            fn()
        e1.record()
        torch.cuda.synchronize()
        return e0.elapsed_time(e1) / it

    rows = []
    for n, d1, d2 in ((233_000, 602, 16), (233_000, 16, 41), (2_450_000, 100, 64), (2_450_000, 64, 64)):
        x, w = torch.randn(n, d1, device="cuda"), torch.randn(d1, d2, device="cuda")
        o = torch.empty(n, d2, device="cuda")
        rows.append({"op": "fp32 update %dx%dx%d" % (n, d1, d2),
                     "library_ms": round(timeit(lambda: host.dense_forward(o, x, w, n, d1, d2), args.steps), 4),
                     "vendor_ms": round(timeit(lambda: torch.mm(x, w, out=o), args.steps), 4)})
    n, d = 2_450_000, 64
    x, wa, wb = torch.randn(n, d, device="cuda"), torch.randn(d, d, device="cuda"), torch.randn(d, d, device="cuda")
    o, t = torch.empty(n, d, device="cuda"), torch.empty(n, d, device="cuda")

    def two():
        torch.mm(x, wa, out=t)
        torch.relu_(t)
        torch.mm(t, wb, out=o)
    rows.append({"op": "fp32 MLP 64->64->64 on %d rows (vendor: mm, relu, mm)" % n,
                 "library_ms": round(timeit(lambda: host.mlp2_forward(o, x, wa, wb, n, d, d, d), args.steps), 4),
                 "vendor_ms": round(timeit(two, args.steps), 4)})
    del x, o, t
    for name, (scale, V, draws, seed), dims in (("GCN graph", (18, 233_000, 216_000_000, 42), (16, 44)),
                                                 ("GIN graph", (22, 2_450_000, 64_000_000, 3), (64,))):
        ptr, col = host.gen_rmat(scale, V, draws, seed=seed)
        d_ptr, d_col = torch.from_numpy(ptr).cuda(), torch.from_numpy(col).cuda()
        zp, zc = torch.zeros(V + 1, dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
        A = torch.sparse_csr_tensor(d_ptr, d_col, torch.ones(len(col), device="cuda"), size=(V, V))
        for dim in dims:
            x, out = torch.randn(V, dim, device="cuda"), torch.empty(V, dim, device="cuda")
            host.tune_np_div(out, x, d_ptr, d_col, zp, zc, 0, V, dim, V, 16)
            t1 = timeit(lambda: host.mgg_SAG_np_div(out, x, d_ptr, d_col, zp, zc, 0, V, dim, V, 0, 0, 0, 0), args.steps)
            t2 = timeit(lambda: torch.sparse.mm(A, x), 3)
            ref = torch.sparse.mm(A, x)
            rows.append({"op": "aggregation, %s nnz=%d width %d" % (name, len(col), dim), "library_ms": round(t1, 4),
                         "vendor_ms": round(t2, 4), "max_diff_over_max": float((out - ref).abs().max() / ref.abs().max())})
            log(rows[-1])
        del A
    worst = min(r["vendor_ms"] / r["library_ms"] for r in rows)
    return {"metric": "vendor_time_over_library_time_min", "value": round(worst, 3), "unit": "x", "n_gpus": 1, "steps": args.steps,
            "warmup": args.warmup, "ms_per_step": None, "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
            "dtype": "f32", "data": "synthetic", "config": {"workload": "library kernels beside torch.mm / torch.sparse.mm"},
            "detail": rows}


def bench_copy(args, torch, host):
    """Plain device copy of a known size: the stream-copy ceiling, and the yardstick the profiler's FETCH_SIZE /
    WRITE_SIZE counters are scaled against.  Three ways, so the ceiling does not rest on one kernel: the library's
    grid-stride copy, its streaming variant (non-temporal loads and stores, one workgroup per 16 KiB), and the runtime's
    own device-to-device copy behind Tensor.copy_; plus a read-only and a write-only pass (what one direction sustains)."""
    nbytes = 1 << 30
    src = torch.empty(nbytes, dtype=torch.uint8, device="cuda").random_(0, 255)
    dst = torch.empty_like(src)
    variants = (("k_copy16", lambda: host.copy_bytes(dst, src, nbytes), 2), ("k_copy16_nt", lambda: host.copy_bytes_nt(dst, src, nbytes), 2),
                ("runtime_d2d_copy", lambda: dst.copy_(src), 2), ("read_only_sum", lambda: src.view(torch.int32).sum(), 1),
                ("write_only_fill", lambda: dst.fill_(7), 1))
    detail = {}
    for name, fn, passes in variants:
        for _ in range(args.warmup):
            fn()
        torch.cuda.synchronize()
        timer = StageTimer(torch, [name], args.steps)
        for _ in range(args.steps):
            timer.step([fn])
        ms = timer.medians()[name]
        detail[name] = {"ms": round(ms, 4), "gbps": round(passes * nbytes / (ms * 1e-3) / 1e9, 1),
                        "bytes_moved": passes * nbytes, "frac_of_hbm_peak": round(passes * nbytes / (ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4)}
        log(name, detail[name])
    assert bool((dst == 7).all())
    best = max(("k_copy16", "k_copy16_nt", "runtime_d2d_copy"), key=lambda k: detail[k]["gbps"])
    return {"metric": "stream_copy_gbps", "value": detail[best]["gbps"], "unit": "GB/s", "n_gpus": 1, "steps": args.steps,
            "warmup": args.warmup, "ms_per_step": detail[best]["ms"], "higher_is_better": True, "scaling": "weak",
            "vs_baseline": None, "dtype": "u8", "data": "synthetic",
            "config": {"workload": "device copy, %d bytes read + %d bytes written per launch; best of three variants: %s" % (nbytes, nbytes, best)},
            "detail": detail}


def bench_convert(args, torch, host):
    """fp32 -> bf16 conversion of the large share's 13.9 M x 128 table, nothing else: what the memory system gives the dense
    update's 2 : 1 read / write stream, by the order in which the chip walks through the arrays -- workgroups in launch order
    with 1 ... 64 consecutive pieces of 8 KB each, and persistent grids striding over everything."""
    n = (13_875_000 >> args.big_scale) * 128
    src = torch.randn(n, device="cuda")
    dst = torch.empty(n, dtype=torch.bfloat16, device="cuda")
    cases = [("launch order, %d piece%s of 8 KB per workgroup" % (c, "" if c == 1 else "s"), c, 0) for c in (1, 2, 4, 8, 16, 64)] + \
            [("persistent grid of %d workgroups striding over all pieces" % g, 1, g) for g in (2048, 8192)]
    detail = {}
    for name, per_wg, persistent in cases:
        fn = lambda: host.convert_probe(dst, src, n, per_wg, persistent)
        for _ in range(args.warmup):
            fn()
        torch.cuda.synchronize()
        timer = StageTimer(torch, [name], args.steps)
        for _ in range(args.steps):
            timer.step([fn])
        ms = timer.medians()[name]
        detail[name] = {"ms": round(ms, 4), "gbps": round(6 * n / (ms * 1e-3) / 1e9, 1), "frac_of_hbm_peak": round(6 * n / (ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4)}
        log(name, detail[name])
    want = (src[:4096].view(torch.int32) >> 16).to(torch.int16)
    assert bool((dst[:4096].view(torch.int16) == want).all()) and bool((dst[-4096:].view(torch.int16) == (src[-4096:].view(torch.int32) >> 16).to(torch.int16)).all())
    best = max(detail, key=lambda k: detail[k]["gbps"])
    return {"metric": "convert_stream_gbps", "value": detail[best]["gbps"], "unit": "GB/s", "n_gpus": 1, "steps": args.steps,
            "warmup": args.warmup, "ms_per_step": detail[best]["ms"], "higher_is_better": True, "scaling": "weak",
            "vs_baseline": None, "dtype": "f32", "data": "synthetic",
            "config": {"workload": "fp32 -> bf16 conversion of %d values (%d bytes read, %d written per launch); best: %s" % (n, 4 * n, 2 * n, best)},
            "detail": detail}


def bench_gather(args, torch, host):
    """Random row gathers from tables of the benchmark shapes, with no index stream and no reduction: what the memory
    system sustains for the access pattern of the aggregation at each table size (the ceiling for cache-resident
    tables, where HBM peak says nothing)."""
    sink = torch.empty(262144, device="cuda")
    cases = (("64 B rows, 3 MB table (one column block of the width-16 GCN table)", 49152, 64, 64),
             ("64 B rows, 15 MB table (whole width-16 GCN table)", 233_000, 64, 64),
             ("64 B rows, 269 MB table (remote table of the 1/8 share)", 4_200_000, 64, 64),
             ("176 B of 192 B rows, 3 MB table", 16384, 192, 176),
             ("176 B of 192 B rows, 9.4 MB table (one column block of the width-41 GCN table)", 49152, 192, 176),
             ("176 B of 192 B rows, 45 MB table (whole width-41 GCN table)", 233_000, 192, 176),
             ("256 B rows, 627 MB table (GIN, width 64 fp32)", 2_450_000, 256, 256),
             ("256 B rows, 4.2 GB table (large share, width 128 bf16, compact staging)", 16_500_000, 256, 256))
    table = torch.zeros(max(r * ld for _, r, ld, _ in cases), dtype=torch.uint8, device="cuda")
    n = 228_000_000
    out = []
    for name, rows, ld, rb in cases:
        for _ in range(max(1, args.warmup)):
            done = host.gather_probe(sink, table, rows, ld, rb, n)
        torch.cuda.synchronize()
        timer = StageTimer(torch, ["probe"])
        for i in range(args.steps):
            timer.step([lambda: host.gather_probe(sink, table, rows, ld, rb, n, seed=i + 2)])
        ms = timer.averages()["probe"]
        out.append({"table": name, "rows_per_s_G": round(done / (ms * 1e-3) / 1e9, 1), "ms": round(ms, 4),
                    "useful_gbps": round(done * rb / (ms * 1e-3) / 1e9, 1)})
        log(out[-1])
    return {"metric": "gather_rows_per_s_G_64B_rows_3MB_table", "value": out[0]["rows_per_s_G"], "unit": "G rows/s", "n_gpus": 1,
            "steps": args.steps, "warmup": args.warmup, "ms_per_step": out[0]["ms"], "higher_is_better": True, "scaling": "weak",
            "vs_baseline": None, "dtype": "f32", "data": "synthetic",
            "config": {"workload": "k_gather_probe: %d random row gathers per launch per table shape" % done}, "detail": out}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=20,
                    help="untimed steps before the timed ones (default 20: a dense-core plan built a moment ago runs up to 10 %% slower "
                         "for its first twenty calls)")
    ap.add_argument("--workload", default="gcn2", choices=["gcn2", "share", "gin", "big", "copy", "convert", "gather", "vendor"])
    ap.add_argument("--ps", type=int, default=16, help="partSize; 0 = let the library choose (the search then tries 16 and 32)")
    ap.add_argument("--col-block-rows", type=int, default=0, help="column-blocked partition order: 0 = library decides, -1 = off, "
                         "N = blocks of N neighbor ids")
    ap.add_argument("--core-rows", type=int, default=0, help="dense core served from LDS: 0 = the search decides, -1 = off, "
                         "N = the N highest-degree rows")
    ap.add_argument("--wpb", type=int, default=0, help="wavefronts per workgroup; 0 = let the library choose")
    ap.add_argument("--dist", type=int, default=0, help="interleaved_dist; 0 = let the library choose.  With --wpb 0 --dist 0 (the default) the "
                         "library's rules pick them")
    ap.add_argument("--tune", action="store_true", help="time the setting the library's search measures fastest instead of the one its rules and "
                         "cost model choose (gcn2 and share otherwise run the search afterwards, for comparison)")
    ap.add_argument("--no-search", action="store_true", help="gcn2 / share: skip the comparison run of the search")
    ap.add_argument("--no-extra", action="store_true", help="gcn2: skip the legs on configs[4] and configs[2] (large bf16 share, GIN forward)")
    ap.add_argument("--only-headline", action="store_true", help="gcn2: the headline forward only (for profiler runs)")
    ap.add_argument("--no-tune", action="store_true", help="gin / big: use the library's rules instead of its search")
    ap.add_argument("--share-density", type=int, default=1, help="multiplies the number of RMAT draws of --workload share")
    ap.add_argument("--small", action="store_true", help="tiny graph, for a quick functional run")
    ap.add_argument("--big-scale", type=int, default=0, help="--workload big: divide every size by 2^k")
    ap.add_argument("--unfused-mlp", action="store_true", help="--workload gin: run each MLP as two dense updates instead of the fused kernel")
    ap.add_argument("--pitch41", type=int, default=0, help="--workload gcn2: row pitch in floats of the 41-wide tables (default 48; at least 44)")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--no-plan-check", action="store_true", help="turn the library's content checks of cached plans off (default: every kernel compares "
                         "the CSR's live edge counts with its plan's)")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py: this build runs one GPU's share on one GPU; --gpus %d is not offered (no collectives, no "
              "second device are used)" % args.gpus, file=sys.stderr)
        sys.exit(2)
    import torch
    from mgg_osdi23_amd import host
    if not torch.cuda.is_available():
        print("bench.py: no GPU visible; the HIP path has no CPU fallback", file=sys.stderr)
        sys.exit(3)
    torch.cuda.set_device(0)
    host.init(0)
    host.use_torch_stream()
    if args.no_plan_check:
        host.set_plan_check(0)
    log("device:", host.device_name())
    res = {"gcn2": bench_gcn2, "share": bench_share, "gin": bench_gin, "big": bench_big, "copy": bench_copy,
           "convert": bench_convert, "gather": bench_gather, "vendor": bench_vendor}[args.workload](args, torch, host)
    checks = res.pop("_checks", None)
    if checks:
        fail_on_parity(res, checks)
    print(json.dumps(res), flush=True)


if __name__ == "__main__":
    main()
