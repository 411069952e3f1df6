"""The work that users of this framework have it do, as cases a timing program can run.

listed() names twelve cases, draw(rng) gives more of the same ranges, prepare(case, seed) makes what a program has in
hand before a pass (inputs on the GPU, weights, output buffers), run(state) is one pass through the public entry points
of mgg_osdi23_amd.host, work(case) counts what a pass cannot do without, tolerance(case) says how far two correct
implementations may lie apart.

The framework runs full-graph GNN inference: there is no backward pass in it.  The gradient of an aggregation with respect
to its input is the same call on the transposed graph, which these symmetric graphs are themselves.

Graphs are RMAT (a = 0.57, b = c = 0.19; a = b = c = 0.25 is a uniform random graph), symmetrised, without duplicates, rows
sorted, one self loop per node -- the generator of the repository's benchmark, made on the GPU here because the inputs are
made many times.
"""
import math

import torch

from mgg_osdi23_amd import host

DEV = "cuda"
_ready = False


def listed():
    return [
        # The smallest forward: a 4,096-node uniform graph of mean degree 16, 64 -> 16 -> 41 (the repository's smoke run).
        # A service that classifies one small graph per request waits for launches and host time, not for memory.
        {"name": "gcn_4k", "kind": "gcn", "n": 4096, "draws": 32_768, "a": 0.25, "d0": 64, "hidden": 16, "classes": 41, "pad": False},
        # The benchmark's GCN at its small setting: 20,000 nodes, power law, wide input features.
        {"name": "gcn_20k", "kind": "gcn", "n": 20_000, "draws": 2_000_000, "a": 0.57, "d0": 602, "hidden": 16, "classes": 41, "pad": False},
        # An ordinary sparse graph with a wide hidden layer: aggregation at 128 and 40 columns, wide dense updates.
        {"name": "gcn_wide", "kind": "gcn", "n": 170_000, "draws": 1_200_000, "a": 0.45, "d0": 128, "hidden": 128, "classes": 40, "pad": False},
        # The headline benchmark: 2-layer GCN, 233 K nodes, 228 M neighbors, 602 -> 16 -> 41, class rows padded to a pitch of 48.
        {"name": "gcn_233k", "kind": "gcn", "n": 233_000, "draws": 216_000_000, "a": 0.57, "d0": 602, "hidden": 16, "classes": 41, "pad": True},
        # The benchmark's 5-layer GIN at its small setting.
        {"name": "gin_50k", "kind": "gin", "n": 50_000, "draws": 1_300_000, "a": 0.57, "d0": 100, "hidden": 64, "classes": 47},
        # The benchmark's 5-layer GIN: 2.45 M nodes, 123 M neighbors -- the largest case.
        {"name": "gin_2450k", "kind": "gin", "n": 2_450_000, "draws": 64_000_000, "a": 0.57, "d0": 100, "hidden": 64, "classes": 47},
        # One rank's eighth of a 4.2 M-node graph, fp32 width 16, remote rows staged compactly: the aggregation of a
        # distributed run as every rank issues it once per layer.
        {"name": "share_f32", "kind": "share", "n": 4_194_304, "ranks": 8, "draws": 52_000_000, "dim": 16, "bf16": False, "compact": True},
        # One rank's eighth of a 13.9 M-node graph, bf16 width 128, remote table indexed by global id, followed by the
        # 128 x 128 bf16 update (the benchmark's large share at an eighth of its size).
        {"name": "share_bf16", "kind": "share", "n": 13_875_000, "ranks": 8, "draws": 98_750_000, "dim": 128, "bf16": True, "compact": False},
        # Explicit partition arrays (build_part's output kept by the caller), rows of 100 floats.
        {"name": "parts_100k", "kind": "parts", "n": 100_000, "draws": 2_500_000, "a": 0.57, "dim": 100, "ps": 16},
        # Whole-graph SpMM on tightly packed rows of 41 floats, as the layer classes of the C++ interface issue it.
        {"name": "spmm_300k", "kind": "spmm", "n": 300_000, "draws": 3_000_000, "a": 0.57, "dim": 41, "ps": 32},
        # Set-up of a rank's share on the GPU: local / remote split, compact staging list, partition arrays, staged rows.
        {"name": "setup_share", "kind": "setup", "n": 1_000_000, "ranks": 8, "draws": 12_000_000, "dim": 16, "ps": 16},
        # A graph that is used once: a sampler rewrites the index arrays of its subgraph in place at every step, so the
        # program calls forget() and the aggregation builds its plan anew each time.
        {"name": "fresh_100k", "kind": "fresh", "n": 100_000, "draws": 1_000_000, "a": 0.57, "dim": 64},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gcn", "gcn", "gcn", "gin", "gin", "share", "share", "parts", "spmm", "setup", "fresh"])
    a = rng.choice([0.57, 0.57, 0.45, 0.25])
    if kind == "gcn":
        n = _log_uniform(rng, 2_000, 233_000)
        degree = _log_uniform(rng, 4, max(5, min(900, n // 20)))
        return {"kind": kind, "n": n, "draws": n * degree // 2, "a": a, "d0": _log_uniform(rng, 24, 700), "hidden": rng.choice([16, 16, 32, 50, 64, 128]),
                "classes": _log_uniform(rng, 3, 120), "pad": rng.random() < 0.5}
    if kind == "gin":
        n = _log_uniform(rng, 3_000, 1_500_000)
        degree = _log_uniform(rng, 4, min(60, n // 50))
        return {"kind": kind, "n": n, "draws": n * degree // 2, "a": a, "d0": _log_uniform(rng, 24, 300), "hidden": rng.choice([16, 32, 48, 64, 64]),
                "classes": _log_uniform(rng, 3, 64)}
    if kind == "share":
        bf16 = rng.random() < 0.5
        n = _log_uniform(rng, 60_000, 4_000_000)
        return {"kind": kind, "n": n, "ranks": rng.choice([2, 4, 8]), "draws": n * _log_uniform(rng, 6, 50) // 2,
                "dim": 8 * rng.randint(1, 16) if bf16 else rng.choice([16, 16, 32, 41, 64, 100, 128]), "bf16": bf16, "compact": rng.random() < 0.5}
    if kind in ("parts", "spmm"):
        n = _log_uniform(rng, 1_500, 500_000)
        return {"kind": kind, "n": n, "draws": n * _log_uniform(rng, 4, 60) // 2, "a": a, "dim": _log_uniform(rng, 7, 256), "ps": rng.choice([4, 16, 16, 32, 64])}
    if kind == "setup":
        n = _log_uniform(rng, 40_000, 3_000_000)
        return {"kind": kind, "n": n, "ranks": rng.choice([2, 4, 8]), "draws": n * _log_uniform(rng, 6, 40) // 2, "dim": rng.choice([16, 32, 64]),
                "ps": rng.choice([4, 16, 32])}
    n = _log_uniform(rng, 3_000, 600_000)
    return {"kind": kind, "n": n, "draws": n * _log_uniform(rng, 4, 60) // 2, "a": a, "dim": rng.choice([16, 41, 64, 64, 100, 128])}


# ---- inputs

def _start():
    global _ready
    if not _ready:
        host.init(torch.cuda.current_device())
        _ready = True
    host.use_torch_stream()


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(1_000_003 * (int(seed) + 1))
    return g


def _rmat(n, draws, a, g, rows=None, scramble=False):
    """-> (ptr, col) int32 on the GPU: rows [lo, hi) (rows = (lo, hi)) or the whole symmetrised graph."""
    b = c = 0.19 if a > 0.5 else (1.0 - a) / 3.0
    scale = max(1, (n - 1).bit_length())
    relabel = torch.randperm(n, device=DEV, generator=g) if scramble else None
    keys, have = [], 0
    lo, hi = rows or (0, n)
    while have < draws:
        m = min(32_000_000, int((draws - have) * 1.3) + 1024)
        u = torch.zeros(m, dtype=torch.int32, device=DEV)
        v = torch.zeros(m, dtype=torch.int32, device=DEV)
        for _ in range(scale):
            r = torch.rand(m, device=DEV, generator=g)
            down = r >= a + b
            u = 2 * u + down
            v = 2 * v + (((r >= a) & ~down) | (r >= a + b + c))
        ok = (u < n) & (v < n)
        u, v = u[ok][: draws - have].long(), v[ok][: draws - have].long()
        have += u.numel()
        if relabel is not None:
            u, v = relabel[u], relabel[v]
        for s, t in ((u, v), (v, u)):
            if rows:
                mine = (s >= lo) & (s < hi)
                s, t = s[mine], t[mine]
            keys.append((s - lo) * n + t)
    i = torch.arange(lo, hi, device=DEV)
    keys.append((i - lo) * n + i)
    key = torch.unique(torch.cat(keys))  # sorted
    del keys
    row = torch.div(key, n, rounding_mode="floor")
    ptr = torch.zeros(hi - lo + 1, dtype=torch.int32, device=DEV)
    ptr[1:] = torch.bincount(row, minlength=hi - lo).cumsum(0)
    return ptr, (key - row * n).int()


def _normal(g, *shape):
    return torch.randn(*shape, device=DEV, generator=g)


def _glorot(g, d1, d2):
    lim = math.sqrt(6.0 / (d1 + d2))
    return torch.rand(d1, d2, device=DEV, generator=g) * (2 * lim) - lim


def _no_remote(n):
    return torch.zeros(n + 1, dtype=torch.int32, device=DEV), torch.zeros(1, dtype=torch.int32, device=DEV)


def _side_by_side(local, remote):
    """The two feature tables of a share out of one allocation, the remote one 256-byte aligned behind the local one."""
    nl = local.numel() * local.element_size()
    first = (nl + 255) & ~255
    block = torch.empty(first + remote.numel() * remote.element_size(), dtype=torch.uint8, device=DEV)
    a = block[:nl].view(local.dtype).view(local.shape)
    b = block[first:].view(remote.dtype).view(remote.shape)
    a.copy_(local)
    b.copy_(remote)
    return a, b


def prepare(case, seed):
    _start()
    g = _gen(seed)
    kind, n = case["kind"], case["n"]
    s = {"case": case}
    if kind in ("share", "setup"):
        npp, lb, ub = host.range_partition(n, case["ranks"], 0)
        ptr, col = _rmat(n, case["draws"], 0.57, g, rows=(lb, ub), scramble=True)
        s.update(npp=npp, lb=lb, ub=ub, dim=case["dim"])
        if kind == "setup":
            # the program's own buffers for lists whose lengths only the set-up tells: twice a rank's mean share
            room = 4 * case["draws"] // case["ranks"] + n
            for name in ("lc", "rc", "ids", "pp_l", "p2n_l", "pp_r", "p2n_r"):
                s[name] = torch.full((room,), -1, dtype=torch.int32, device=DEV)
            s.update(ptr=ptr, col=col, table=_normal(g, n, case["dim"]), staged=torch.zeros(min(room, n), case["dim"], device=DEV))
            return s
        full = _normal(g, case["ranks"] * npp, case["dim"])
        if case["bf16"]:
            full = full.bfloat16()
        lp, rp, lc, rc = host.split_CSR_device(ptr, col, lb, ub)
        remote = full
        if case["compact"]:
            rc, ids = host.compact_remote_device(rc, rc.numel())
            remote = full[ids.long()]
        s["xl"], s["xr"] = _side_by_side(full[lb:ub], remote)
        s.update(csr=(lp, lc.contiguous(), rp, rc.contiguous()), out=torch.empty(ub - lb, case["dim"], device=DEV))
        if case["bf16"]:
            s["w"] = _glorot(g, case["dim"], case["dim"]).bfloat16()
            s["next"] = torch.empty(ub - lb, case["dim"], device=DEV, dtype=torch.bfloat16)
        return s
    ptr, col = _rmat(n, case["draws"], case["a"], g)
    zp, zc = _no_remote(n)
    s.update(ptr=ptr, col=col, zp=zp, zc=zc)
    if kind == "gcn":
        d0, h, k = case["d0"], case["hidden"], case["classes"]
        wide = (k + 3) & ~3 if case["pad"] else k            # columns computed by the last update (zero columns behind the classes)
        pitch = (k + 15) & ~15 if case["pad"] else k         # row pitch of the class tables
        w2 = torch.zeros(h, wide, device=DEV)
        w2[:, :k] = _glorot(g, h, k)
        s.update(x=_normal(g, n, d0), w1=_glorot(g, d0, h), w2=w2, wide=wide, pitch=pitch,
                 scale=(ptr[1:] - ptr[:-1]).clamp(min=1).float().rsqrt(),
                 y1=torch.empty(n, h, device=DEV), h1=torch.empty(n, h, device=DEV),
                 y2=torch.zeros(n, pitch, device=DEV), p=torch.zeros(n, pitch, device=DEV))
    elif kind == "gin":
        d0, h, k = case["d0"], case["hidden"], case["classes"]
        gain = 0.5 * n / col.numel()                         # keeps activations of ordinary rows near 1 through five sums
        s.update(x=_normal(g, n, d0), w0=_glorot(g, d0, h), wa=[_glorot(g, h, h) for _ in range(5)],
                 wb=[_glorot(g, h, k if l == 4 else h) * gain for l in range(5)],
                 y=torch.empty(n, h, device=DEV), h=torch.empty(n, h, device=DEV), logits=torch.empty(n, k, device=DEV))
    else:
        dim = case["dim"]
        s.update(x=_normal(g, n, dim), out=torch.empty(n, dim, device=DEV))
        if kind == "parts":
            s["parts"] = host.build_part_device(ptr, n, case["ps"])
    return s


# ---- one pass

def run(s):
    case = s["case"]
    return _RUN[case["kind"]](s, case, case["n"])


def _run_gcn(s, case, n):
    d0, h, k, wide, pitch, scale = case["d0"], case["hidden"], case["classes"], s["wide"], s["pitch"], s["scale"]
    host.dense_forward(s["y1"], s["x"], s["w1"], n, d0, h, row_scale=scale)
    host.mgg_SAG_np_div(s["h1"], s["y1"], s["ptr"], s["col"], s["zp"], s["zc"], 0, n, h, n, 0, 16, 0, 0, row_scale_out=scale)
    host.dense_forward(s["y2"], s["h1"], s["w2"], n, h, wide, row_scale=scale, ld_out=pitch)
    host.mgg_SAG_np_div(s["p"], s["y2"], s["ptr"], s["col"], s["zp"], s["zc"], 0, n, k, n, 0, 16, 0, 0, row_scale_out=scale,
                        ld_in=pitch, ld_out=pitch, softmax=True)
    return s["h1"], s["p"][:, :k]


def _run_gin(s, case, n):
    d0, h, k = case["d0"], case["hidden"], case["classes"]
    host.dense_forward(s["y"], s["x"], s["w0"], n, d0, h)
    for l in range(5):
        host.mgg_GIN_np_div(s["h"], s["y"], s["ptr"], s["col"], s["zp"], s["zc"], 0, n, h, n, 0, 16, 0, 0, 0.0)
        last = l == 4
        host.mlp2_forward(s["logits"] if last else s["y"], s["h"], s["wa"][l], s["wb"][l], n, h, h, k if last else h)
    return s["h"], s["logits"]


def _run_share(s, case, n):
    lp, lc, rp, rc = s["csr"]
    dim, rows = s["dim"], s["ub"] - s["lb"]
    host.mgg_SAG_np_div(s["out"], s["xl"], lp, lc, rp, rc, s["lb"], s["ub"], dim, s["npp"], 0, 16, 0, 0, input_remote=s["xr"])
    if not case["bf16"]:
        return s["out"]
    host.dense_forward_bf16(s["next"], s["out"], s["w"], rows, dim, dim)
    return s["out"], s["next"]


def _run_parts(s, case, n):
    pp, p2n, _ = s["parts"]
    s["out"].zero_()  # the call adds to its output, as the reference's does
    host.SAG_host(s["out"], s["x"], s["ptr"], s["col"], pp, p2n, 0, n, p2n.numel(), case["ps"], case["dim"], 16, 4, 2)
    return s["out"]


def _run_spmm(s, case, n):
    s["out"].zero_()
    host.SpMM(s["out"], s["x"], s["ptr"], s["col"], n, case["dim"], case["ps"], 4)
    return s["out"]


def _run_setup(s, case, n):
    lb, ub, dim = s["lb"], s["ub"], s["dim"]
    lp, rp, lc, rc = host.split_CSR_device(s["ptr"], s["col"], lb, ub)
    compact, ids = host.compact_remote_device(rc, rc.numel())
    part_l = host.build_part_device(lp, ub - lb, case["ps"])
    part_r = host.build_part_device(rp, ub - lb, case["ps"])
    host.gather_rows(s["staged"], s["table"], ids, ids.numel(), dim * 4)
    for name, part in (("lc", lc), ("rc", compact), ("ids", ids), ("pp_l", part_l[0]), ("p2n_l", part_l[1]), ("pp_r", part_r[0]), ("p2n_r", part_r[1])):
        s[name][: part.numel()].copy_(part)
    return [lp, rp, part_l[2], part_r[2], s["staged"]] + [s[name] for name in ("lc", "rc", "ids", "pp_l", "p2n_l", "pp_r", "p2n_r")]


def _run_fresh(s, case, n):
    host.forget(s["ptr"])
    host.mgg_SAG_np_div(s["out"], s["x"], s["ptr"], s["col"], s["zp"], s["zc"], 0, n, case["dim"], n, 0, 0, 0, 0)
    return s["out"]


_RUN = {"gcn": _run_gcn, "gin": _run_gin, "share": _run_share, "parts": _run_parts, "spmm": _run_spmm, "setup": _run_setup, "fresh": _run_fresh}


# ---- what a pass cannot do without

def _neighbors(case):
    """About how many neighbors the graph keeps of its draws: dense graphs draw many pairs twice (fit on graphs of 4 K to 2.4 M nodes)."""
    n, both, a = case["n"], 2 * case["draws"], case.get("a", 0.57)
    keep = 1.0 / (1.0 + (both / n / n / (0.012 if a > 0.5 else 0.3)) ** 0.6) if a > 0.3 else 1.0
    return int(both * keep) + n


def work(case):
    kind, n, e = case["kind"], case["n"], _neighbors(case)
    csr = 4 * (e + n + 1)
    if kind == "gcn":
        d0, h, k = case["d0"], case["hidden"], case["classes"]
        return {"bytes": csr + 4 * (n * d0 + d0 * h + h * k + n + n * h + n * k), "flops": 2 * n * (d0 * h + h * k) + e * (h + k)}
    if kind == "gin":
        d0, h, k = case["d0"], case["hidden"], case["classes"]
        return {"bytes": csr + 4 * (n * d0 + d0 * h + 9 * h * h + h * k + n * h + n * k), "flops": 2 * n * (d0 * h + 9 * h * h + h * k) + 5 * e * h}
    if kind in ("share", "setup"):
        rows, mine = -(-n // case["ranks"]), e // case["ranks"]
        distinct = min(n - rows, int(0.7 * mine))            # remote rows that are asked for at least once, about
        dim, size = case["dim"], 2 if case.get("bf16") else 4
        if kind == "setup":
            return {"bytes": 4 * (2 * mine + 3 * rows + distinct + 4 * mine // case["ps"] + 4 * rows) + 8 * distinct * dim, "flops": 0}
        b = 4 * (mine + 2 * rows) + (rows + distinct) * dim * size + 4 * rows * dim
        if case["bf16"]:
            return {"bytes": b + 2 * dim * dim + 2 * rows * dim, "flops": mine * dim + 2 * rows * dim * dim}
        return {"bytes": b, "flops": mine * dim}
    dim = case["dim"]
    b = csr + 8 * n * dim
    if kind == "parts":
        b += 8 * (e // case["ps"] + n // 2)
    return {"bytes": b, "flops": e * dim}


def tolerance(case):
    """About four times what the passes show against the same passes in 64 bits.  fp32: up to 2.7e-7 (five GIN layers), single
    values up to 1.3e-5 of their size; bf16: 1.7e-3, the rounding of the updated rows, single values up to 6.8e-3."""
    if case["kind"] == "setup":
        return "exact"
    if case.get("bf16"):
        return {"rel": 6e-3, "max": 3e-2}
    return {"rel": 1.2e-6, "max": 6e-5}
