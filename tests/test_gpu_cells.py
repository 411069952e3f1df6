"""Dense cells of the aggregation on the matrix cores (mggx_cells.hip): the same sums as the oracle with every epilogue, at widths on
both sides of the 16-column groups, at row counts on both sides of the 512-row groups and 192-column tiles, from one cell to all of
them, with values whose bf16 parts are at the ends of the format, and what a bitmap cannot hold."""
import numpy as np
import pytest

from oracle import orc
from tests.test_gpu_parity import oracle_agg
from tests.util import FP32_TOL, assert_close_to_oracle, share_of, to_dev

pytestmark = pytest.mark.gpu


def graph(V, draws, seed=5):
    from mgg_osdi23_amd import host
    return host.gen_rmat(max(1, (V - 1).bit_length()), V, draws, seed=seed)


def no_remote(V):
    import torch
    return torch.zeros(V + 1, dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")


# rows: one short of / equal to / one past a row group (512), a tile (192), a multiple of neither; least: one edge (every cell that holds
# any, both layers) or so many that only the fullest stay
@pytest.mark.parametrize("V,dim,least,flags", [(191, 1, 1, "plain"), (192, 4, 1, "scale"), (193, 15, 1, "gin"), (511, 16, 1, "plain"), (512, 17, 1, "acc_relu"),
                                               (513, 32, 1, "softmax"), (1000, 33, 60, "scale"), (1537, 41, 1, "softmax"), (2048, 48, 300, "gin"),
                                               (3000, 49, 1, "plain"), (3000, 64, 1, "acc_relu"), (6000, 64, 2000, "softmax"), (6000, 16, 2000, "plain"),
                                               (6000, 44, 400, "scale")])
def test_dense_cells(gpu, V, dim, least, flags):
    import torch
    ptr, col = graph(V, 24 * V)
    x = gpu.fill_normal((V, dim), seed=191)
    sh = share_of(ptr, col, V, 1, 0)
    d_ptr, d_col = to_dev(ptr), to_dev(col)
    z, zc = no_remote(V)
    ld = dim + 3
    d_x = torch.zeros(V, ld, device="cuda")
    d_x[:, :dim] = to_dev(x)
    s = gpu.fill_uniform((V,), 0.5, 2.0, seed=192)
    base = gpu.fill_normal((V, dim), seed=193)
    cells, edges = gpu.cells_prepare(d_ptr, d_col, z, zc, 0, V, dim, least)
    assert 0 < cells and 0 < edges <= len(col) and (least > 1 or edges == len(col))
    kw = dict(flags=orc.GIN, eps=0.5) if flags == "gin" else {}
    want, mag = oracle_agg(sh, x, x, dim, **kw)
    if flags == "scale":
        want, mag = want * s[:, None], mag * s[:, None]
    if flags == "acc_relu":
        want, mag = np.maximum(want + base, 0), mag + np.abs(base)
    # the library's wpb and dist, and others (too few neighbors are left for column blocks: test_column_blocked_rest_beside_cells has those)
    for blk, ps, wpb, dist in ((-1, 16, 0, 0), (max(64, V // 5), 16, 4, 2)):
        out = torch.full((V, ld), 7.5, device="cuda")
        if flags == "acc_relu":
            out[:, :dim] = to_dev(base)
        args = (out, d_x, d_ptr, d_col, z, zc, 0, V, dim, V, 0, ps, wpb, dist)
        if flags == "gin":
            gpu.mgg_GIN_np_div(*args, 0.5, col_block_rows=blk, ld_in=ld, ld_out=ld)
        else:
            gpu.mgg_SAG_np_div(*args, col_block_rows=blk, accumulate=flags == "acc_relu", relu=flags == "acc_relu", softmax=flags == "softmax",
                               row_scale_out=to_dev(s) if flags == "scale" else None, ld_in=ld, ld_out=ld)
        gpu.sync()
        assert "cells=%d" % cells in gpu.last_agg_kernel()
        got = out.cpu().numpy()
        assert np.all(got[:, dim:] == 7.5)
        if flags == "softmax":
            e = np.exp(want.astype(np.float64) - want.max(1, keepdims=True))
            # a logit off by d moves a probability by at most d (of itself); __expf and the sum add a few 1e-7
            assert np.abs(got[:, :dim] - e / e.sum(1, keepdims=True)).max() < FP32_TOL * mag.max() + 1e-6
        else:
            assert_close_to_oracle(got[:, :dim], want, mag, FP32_TOL, "dense cells, blk=%d" % blk)
    ones = torch.ones(V, ld, device="cuda")  # closed form: the degree exactly
    out = torch.zeros(V, ld, device="cuda")
    gpu.mgg_SAG_np_div(out, ones, d_ptr, d_col, z, zc, 0, V, dim, V, 0, 16, 0, 0, ld_in=ld, ld_out=ld)
    gpu.sync()
    assert np.array_equal(out.cpu().numpy()[:, :dim], np.repeat(np.diff(ptr).astype(np.float32)[:, None], dim, 1))
    gpu.forget(d_ptr)


def aggregate(gpu, out, x, csr, lb, dim, flags, scale, **kw):
    """One call with the epilogue `flags` and the knobs left to the library."""
    V = csr[0].numel() - 1
    args = (out, x, *csr, lb, lb + V, dim, V, 0, 16, 0, 0)
    if flags == "gin":
        gpu.mgg_GIN_np_div(*args, 0.5, **kw)
    else:
        gpu.mgg_SAG_np_div(*args, accumulate=flags == "acc_relu", relu=flags == "acc_relu", softmax=flags == "softmax",
                           row_scale_out=scale if flags == "scale" else None, **kw)
    gpu.sync()


def check_epilogue(got, want, mag, base, scale, flags, what):
    """want, mag: the oracle's sums (with the GIN term) and sums of magnitudes, before the other epilogues."""
    if flags == "scale":
        want, mag = want * scale[:, None], mag * scale[:, None]
    if flags == "acc_relu":
        want, mag = np.maximum(want + base, 0), mag + np.abs(base)
    if flags != "softmax":
        return assert_close_to_oracle(got, want, mag, FP32_TOL, what)
    e = np.exp(want.astype(np.float64) - want.max(1, keepdims=True))
    e /= e.sum(1, keepdims=True)
    # a logit off by d moves a probability by at most a factor of exp(2 d); the quotient's own rounding and __expf add some 1e-6
    off = 2 * FP32_TOL * mag.max(1, keepdims=True)
    assert (np.abs(got - e) <= e * np.expm1(2 * off) + 4e-6).all(), what


@pytest.mark.parametrize("flags", ["plain", "scale", "gin", "acc_relu", "softmax"])
@pytest.mark.parametrize("dim", [12, 16, 17, 41, 64])
def test_column_blocked_rest_beside_cells(gpu, dim, flags):
    """Enough neighbors outside the cells for the rest to stay in column blocks: the kernel that finishes those adds the cells' sums (no
    second stream to join) and applies the epilogue.  20 neighbors per row and block are asked for up to width 16, 10 beyond."""
    import torch
    V, least = 2000, 20_000
    ptr, col = graph(V, 100 * V)
    x = gpu.fill_normal((V, dim), seed=211)
    want, mag = oracle_agg(share_of(ptr, col, V, 1, 0), x, x, dim, **(dict(flags=orc.GIN, eps=0.5) if flags == "gin" else {}))
    csr = (to_dev(ptr), to_dev(col), *no_remote(V))
    cells, edges = gpu.cells_prepare(*csr, 0, V, dim, least)
    blocks = 2 if dim <= 16 else 4
    assert 0 < cells and (len(col) - edges) >= (20 if dim <= 16 else 10) * blocks * V
    s, base = gpu.fill_uniform((V,), 0.5, 2.0, seed=212), gpu.fill_normal((V, dim), seed=213)
    ld = dim + 2
    out = torch.full((V, ld), 7.5, device="cuda")
    if flags == "acc_relu":
        out[:, :dim] = to_dev(base)
    aggregate(gpu, out, to_dev(x), csr, 0, dim, flags, to_dev(s), col_block_rows=V // blocks, ld_out=ld)
    k = gpu.last_agg_kernel()
    assert "blocks=%d " % blocks in k and "merged_finish" in k and "cells=%d" % cells in k, k
    got = out.cpu().numpy()
    assert np.all(got[:, dim:] == 7.5)
    check_epilogue(got[:, :dim], want, mag, base, s, flags, k)
    gpu.forget(csr[0])


@pytest.mark.parametrize("flags", ["plain", "scale", "gin", "acc_relu", "softmax"])
@pytest.mark.parametrize("dim,long_row,form", [(16, 0, "whole"), (16, 1, "fused"), (41, 0, "whole"), (41, 1, "fused"), (64, 0, "whole"), (64, 1, "fused")])
def test_small_rest_beside_cells(gpu, dim, long_row, form, flags):
    """The rest of a small graph in the forms of k_agg that finish their own rows: whole rows per workgroup, and counters where one row is
    long.  The rest leaves ReLU and softmax to the kernel that adds the cells' sums."""
    import torch
    V, hubs = 3000, 512
    rng = np.random.default_rng(dim)
    rows = [set(range(hubs)) if v < hubs else set() for v in range(V)]
    for v in range(V):
        rows[v] |= set((hubs + rng.choice(V - hubs, rng.integers(17, 30), replace=False)).tolist())
    if long_row:
        rows[5] |= set(range(V))
    ptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    col = np.concatenate([np.sort(np.fromiter(r, np.int32)) for r in rows]).astype(np.int32)
    x = gpu.fill_normal((V, dim), seed=221)
    want, mag = oracle_agg(share_of(ptr, col, V, 1, 0), x, x, dim, **(dict(flags=orc.GIN, eps=0.5) if flags == "gin" else {}))
    csr = (to_dev(ptr), to_dev(col), *no_remote(V))
    cells, edges = gpu.cells_prepare(*csr, 0, V, dim, 12_000)
    assert 0 < cells and 0.9 * hubs * hubs < edges
    s, base = gpu.fill_uniform((V,), 0.5, 2.0, seed=222), gpu.fill_normal((V, dim), seed=223)
    out = to_dev(base) if flags == "acc_relu" else torch.full((V, dim), 7.5, device="cuda")
    aggregate(gpu, out, to_dev(x), csr, 0, dim, flags, to_dev(s))
    k = gpu.last_agg_kernel()
    assert "fused=1 whole=%d " % (form == "whole") in k and "cells=%d" % cells in k, k
    check_epilogue(out.cpu().numpy(), want, mag, base, s, flags, k)
    gpu.forget(csr[0])


@pytest.mark.parametrize("dim,block_rows", [(33, -1), (41, -1), (41, 70_000), (64, -1), (64, 70_000)])
@pytest.mark.parametrize("flags", ["acc_relu", "softmax"])
def test_sliced_rest_beside_cells(gpu, dim, block_rows, flags):
    """Rows of two cache lines out of a table of 32 MB and more: the rest is gathered in two slices of columns, in plain order and in
    column blocks."""
    import torch
    V, ld = 140_000, 64
    ptr, col = graph(V, (3 if block_rows < 0 else 24) * V)
    x = gpu.fill_normal((V, dim), seed=231)
    want, mag = oracle_agg(share_of(ptr, col, V, 1, 0), x, x, dim)
    csr = (to_dev(ptr), to_dev(col), *no_remote(V))
    cells, edges = gpu.cells_prepare(*csr, 0, V, dim, 1000 if block_rows < 0 else 4000)
    assert 0 < cells and 0 < edges < len(col)
    base = gpu.fill_normal((V, dim), seed=233)
    d_x = torch.full((V, ld), 1e30, device="cuda")
    d_x[:, :dim] = to_dev(x)
    out = to_dev(base) if flags == "acc_relu" else torch.full((V, dim), 7.5, device="cuda")
    aggregate(gpu, out, d_x, csr, 0, dim, flags, None, ld_in=ld, col_block_rows=block_rows)
    k = gpu.last_agg_kernel()
    assert "slices=2" in k and "cells=%d" % cells in k and ("blocks=1 " in k) == (block_rows < 0) == ("merged_finish" not in k), k
    check_epilogue(out.cpu().numpy(), want, mag, base, None, flags, k)
    gpu.forget(csr[0])


@pytest.mark.parametrize("dim", [41, 64])
def test_dense_cells_refused_by_the_rule(gpu, dim):
    """A graph whose degrees promise more than its cells hold (58 % of the edges in cells of 1,400 and more, the rule asks for 67): the core
    from LDS runs, with the cells counted once; asked for, the cells run; both give the plain order's sums."""
    import torch
    V = 250_000
    ptr, col = graph(V, 10_000_000, seed=7)
    csr = (to_dev(ptr), to_dev(col), *no_remote(V))
    x = torch.randn(V, dim, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    out = torch.empty(V, dim, device="cuda")

    def run(want, **kw):
        gpu.mgg_SAG_np_div(out, kw.pop("x", x), *csr, 0, V, dim, V, 0, 0, 0, 0, **kw)
        gpu.sync()
        k = gpu.last_agg_kernel()
        assert ("cells=" in k, "core=" in k) == dict(none=(False, False), LDS=(False, True), cells=(True, True))[want], k
        return out.cpu().numpy().astype(np.float64)

    plain, mag = run("none", core_rows=-1), run("none", core_rows=-1, x=x.abs())
    refused = run("LDS")
    built = gpu.cache_stats()["core_plan_build_ms"]
    assert np.array_equal(run("LDS"), refused) and gpu.cache_stats()["core_plan_build_ms"] == built
    assert gpu.cells_prepare(*csr, 0, V, dim, 1400)[0] > 0
    asked = run("cells")
    for got in (refused, asked):
        assert np.all(np.abs(got - plain) <= 2 * FP32_TOL * mag)
    gpu.forget(csr[0])


def test_dense_cells_of_a_complete_graph(gpu):
    """Every position set, so every row has a third neighbor among each three columns: both layers are full."""
    import torch
    V, dim = 700, 20
    ptr = (np.arange(V + 1) * V).astype(np.int32)
    col = np.tile(np.arange(V, dtype=np.int32), V)
    x = gpu.fill_normal((V, dim), seed=3)
    d_ptr, d_col = to_dev(ptr), to_dev(col)
    z, zc = no_remote(V)
    cells, edges = gpu.cells_prepare(d_ptr, d_col, z, zc, 0, V, dim, 1)
    assert cells == 2 * 2 * 4 and edges == V * V  # 2 row groups x 4 tiles x 2 layers
    out = torch.full((V, dim), 7.5, device="cuda")
    gpu.mgg_SAG_np_div(out, to_dev(x), d_ptr, d_col, z, zc, 0, V, dim, V, 0, 16, 0, 0)
    gpu.sync()
    want, mag = x.astype(np.float64).sum(0), np.abs(x).astype(np.float64).sum(0)
    assert_close_to_oracle(out.cpu().numpy(), np.repeat(want[None], V, 0), np.repeat(mag[None], V, 0), FP32_TOL, "complete graph")
    gpu.forget(d_ptr)


@pytest.mark.parametrize("kind", ["subnormal", "tiny", "wide", "huge", "overflow", "inf", "nan"])
def test_dense_cells_at_the_ends_of_the_format(gpu, kind):
    """Values whose lower bf16 parts would fall out of the format unscaled, values that have no parts once scaled, sums beyond fp32, and
    infinities and NaN, which reach the rows that have their column and no other."""
    import torch
    V, dim = 1500, 18
    ptr, col = graph(V, 60_000, seed=9)
    x = gpu.fill_normal((V, dim), seed=5)
    hub = int(np.argmax(np.diff(ptr)))
    leaf = int(np.argmin(np.diff(ptr)))
    if kind == "subnormal":
        x = (x * np.float32(2.0 ** -126)).astype(np.float32)
    elif kind == "tiny":
        x = (x * np.float32(2.0 ** -112)).astype(np.float32)
    elif kind == "wide":
        x = (x * np.exp2(np.random.default_rng(1).integers(-60, 60, x.shape)).astype(np.float32)).astype(np.float32)
    elif kind == "huge":
        x[hub, 3] = np.float32(3e35)
        x[leaf, 4] = np.float32(-2e33)
    elif kind == "overflow":
        x[:, 2] = np.float32(2e38)
        x[:, 7] = np.where(np.arange(V) % 2 == 0, 3e38, -3e38).astype(np.float32)
    elif kind == "inf":
        x[hub, 1], x[leaf, 5] = np.inf, -np.inf
        x[leaf, 1] = -np.inf
    else:
        x[hub, 0], x[leaf, 17] = np.nan, np.nan
    d_ptr, d_col, d_x = to_dev(ptr), to_dev(col), to_dev(x)
    z, zc = no_remote(V)
    outs = []
    for cells in (False, True):
        if cells:
            assert gpu.cells_prepare(d_ptr, d_col, z, zc, 0, V, dim, 1)[1] == len(col)
        out = torch.full((V, dim), 7.5, device="cuda")
        gpu.mgg_SAG_np_div(out, d_x, d_ptr, d_col, z, zc, 0, V, dim, V, 0, 16, 0, 0)
        gpu.sync()
        assert ("cells=" in gpu.last_agg_kernel()) == cells
        outs.append(out.cpu().numpy())
    plain, got = outs
    if kind == "overflow":  # which partial sums overflow depends on the order: finite sums where all orders stay finite
        one_sided = [c for c in range(dim) if c != 7]
        assert np.array_equal(np.isfinite(plain[:, one_sided]), np.isfinite(got[:, one_sided]))
        assert np.array_equal(plain[:, 2] == np.inf, got[:, 2] == np.inf)
    else:
        assert np.array_equal(np.isnan(plain), np.isnan(got)) and np.array_equal(plain == np.inf, got == np.inf) and np.array_equal(plain == -np.inf, got == -np.inf)
    with np.errstate(all="ignore"):
        rows = np.repeat(np.arange(V), np.diff(ptr))
        want, mag = np.zeros((V, dim)), np.zeros((V, dim))
        np.add.at(want, rows, x[col].astype(np.float64))
        np.add.at(mag, rows, np.abs(x[col]).astype(np.float64))
    ok = np.isfinite(got) & (mag < 3e38)
    # (half an ulp of the smallest subnormal per addition on top of the relative bound)
    floor = np.diff(ptr)[:, None] * 2.0 ** -149
    with np.errstate(all="ignore"):
        assert np.all(np.abs(got - want)[ok] <= (FP32_TOL * mag + floor)[ok])
    gpu.forget(d_ptr)


def test_dense_cells_share_unsorted_rows_parallel_edges_and_capture(gpu):
    """Rows that start at lb > 0 with shuffled neighbor lists; a CSR with an edge listed twice has no such plan and keeps the ordinary path;
    a call replayed from a graph gives the eager result bit for bit."""
    import torch
    V, dim, lb = 1300, 37, 3900
    ptr, col = graph(V, 50_000, seed=4)
    rng = np.random.default_rng(3)
    col = (col + lb).astype(np.int32)
    for v in range(0, V, 3):
        rng.shuffle(col[ptr[v]:ptr[v + 1]])
    x = gpu.fill_normal((V, dim), seed=197)
    sh = dict(npp=V, lb=lb, ub=lb + V, ptr_l=ptr, col_l=col, ptr_r=np.zeros(V + 1, np.int32), col_r=np.zeros(0, np.int32))
    want, mag = oracle_agg(sh, x, x, dim)
    d_ptr, d_col, d_x = to_dev(ptr), to_dev(col), to_dev(x)
    z, zc = no_remote(V)
    cells, edges = gpu.cells_prepare(d_ptr, d_col, z, zc, lb, lb + V, dim, 40)
    assert 0 < edges < len(col)
    out = torch.full((V, dim), 7.5, device="cuda")
    call = lambda: gpu.mgg_SAG_np_div(out, d_x, d_ptr, d_col, z, zc, lb, lb + V, dim, V, 0, 16, 0, 0)
    call()
    gpu.sync()
    assert "cells=%d" % cells in gpu.last_agg_kernel()
    eager = out.cpu().numpy()
    assert_close_to_oracle(eager, want, mag, FP32_TOL, "dense cells, lb > 0, shuffled rows")
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        gpu.use_torch_stream()
        call()
        stream.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            call()
    gpu.use_torch_stream()
    for _ in range(3):
        out.fill_(-3.0)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), eager)
        call()  # live work of the library between the replays
        gpu.sync()
        assert np.array_equal(out.cpu().numpy(), eager)
    del g
    gpu.forget(d_ptr)
    hub = int(np.argmax(np.diff(ptr)))
    twice = np.insert(col, ptr[hub], col[ptr[hub]])
    ptr2 = ptr.copy()
    ptr2[hub + 1:] += 1
    d_ptr2, d_col2 = to_dev(ptr2), to_dev(twice.astype(np.int32))
    assert gpu.cells_prepare(d_ptr2, d_col2, z, zc, lb, lb + V, dim, 1) == (0, 0)
    gpu.mgg_SAG_np_div(out, d_x, d_ptr2, d_col2, z, zc, lb, lb + V, dim, V, 0, 16, 0, 0)
    gpu.sync()
    assert "cells=" not in gpu.last_agg_kernel()
    want2 = want.copy()
    want2[hub] += x[col[ptr[hub]] - lb]
    assert_close_to_oracle(out.cpu().numpy(), want2, mag + np.abs(x).max(), FP32_TOL, "an edge listed twice")
    gpu.forget(d_ptr2)


def test_dense_cells_by_rule(gpu):
    """A graph whose hubs hold most edges among themselves, large enough for a core to pay: the rule takes the cells, explicit sizes the
    LDS, -1 neither; a graph without hubs takes neither."""
    import torch
    V, dim = 100_000, 16
    z, zc = no_remote(V)
    out = torch.empty(V, dim, device="cuda")
    x = torch.randn(V, dim, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    ptr, col = gpu.gen_rmat(17, V, 45_000_000, seed=7)
    d_ptr, d_col = to_dev(ptr), to_dev(col)
    outs = {}
    for core in (0, 20480, -1):
        gpu.mgg_SAG_np_div(out, x, d_ptr, d_col, z, zc, 0, V, dim, V, 0, 0, 0, 0, core_rows=core)
        gpu.sync()
        k = gpu.last_agg_kernel()
        assert ("cells=" in k) == (core == 0) and ("core=" in k) == (core >= 0), k
        outs[core] = out.cpu().numpy().astype(np.float64)
    mag = np.zeros((V, dim))
    gpu.mgg_SAG_np_div(out, x.abs(), d_ptr, d_col, z, zc, 0, V, dim, V, 0, 0, 0, 0, core_rows=-1)
    gpu.sync()
    mag = out.cpu().numpy().astype(np.float64)
    for core in (0, 20480):
        assert np.all(np.abs(outs[core] - outs[-1]) <= 2 * FP32_TOL * mag)
    gpu.forget(d_ptr)
