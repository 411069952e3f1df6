"""Small plans whose workgroups take whole rows (k_agg, FORM_WHOLE): the oracle's sums with rows of the most descriptors that the rule lets
in and of one more, rows that end on and one slot around every workgroup's line, both sides of a share, every epilogue, slices of
columns, 16- and 64-column rows in windows of wider tables; and a captured call replays the eager result."""
import numpy as np
import pytest

from tests.test_gpu_parity import oracle_agg
from tests.util import FP32_TOL, assert_close_to_oracle, share_of, to_dev
from oracle import orc

pytestmark = pytest.mark.gpu


def csr(V, longest, seed, at_line=0):
    """Rows of 1 to `longest` descriptors of 16 neighbors; the first ones fill `at_line` slots less one, so that the long ones behind
    them begin, end and lie across a workgroup's line."""
    rng = np.random.default_rng(seed)
    deg = rng.integers(1, 40, V)
    deg[rng.integers(0, V, V // 8)] = 16 * longest
    if at_line:
        deg[: at_line - 1] = 16
        deg[at_line - 1 : at_line + 1] = 16 * longest
    deg = np.minimum(deg, 16 * longest)
    ptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    return ptr, np.concatenate([np.sort(rng.integers(0, V, d)) for d in deg]).astype(np.int32)


# (width, slots of a workgroup of four wavefronts of one round): a fifth of the slots may be held back, so 64 slots let in 13 descriptors
@pytest.mark.parametrize("dim,slots", [(9, 64), (16, 64), (17, 32), (32, 32), (41, 16), (64, 16), (100, 8), (128, 8)])
@pytest.mark.parametrize("flags", ["plain", "softmax", "gin", "acc_relu", "scale"])
@pytest.mark.parametrize("more", [0, 1])
def test_whole_rows(gpu, dim, slots, flags, more):
    import torch
    longest = slots // 5 + 1 + more
    V = 700
    ptr, col = csr(V, longest, dim + more, at_line=slots - longest)
    ld = dim + 3 if flags == "scale" else dim
    x = gpu.fill_normal((V, dim), seed=31)
    base, s = gpu.fill_normal((V, dim), seed=32), gpu.fill_uniform((V,), 0.5, 2.0, seed=33)
    d_x = torch.full((V, ld), 1e30, device="cuda")
    d_x[:, :dim] = to_dev(x)
    sh = share_of(ptr, col, V, 1, 0)
    want, mag = oracle_agg(sh, x, x, dim, **(dict(flags=orc.GIN, eps=0.25) if flags == "gin" else {}))
    if flags == "scale":
        want, mag = want * s[:, None], mag * s[:, None]
    if flags == "acc_relu":
        want, mag = np.maximum(want + base, 0), mag + np.abs(base)
    z, zc = torch.zeros(V + 1, dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    d_ptr, d_col, d_base, d_s = to_dev(ptr), to_dev(col), to_dev(base), to_dev(s)

    def run(out):
        args = (out, d_x, d_ptr, d_col, z, zc, 0, V, dim, V, 0, 16, 0, 0)
        if flags == "gin":
            gpu.mgg_GIN_np_div(*args, 0.25, ld_in=ld)
        else:
            gpu.mgg_SAG_np_div(*args, ld_in=ld, **{"plain": {}, "softmax": dict(softmax=True), "acc_relu": dict(accumulate=True, relu=True),
                                                   "scale": dict(row_scale_out=d_s)}[flags])

    fresh = lambda: d_base.clone() if flags == "acc_relu" else torch.full((V, dim), 7.5, device="cuda")
    out = fresh()
    run(out)
    gpu.sync()
    k = gpu.last_agg_kernel()
    assert "wpb=4 dist=1 " in k and "whole=%d" % (not more) in k and "fused=1" in k, k
    got = out.cpu().numpy()
    if flags == "softmax":
        e = np.exp(want - want.max(1, keepdims=True))
        e /= e.sum(1, keepdims=True)
        # a logit off by d moves a probability by at most a factor of exp(2 d); the quotient's own rounding and __expf add some 1e-6
        off = 2 * FP32_TOL * mag.max(1, keepdims=True)
        assert (np.abs(got - e) <= e * np.expm1(2 * off) + 4e-6).all()
    else:
        assert_close_to_oracle(got, want, mag, FP32_TOL, k)
    if more or flags == "acc_relu":
        return
    stream = torch.cuda.Stream()
    try:
        with torch.cuda.stream(stream):
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                gpu.use_torch_stream()
                run(out)
                assert "whole=1" in gpu.last_agg_kernel()
            for _ in range(3):
                out.fill_(-1.0)
                graph.replay()
                stream.synchronize()
                assert np.array_equal(out.cpu().numpy(), got)
    finally:
        torch.cuda.synchronize()
        gpu.use_torch_stream()
        gpu.release_cached()


def test_whole_rows_of_a_share_and_of_slices(gpu):
    """Rows with local and remote descriptors; and two slices of columns (512-byte rows, a table of 12 MB without hubs)."""
    import torch
    V, dim = 2000, 41
    ptr, col = csr(V, 3, 7)
    x = gpu.fill_normal((V, dim), seed=41)
    sh = share_of(ptr, col, V, 2, 1)
    lb, ub = sh["lb"], sh["ub"]
    xr = gpu.fill_normal((2 * sh["npp"], dim), seed=42)
    xr[:V] = x
    want, mag = oracle_agg(sh, xr[lb:ub], xr, dim)
    out = torch.full((ub - lb, dim), 7.5, device="cuda")
    d = [to_dev(sh[k]) for k in ("ptr_l", "col_l", "ptr_r", "col_r")]
    both = to_dev(xr)
    gpu.mgg_SAG_np_div(out, both[lb:ub], *d, lb, ub, dim, sh["npp"], 1, 16, 0, 0, input_remote=both)
    gpu.sync()
    assert "whole=1" in gpu.last_agg_kernel(), gpu.last_agg_kernel()
    assert_close_to_oracle(out.cpu().numpy(), want, mag, FP32_TOL, "share")

    V, dim = 24_576, 128
    rng = np.random.default_rng(8)
    deg = rng.integers(1, 40, V)
    ptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    col = rng.integers(0, V, ptr[-1]).astype(np.int32)
    x = gpu.fill_normal((V, dim), seed=43)
    want, mag = oracle_agg(share_of(ptr, col, V, 1, 0), x, x, dim)
    out = torch.full((V, dim), 7.5, device="cuda")
    z, zc = torch.zeros(V + 1, dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    gpu.mgg_SAG_np_div(out, to_dev(x), to_dev(ptr), to_dev(col), z, zc, 0, V, dim, V, 0, 16, 0, 0)
    gpu.sync()
    assert "whole=1 slices=2" in gpu.last_agg_kernel(), gpu.last_agg_kernel()
    assert_close_to_oracle(out.cpu().numpy(), want, mag, FP32_TOL, "slices")


@pytest.mark.parametrize("V", [1, 1023, 1025, 262_145, 1_048_579])
def test_longest_and_empty_rows_are_found_wherever_they_are(gpu, V):
    """One row too long for the rule, or without neighbors, at the first and last places and around the strides in which a plan's build
    goes over the rows."""
    import torch
    dim = 16
    x = torch.ones(V, dim, device="cuda")
    z, zc = torch.zeros(V + 1, dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    for at in sorted({r for r in (0, 63, 64, 1023, 1024, 262_143, 262_144, 786_432, V - 1) if r < V}):
        for of_row in (2, 2000, 0):
            deg = torch.full((V,), 2, dtype=torch.int32, device="cuda")
            deg[at] = of_row
            ptr = torch.zeros(V + 1, dtype=torch.int32, device="cuda")
            ptr[1:] = deg.cumsum(0)
            col = torch.arange(int(ptr[-1]) + 1, device="cuda", dtype=torch.int32) % V
            out = torch.full((V, dim), 7.5, device="cuda")
            gpu.mgg_SAG_np_div(out, x, ptr, col, z, zc, 0, V, dim, V, 0, 16, 0, 0, core_rows=-1)
            gpu.sync()
            k = gpu.last_agg_kernel()
            assert V < 64 * 16 or "whole=%d" % (of_row == 2) in k, (at, of_row, k)
            assert torch.equal(out, deg.float()[:, None].expand(V, dim)), (at, of_row)
            gpu.forget(ptr)
