"""Rows of several cache lines aggregated one slice of columns per XCD (k_agg): the oracle's sums at the smallest tables that are
sliced, at widths that end inside the last slice's last line, with rows that cross workgroups finished in the same launch and in the
second one, rows without neighbors, every epilogue, a share's two tables, column blocks and both ways of addressing."""
import numpy as np
import pytest

from tests.test_gpu_parity import oracle_agg
from tests.util import FP32_TOL, assert_close_to_oracle, share_of, to_dev
from oracle import orc

pytestmark = pytest.mark.gpu


def csr(V, seed, hubs=3, empty=False):
    """A few long rows (they cross workgroups), a few neighbors per row otherwise, sorted."""
    rng = np.random.default_rng(seed)
    deg = rng.integers(0 if empty else 1, 5, V)
    deg[rng.integers(0, V, hubs)] = min(V, 6000)
    ptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    col = rng.integers(0, V, ptr[-1]).astype(np.int32)
    row = np.repeat(np.arange(V), deg)
    return ptr, col[np.lexsort((col, row))]


# table sizes on both sides of the lines of the rule, in rows: 256-byte rows 32 MB; 512 bytes 12 MB and 80 MB; 1,024 bytes 12 and 31 MB
@pytest.mark.parametrize("V,dim,ld,slices,flags,empty", [
    (131_072, 64, 64, 2, "plain", False), (131_071, 64, 64, 1, "plain", False), (131_072, 33, 64, 2, "scale", True), (24_576, 128, 128, 2, "gin", False),
    (24_575, 128, 128, 1, "plain", False), (24_576, 97, 128, 2, "acc_relu", True), (163_840, 128, 128, 4, "scale", False), (163_840, 125, 128, 4, "plain", True),
    (12_288, 256, 256, 2, "acc_relu", False), (31_744, 256, 256, 4, "gin", False), (31_744, 250, 256, 4, "scale", True), (16_384, 192, 192, 2, "plain", False),
    (32_768, 96, 96, 1, "plain", False), (40_000, 128, 129, 1, "plain", False)])
def test_slices_of_columns(gpu, V, dim, ld, slices, flags, empty):
    import torch
    ptr, col = csr(V, dim + V, empty=empty)
    x = gpu.fill_normal((V, dim), seed=5)
    sh = share_of(ptr, col, V, 1, 0)
    d_ptr, d_col = to_dev(ptr), to_dev(col)
    z, zc = torch.zeros(V + 1, dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    d_x = torch.full((V, ld), 1e30, device="cuda")
    d_x[:, :dim] = to_dev(x)
    s = gpu.fill_uniform((V,), 0.5, 2.0, seed=6)
    base = gpu.fill_normal((V, dim), seed=7)
    want, mag = oracle_agg(sh, x, x, dim, **(dict(flags=orc.GIN, eps=0.25) if flags == "gin" else {}))
    if flags == "scale":
        want, mag = want * s[:, None], mag * s[:, None]
    if flags == "acc_relu":
        want, mag = np.maximum(want + base, 0), mag + np.abs(base)
    for mode in (0, 1):  # 32-bit offsets and 64-bit addresses
        gpu.set_gather_addressing(mode)
        try:
            out = torch.full((V, ld + 1), 7.5, device="cuda")
            if flags == "acc_relu":
                out[:, :dim] = to_dev(base)
            args = (out, d_x, d_ptr, d_col, z, zc, 0, V, dim, V, 0, 16, 0, 0)
            if flags == "gin":
                gpu.mgg_GIN_np_div(*args, 0.25, ld_in=ld, ld_out=ld + 1)
            else:
                gpu.mgg_SAG_np_div(*args, accumulate=flags == "acc_relu", relu=flags == "acc_relu", row_scale_out=to_dev(s) if flags == "scale" else None,
                                   ld_in=ld, ld_out=ld + 1)
            gpu.sync()
            assert "slices=%d" % slices in gpu.last_agg_kernel(), gpu.last_agg_kernel()
            got = out.cpu().numpy()
            assert np.all(got[:, dim:] == 7.5)
            assert_close_to_oracle(got[:, :dim], want, mag, FP32_TOL, "slices, addressing %d" % mode)
        finally:
            gpu.set_gather_addressing(0)
    gpu.forget(d_ptr)


def test_slices_on_a_share_and_in_column_blocks_and_small_workgroups(gpu):
    """Both tables of a share count towards the size and have to be aligned; a column-blocked plan's partial rows; many short wavefronts
    (more workgroups than finish their rows in the same launch)."""
    import torch
    V, dim = 60_000, 128
    ptr, col = csr(V, 1)
    x = gpu.fill_normal((V, dim), seed=5)
    sh = share_of(ptr, col, V, 2, 1)
    lb, ub = sh["lb"], sh["ub"]
    want, mag = oracle_agg(sh, x[lb:ub], x, dim)
    block = torch.zeros((ub - lb + V) * dim + 32, device="cuda")
    for shift, slices in ((0, 2), (4, 1)):  # (rows off the line boundaries are not sliced)
        xl, xr = block[:(ub - lb) * dim].view(-1, dim), block[(ub - lb) * dim + shift:(ub - lb + V) * dim + shift].view(-1, dim)
        xl.copy_(to_dev(x[lb:ub]))
        xr.copy_(to_dev(x))
        out = torch.full((ub - lb, dim), 7.5, device="cuda")
        d = [to_dev(sh[k]) for k in ("ptr_l", "col_l", "ptr_r", "col_r")]
        gpu.mgg_SAG_np_div(out, xl, *d, lb, ub, dim, sh["npp"], 1, 16, 0, 0, input_remote=xr)
        gpu.sync()
        assert "slices=%d" % slices in gpu.last_agg_kernel()
        assert_close_to_oracle(out.cpu().numpy(), want, mag, FP32_TOL, "share, shift %d" % shift)
        for t in d:
            gpu.forget(t)
    sh = share_of(ptr, col, V, 1, 0)
    want, mag = oracle_agg(sh, x, x, dim)
    d_ptr, d_col, d_x = to_dev(ptr), to_dev(col), to_dev(x)
    z, zc = torch.zeros(V + 1, dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    for blk, wpb, dist, fused in ((20_000, 4, 4, 0), (-1, 1, 1, 0), (-1, 4, 16, 1), (-1, 16, 3, 1)):
        out = torch.full((V, dim), 7.5, device="cuda")
        gpu.mgg_SAG_np_div(out, d_x, d_ptr, d_col, z, zc, 0, V, dim, V, 0, 16, wpb, dist, col_block_rows=blk)
        gpu.sync()
        k = gpu.last_agg_kernel()
        assert "slices=2" in k and "fused=%d" % fused in k and ("blocks=3" in k) == (blk > 0), k
        assert_close_to_oracle(out.cpu().numpy(), want, mag, FP32_TOL, k)
    gpu.forget(d_ptr)


def test_explicit_partitions_stay_whole_and_bit_identical_in_the_static_form(gpu):
    import torch
    V, dim = 30_000, 128
    ptr, col = csr(V, 2)
    x = gpu.fill_normal((V, dim), seed=5)
    d_ptr, d_col, d_x = to_dev(ptr), to_dev(col), to_dev(x)
    pp, p2n, _ = gpu.build_part_device(d_ptr, V, 16)
    outs = []
    for call in (gpu.SAG_host, gpu.SAG_host_static):
        out = torch.zeros(V, dim, device="cuda")
        call(out, d_x, d_ptr, d_col, pp, p2n, 0, V, p2n.numel(), 16, dim, 16, 4, 2)
        gpu.sync()
        assert "slices=1" in gpu.last_agg_kernel()
        outs.append(out.cpu().numpy())
    assert np.array_equal(outs[0], outs[1])
    want, mag = oracle_agg(share_of(ptr, col, V, 1, 0), x, x, dim)
    assert_close_to_oracle(outs[0], want, mag, FP32_TOL, "explicit partitions")
    gpu.forget(d_ptr)
