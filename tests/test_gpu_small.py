"""The kernels for a handful of rows per expert (experts_small.hip) at the sizes where their phases, rings, tails and block
sizes change: bit-identical to the producer/consumer kernels, which add in the same order (the oracle checks the block in
test_gpu_parity.py)."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

# (H, I): contraction lengths of 0.5 to 17 stages of 128; 2880 = 22.5 stages, the lengths of the model shapes
DIMS = [(64, 64), (128, 192), (320, 576), (1088, 960), (2176, 1024), (2880, 2880)]


@pytest.mark.parametrize("fmt", ["bf16", "mxfp4"])
@pytest.mark.parametrize("H,I", DIMS)
def test_small_kernel_equals_streaming_kernels(pkg, wl, dev, H, I, fmt):
    table = pkg.normal_table()
    E = 128
    shape = wl.MoeShape("small", T=66, H=H, I=I, E=E, K=2, fmt=fmt, zipf_s=4.0, seed=H + I)  # one expert gets most rows
    blk, _ = wl.make_device_layer(shape, table, dev)
    x = wl.make_device_input(shape, table, dev)
    sizes = set()
    for n in [1, 2, 3, 4, 5, 8, 9, 13, 16, 17, 20, 31, 33, 48, 66]:
        print("small kernel", H, I, fmt, n, flush=True)
        t = x[:n].contiguous()
        y, ti, _ = blk.forward(t)
        p = blk.params(t, y, ti, y)
        assert blk.describe(p)["gate_up"] == "expert_small_kernel<%d, 0>" % (fmt == "mxfp4")
        sizes |= set(torch.bincount(ti.flatten().long(), minlength=E).tolist())
        want, wi, _ = blk.forward(t, flags=pkg.MOE_FLAG_FORCE_DIRECT)
        assert torch.equal(ti, wi) and torch.equal(y, want), (H, I, n)
    assert 0 in sizes and max(sizes) > 16


@pytest.mark.parametrize("T,E,K", [(1, 32, 4), (1, 1000, 8), (3, 130, 8), (40, 1000, 3), (64, 512, 8), (20, 128, 4), (41, 33, 1)])
def test_small_kernel_finds_its_experts(pkg, wl, dev, T, E, K):
    """Blocks count the experts that got rows off in the assignment list: few and many experts, few and many of them used."""
    table = pkg.normal_table()
    for fmt in ("bf16", "mxfp4"):
        shape = wl.MoeShape("small", T=T, H=128, I=64, E=E, K=K, fmt=fmt, seed=T + E)
        blk, _ = wl.make_device_layer(shape, table, dev)
        x = wl.make_device_input(shape, table, dev)
        print("small kernel", shape, flush=True)
        y, ti, _ = blk.forward(x)
        tiny = T * K <= (16 if fmt == "mxfp4" else 12)
        assert blk.describe(blk.params(x, y, ti, y))["gate_up"] == "expert_small_kernel<%d, 0>" % (fmt == "mxfp4")
        assert blk.describe(blk.params(x, y, ti, y))["down"] == ("expert_tiny_down_kernel<%d>" if tiny else "expert_small_kernel<%d, 1>") % (fmt == "mxfp4")
        want, _, _ = blk.forward(x, flags=pkg.MOE_FLAG_FORCE_DIRECT)
        assert torch.equal(y, want)


@pytest.mark.parametrize("T,H,I,small", [(32, 2880, 64, True), (48, 2880, 64, False), (48, 2880, 320, True), (48, 64, 1472, False)])
def test_many_short_mxfp4_blocks_go_to_the_streaming_kernels(pkg, wl, dev, T, H, I, small):
    """More than 16 blocks per compute unit of at most two stages of 128."""
    E, K = 512, 4
    table = pkg.normal_table()
    shape = wl.MoeShape("small", T=T, H=H, I=I, E=E, K=K, fmt="mxfp4", seed=T)
    blk, _ = wl.make_device_layer(shape, table, dev)
    x = wl.make_device_input(shape, table, dev)
    print("small kernel", shape, flush=True)
    y, ti, _ = blk.forward(x)
    assert blk.describe(blk.params(x, y, ti, y))["down"].startswith("expert_small" if small else "expert_stream_direct")
    want, _, _ = blk.forward(x, flags=pkg.MOE_FLAG_FORCE_DIRECT)
    assert torch.equal(y, want)


@pytest.mark.parametrize("fmt", ["bf16", "mxfp4"])
def test_ids_that_name_no_expert_are_skipped(pkg, wl, dev, fmt):
    """The down GEMM entry takes its assignment list from the caller: ids outside [0, E) write no row and change no other."""
    T, H, I, E, K = 20, 192, 320, 48, 2
    shape = wl.MoeShape("small", T=T, H=H, I=I, E=E, K=K, fmt=fmt, seed=7)
    blk, _ = wl.make_device_layer(shape, pkg.normal_table(), dev)
    ids = (torch.arange(T * K, dtype=torch.int32) * 7 % E).view(T, K)
    bad = torch.zeros(T * K, dtype=torch.bool)
    for i, v in enumerate([-1, E, E + 1, 63, 64, 1000, 1023, 1024, 1 << 20, 0x7FFFFFFF, -(1 << 31)]):
        ids.view(-1)[3 * i + 1] = v
        bad[3 * i + 1] = True
    ids, bad = ids.to(dev), bad.to(dev)
    h = torch.randn(T * K, I, device=dev).bfloat16()
    tv = torch.ones(T, K, device=dev)
    got = []
    print("ids out of range", fmt, flush=True)
    for flags in (0, pkg.MOE_FLAG_FORCE_DIRECT):
        y = torch.full((T * K, H), 123.0, device=dev)
        p = blk.params(None, None, ids, tv, flags=flags)
        assert pkg.lib.moe_block_down_gemm(ctypes.byref(p), h.data_ptr(), y.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
        assert blk.describe(p)["down"].startswith("expert_stream_direct" if flags else "expert_small")
        assert (y[bad] == 123.0).all() and not (y[~bad] == 123.0).all(dim=1).any()
        got.append(y)
    assert torch.equal(*got)
