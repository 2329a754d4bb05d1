"""The kernels for a handful of rows per expert (experts_small.hip) at the sizes where their phases, rings, tails and block
sizes change: bit-identical to the producer/consumer kernels, which add in the same order (the oracle checks the block in
test_gpu_parity.py)."""
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
        assert blk.describe(blk.params(x, y, ti, y))["down"] == "expert_small_kernel<%d, 1>" % (fmt == "mxfp4")
        want, _, _ = blk.forward(x, flags=pkg.MOE_FLAG_FORCE_DIRECT)
        assert torch.equal(y, want)
