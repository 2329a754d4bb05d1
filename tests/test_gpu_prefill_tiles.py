"""Token blocks of every tile count of the MXFP4 prefill kernel, odd ones too: one expert takes all tokens, so up to 128 rows its bucket is one
block of exactly the rows asked for (and two even ones past that).  Bit-identical to the streaming kernels, which add in the same order."""
import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = [1, 16, 17, 33, 47, 48, 49, 64, 65, 79, 80, 81, 96, 97, 111, 112, 113, 127, 128, 129, 128 + 40, 128 + 75, 256 + 105]


@pytest.mark.parametrize("H,I", [(64, 320), (320, 192), (2880, 576)])
def test_every_tile_count(pkg, wl, dev, H, I):
    table = pkg.normal_table()
    shape = wl.MoeShape("tiles", T=max(ROWS), H=H, I=I, E=1, K=1, fmt="mxfp4", seed=H + I)
    blk, _ = wl.make_device_layer(shape, table, dev)
    x = wl.make_device_input(shape, table, dev)
    for n in ROWS:
        print("prefill tiles", H, I, n, flush=True)
        t = x[:n].contiguous()
        y, ti, tv = blk.forward(t, flags=pkg.MOE_FLAG_FORCE_TILED)
        p = blk.params(t, y, ti, tv, flags=pkg.MOE_FLAG_FORCE_TILED)
        assert blk.describe(p)["gate_up"] == "expert_prefill_kernel<1, 0, 4>"
        want, _, _ = blk.forward(t, flags=pkg.MOE_FLAG_FORCE_STREAM)
        assert torch.equal(y, want), (n, (y - want).abs().max().item())


def test_block_input_past_4_gib(pkg, wl, dev):
    """The bf16 copy of the block input is 4.3 GB: rows at its end have byte offsets of 33 bits."""
    T, H = 65535, 32832
    shape = wl.MoeShape("far rows", T=T, H=H, I=64, E=2, K=1, fmt="mxfp4", seed=3)
    blk, _ = wl.make_device_layer(shape, pkg.normal_table(), dev)
    x = wl.make_device_input(shape, pkg.normal_table(), dev)
    print("block input past 4 GiB", flush=True)
    y, ti, tv = blk.forward(x)
    assert blk.describe(blk.params(x, y, ti, tv))["gate_up"] == "expert_prefill_kernel<1, 0, 4>"
    for first in (0, T // 2, T - 300):  # the same rows by themselves: the same kernel adds in the same order
        part = x[first:first + 300].contiguous()
        want, wi, _ = blk.forward(part, flags=pkg.MOE_FLAG_FORCE_TILED)
        assert torch.equal(ti[first:first + 300], wi) and torch.equal(y[first:first + 300], want), first
