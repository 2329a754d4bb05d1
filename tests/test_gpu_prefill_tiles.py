"""Token blocks of every tile count of the MXFP4 prefill kernel, odd ones too: one expert takes all tokens, so the last block of its
bucket has exactly the rows asked for.  Bit-identical to the streaming kernels, which add in the same order."""
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
