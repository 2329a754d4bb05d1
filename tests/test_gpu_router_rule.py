"""Which router kernels run (a block per token, partial sums and finalize, screening and exact scores) does not change the
result: batches on either side of every line of the rule against the single exact pass in the reference's order."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [64, 2880, 3136])  # the last is too long for the one-launch kernel
@pytest.mark.parametrize("E,tokens", [(32, (1, 640, 641, 2047, 2048)), (33, (1, 128, 129, 256, 257)), (250, (5, 128, 129, 256, 263))])
def test_router_kernels_agree(pkg, wl, dev, H, E, tokens):
    table = pkg.normal_table()
    shape = wl.MoeShape("router", T=max(tokens), H=H, I=64, E=E, K=4, fmt="mxfp4", seed=H + E)
    blk, _ = wl.make_device_layer(shape, table, dev)
    x = wl.make_device_input(shape, table, dev)
    for T in tokens:
        print("router", H, E, T, flush=True)
        t = x[:T].contiguous()
        _, ti, tv = blk.forward(t)
        _, wi, wv = blk.forward(t, flags=pkg.MOE_FLAG_ROUTER_STRICT_ORDER)
        assert torch.equal(ti, wi)
        # logits differ, if at all, in the last place of their rounding to fp32: 2^-23 of |logit| < 16
        assert (tv - wv).abs().max().item() <= 4e-6
