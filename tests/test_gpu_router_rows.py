"""The one-launch form of the two-pass router (a block per 1, 2, 4, 8 or 16 tokens) against the single exact pass in the
reference's order, at the edges of its blocks, expert tiles and k ranges."""
import pytest
import torch

pytestmark = pytest.mark.gpu

TOKENS = [1, 193, 256, 257, 511, 513, 1025, 2050]  # 1, 1, 1, 2, 2, 4, 8, 16 (8 with more than 64 experts) tokens to a block


@pytest.mark.parametrize("H", [64, 1088, 2880, 3072])  # 1, 17, 45 and 48 pairs of k-steps over 16 waves
@pytest.mark.parametrize("E,K", [(3, 2), (16, 1), (17, 4), (32, 8), (33, 4), (64, 4), (65, 4), (128, 8)])
def test_one_launch_router(pkg, wl, dev, H, E, K):
    table = pkg.normal_table()
    shape = wl.MoeShape("rows", T=max(TOKENS), H=H, I=64, E=E, K=K, fmt="mxfp4", seed=H + E)
    blk, raw = wl.make_device_layer(shape, table, dev)
    x = wl.make_device_input(shape, table, dev)
    w, b = raw["w_router"], raw["b_router"]
    w[E - 1] = w[0]  # ties, and near ties, of the first and the last expert
    b[E - 1] = b[0]
    if E > 16:
        w[E // 2] = w[0]
        w[E // 2, 5] *= 1.01
    for T in TOKENS:
        print("one-launch router", H, E, K, T, flush=True)
        t = x[:T].contiguous()
        wy, wi, wv = blk.forward(t, flags=pkg.MOE_FLAG_ROUTER_STRICT_ORDER)
        tv, ti, _, _, n = pkg.router_two_pass_report(t, w, b, K)
        # logits differ, if at all, in the last place of their rounding to fp32: 2^-23 of |logit| < 16
        assert torch.equal(ti, wi) and (tv - wv).abs().max().item() <= 4e-6
        assert int(n.min()) >= K and int(n.max()) <= E
        y, ti, tv = blk.forward(t)  # whichever router the batch takes: the bf16 rows it leaves are the same
        assert torch.equal(ti, wi) and (tv - wv).abs().max().item() <= 4e-6
        assert (y - wy).abs().max().item() <= 1e-5 * max(1.0, wy.abs().max().item())


@pytest.mark.parametrize("H", [256, 1024, 1088, 3072])
def test_one_launch_router_infinite_last_activation(pkg, wl, dev, H):
    """A wave that holds a row in registers has places past the row's end: they take no part, whatever the last value is."""
    T, E, K = 300, 32, 4
    shape = wl.MoeShape("rows", T=T, H=H, I=64, E=E, K=K, fmt="mxfp4", seed=H)
    blk, raw = wl.make_device_layer(shape, pkg.normal_table(), dev)
    x = wl.make_device_input(shape, pkg.normal_table(), dev)
    w = raw["w_router"]
    w[:, H - 1] = 0.0
    w[3, H - 1] = 0.5
    if H % 256 == 0:  # other lengths leave lanes without a value in the last trip, which multiply the row's last by zero
        x[::7, H - 1] = float("inf")
        w[:, H - 1] = 0.25
        w[4:, H - 1] = -0.25
    print("one-launch router, infinite value", H, flush=True)
    _, ti, tv = blk.forward(x)
    assert blk.describe(blk.params(x, x, ti, tv))["router"] == "router_rows_kernel"
    _, wi, wv = blk.forward(x, flags=pkg.MOE_FLAG_ROUTER_STRICT_ORDER)
    assert torch.equal(ti, wi) and (tv.nan_to_num(0.0) - wv.nan_to_num(0.0)).abs().max().item() <= 4e-6
