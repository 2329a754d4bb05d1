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


# every kernel with lanes past the row's end, and 300, 600 and 2050 tokens for the forms of the one-launch kernel
ROUTES = [(3, 32, "router_scores_kernel"), (30, 128, "router_scores_kernel + router_finalize_kernel"), (100, 32, "router_fused_kernel"),
          (150, 200, "router_fused_kernel"), (300, 32, "router_rows_kernel"), (600, 32, "router_rows_kernel"), (2050, 32, "router_rows_kernel"),
          (300, 200, "router_screen_kernel + router_refine_kernel")]


@pytest.mark.parametrize("H", [256, 1024, 1088, 2880, 3072])  # 1088 and 2880 leave lanes without a value in a wave's last 256
@pytest.mark.parametrize("T,E,router", ROUTES)
def test_infinite_last_value(pkg, wl, dev, T, E, router, H):
    """Lanes past the row's end take no part, whatever the last value of the row, or of a router row, is."""
    K = 4
    shape = wl.MoeShape("rows", T=T, H=H, I=64, E=E, K=K, fmt="mxfp4", seed=H)
    blk, raw = wl.make_device_layer(shape, pkg.normal_table(), dev)
    x0 = wl.make_device_input(shape, pkg.normal_table(), dev)
    w = raw["w_router"]
    w[:, H - 1] = -0.25
    w[[5, 9, 20, E - 1], H - 1] = 0.25
    for what in ("activation", "weight"):
        x = x0.clone()
        if what == "activation":
            x[::7, H - 1] = float("inf")
        else:
            w[11, H - 1] = float("inf")
        print("infinite last", what, T, E, H, flush=True)
        _, ti, tv = blk.forward(x)
        assert blk.describe(blk.params(x, x, ti, tv))["router"] == router
        _, wi, wv = blk.forward(x, flags=pkg.MOE_FLAG_ROUTER_STRICT_ORDER)
        if what == "activation":
            assert (wi[::7] == torch.tensor([5, 9, 20, E - 1], dtype=torch.int32, device=dev)).all()
        assert torch.equal(ti, wi) and torch.equal(tv.isnan(), wv.isnan())
        assert (tv.nan_to_num(0.0) - wv.nan_to_num(0.0)).abs().max().item() <= 4e-6  # as above
