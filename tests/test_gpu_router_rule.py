"""Which router kernels run (a block per token, partial sums and finalize, screening and exact scores) does not change the
result: batches on either side of every line of the rule against the single exact pass in the reference's order."""
import pytest
import torch

pytestmark = pytest.mark.gpu

FUSED, SPLIT, TWO = "router_fused_kernel", "router_partial_kernel + router_finalize_kernel", "router_screen_kernel + router_refine_kernel"
ROWS, SCORES, TOPK_LATER = "router_rows_kernel", "router_scores_kernel + router_finalize_kernel", "router_scores_kernel"
# experts -> tokens and the router of rows that the one-launch kernels take, on both sides of each line
LINES = {
    4: [(1, TOPK_LATER), (8000, FUSED), (16383, FUSED), (16384, ROWS)],
    6: [(2000, FUSED), (3300, ROWS), (4096, ROWS), (4200, FUSED)],
    8: [(2, TOPK_LATER), (3, FUSED), (1500, FUSED), (2048, ROWS), (4096, ROWS), (8191, ROWS), (8192, ROWS)],
    16: [(750, FUSED), (751, ROWS), (2048, ROWS), (4095, ROWS), (4096, ROWS), (4097, TWO)],
    17: [(256, FUSED), (257, ROWS), (1204, ROWS), (1205, ROWS)],
    32: [(8, TOPK_LATER), (9, FUSED), (256, FUSED), (257, ROWS), (640, ROWS), (2047, ROWS), (2048, ROWS)],
    33: [(1, TOPK_LATER), (16, SCORES), (17, ROWS), (128, ROWS), (513, ROWS)],
    48: [(16, SCORES), (17, ROWS), (513, ROWS)],
    49: [(40, SCORES), (41, SPLIT), (64, SPLIT), (65, ROWS), (257, ROWS)],
    128: [(8, TOPK_LATER), (9, SCORES), (64, SPLIT), (65, ROWS), (128, ROWS), (129, ROWS), (2048, ROWS), (2049, ROWS)],
    250: [(5, TOPK_LATER), (9, SCORES), (40, SCORES), (41, SPLIT), (128, SPLIT), (129, FUSED), (256, FUSED), (257, TWO), (263, TWO)],
    257: [(128, SPLIT), (129, FUSED), (255, FUSED), (256, TWO)],
    800: [(40, SCORES), (41, SPLIT)],
    1000: [(1, TOPK_LATER), (32, SCORES), (33, SPLIT), (65, SPLIT), (66, TWO), (128, TWO), (129, TWO)],
}


def other_rows(H, T, E, router):
    """The router of rows of 64, which the one-launch kernel leaves to the others more often, and of rows past its 3072 values."""
    if H == 2880 or router != ROWS:
        return (SCORES if T <= 40 else SPLIT) if router == FUSED and H > 3072 else router
    two = T * E >= (20480 if 16 < E <= 32 else 65536) or T > (256 if E > 48 else 512) and E > 32
    if H == 64:
        return TWO if two and (E <= 16 or E > 64 and T > 2048) else SPLIT if E > 64 and T <= 128 else ROWS
    return TWO if two else SCORES if T <= 40 else SPLIT


@pytest.mark.parametrize("H", [64, 2880, 3136])  # the last is too long for the one-launch kernel
@pytest.mark.parametrize("E", LINES)
def test_router_kernels_agree(pkg, wl, dev, H, E):
    table = pkg.normal_table()
    most = max(T for T, _ in LINES[E])
    shape = wl.MoeShape("router", T=most, H=H, I=64, E=E, K=4, fmt="mxfp4", seed=H + E)
    blk, _ = wl.make_device_layer(shape, table, dev)
    x = wl.make_device_input(shape, table, dev)
    for T, router in LINES[E]:
        print("router", H, E, T, flush=True)
        t = x[:T].contiguous()
        _, ti, tv = blk.forward(t)
        assert blk.describe(blk.params(t, x, ti, tv))["router"] == other_rows(H, T, E, router)
        _, wi, wv = blk.forward(t, flags=pkg.MOE_FLAG_ROUTER_STRICT_ORDER)
        assert torch.equal(ti, wi)
        # logits differ, if at all, in the last place of their rounding to fp32: 2^-23 of |logit| < 16
        assert (tv - wv).abs().max().item() <= 4e-6


@pytest.mark.parametrize("T", [700, 2100])
@pytest.mark.parametrize("H,E,router", [(320, 32, ROWS), (320, 160, TWO), (3136, 32, TWO)])
@pytest.mark.parametrize("what", ["inf weight", "nan weight", "neg nan weight", "nan weight, ties", "nan bias", "inf bias", "inf row", "nan row", "huge row"])
def test_screening_keeps_non_finite_scores(pkg, wl, dev, T, H, E, router, what):
    """Scores that are infinite or not a number rank as in the single exact pass: the screening pass drops an expert for a
    finite approximate score below the bound only."""
    K = 4
    table = pkg.normal_table()
    shape = wl.MoeShape("router", T=T, H=H, I=64, E=E, K=K, fmt="mxfp4", seed=11)
    blk, _ = wl.make_device_layer(shape, table, dev)
    x = wl.make_device_input(shape, table, dev)
    w, b = blk.tensors["w_router"], blk.tensors["b_router"]
    if "ties" in what:  # every other expert inside the bound of the K-th best
        w.copy_(w[:1].expand(E, H).clone())
        b.fill_(0.5)
    if what == "neg nan weight":  # ranks last
        w.view(torch.int16)[5, 7] = -64
        w.view(torch.int16)[E - 1, 9] = -64
    v = float(what[:3]) if what[:3] in ("inf", "nan") else 3.39e38  # the last rounds to an infinity in bf16
    {"nan weight": w[6:6], "weight": w[5], "weight, ties": w[5], "bias": b, "row": x[::3]}[what.split(" ", 1)[1]][..., 7] = v
    print("non-finite router", T, H, E, what, flush=True)
    _, ti, tv = blk.forward(x)
    assert blk.describe(blk.params(x, x, ti, tv))["router"] == router
    _, wi, wv = blk.forward(x, flags=pkg.MOE_FLAG_ROUTER_STRICT_ORDER)
    assert torch.equal(ti, wi)
    assert torch.equal(tv.isnan(), wv.isnan())
    assert (tv.nan_to_num(0.0) - wv.nan_to_num(0.0)).abs().max().item() <= 4e-6


@pytest.mark.parametrize("T,H,E,router", [(300, 2880, 32, ROWS), (300, 320, 128, ROWS), (1000, 2880, 200, TWO), (700, 3136, 32, TWO)])
@pytest.mark.parametrize("x_scale,w_scale", [(1e-38, 1.0), (1e-30, 1.0), (1e-20, 1.0), (1.0, 1e-25), (1e-12, 1e-12), (1e30, 1.0)])
def test_screening_at_the_ends_of_the_float_range(pkg, wl, dev, T, H, E, router, x_scale, w_scale):
    """Norms whose squares are no longer floats: near ties of such rows are decided by exact scores, rows of zeros by the biases."""
    shape = wl.MoeShape("router", T=T, H=H, I=64, E=E, K=4, fmt="mxfp4", seed=5)
    blk, _ = wl.make_device_layer(shape, pkg.normal_table(), dev)
    x = wl.make_device_input(shape, pkg.normal_table(), dev) * x_scale
    w, b = blk.tensors["w_router"], blk.tensors["b_router"]
    b.zero_()
    for e in range(1, E // 2):  # bf16 steps apart
        w[e] = w[0]
        w[e, (7 * e) % H] *= 1.01
    w *= w_scale
    x[5:9] = 0.0
    b[E - 3:] = 1e-30
    print("router, float range", T, H, E, x_scale, w_scale, flush=True)
    _, ti, tv = blk.forward(x)
    assert blk.describe(blk.params(x, x, ti, tv))["router"] == router
    _, wi, wv = blk.forward(x, flags=pkg.MOE_FLAG_ROUTER_STRICT_ORDER)
    assert torch.equal(ti, wi) and torch.equal(tv.isnan(), wv.isnan()) and (tv - wv).nan_to_num(0.0).abs().max().item() <= 4e-6


@pytest.mark.parametrize("E", [1, 63, 64, 65, 128, 129, 192, 256, 257, 512, 513, 1000, 1024])
def test_topk_register_forms(pkg, dev, E):
    """Every number of keys per lane, at its edges: ties to the lower index, infinities and signed zeros in the order of the values,
    rows that are one value throughout."""
    g = torch.Generator().manual_seed(E)
    rows = torch.randn(41, E, generator=g)
    rows[1] = 0.25
    rows[2] = float("-inf")
    rows[3] = torch.where(torch.rand(E, generator=g) < 0.5, -0.0, 0.0)
    rows[4::3] = rows[4::3].mul(2).round()  # few values, many ties
    rows[5, E // 2], rows[5, E - 1], rows[5, 0] = float("inf"), float("inf"), float("-inf")
    rows[6] = torch.arange(E)
    rows[7] = -torch.arange(E).float()
    for K in (1, 3, 8):
        if K > E:
            continue
        v = torch.empty(41, K, device=dev)
        i = torch.empty(41, K, dtype=torch.int32, device=dev)
        print("top-k", E, K, flush=True)
        pkg.topk(v, i, rows.to(dev), 41, E, K)
        want_v, want_i = rows.sort(dim=1, descending=True, stable=True)
        assert torch.equal(i.cpu().long(), want_i[:, :K]) and torch.equal(v.cpu(), want_v[:, :K])
