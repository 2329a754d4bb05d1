"""A few tokens: scores, then top-k inside the gate/up kernel, and the down GEMM that combines (experts_small.hip), against the same
block over the router, streaming and combine kernels, which add in the same order."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["bf16", "mxfp4"])
@pytest.mark.parametrize("E,K", [(4, 4), (32, 4), (70, 1), (129, 8), (1000, 3)])  # top-k keys in one and two registers, and read anew
@pytest.mark.parametrize("H,I", [(64, 3136), (320, 192), (2880, 2880)])  # rows past the first loads, ragged stages
def test_few_tokens(pkg, wl, dev, H, I, E, K, fmt):
    if E > 200 and H > 320:
        E = 200
    table = pkg.normal_table()
    shape = wl.MoeShape("tiny", T=10, H=H, I=I, E=E, K=K, fmt=fmt, seed=H + E)
    blk, raw = wl.make_device_layer(shape, table, dev)
    raw["w_router"][E - 1] = raw["w_router"][0]  # a tie
    raw["b_router"][E - 1] = raw["b_router"][0]
    x = wl.make_device_input(shape, table, dev)
    for n in range(1, 11):
        print("few tokens", H, I, E, K, fmt, n, flush=True)
        t = x[:n].contiguous()
        before = torch.randn(n, H, device=dev)
        r0, r1 = before.clone(), before.clone()
        scores = torch.full((n, E), float("nan"), device=dev)
        want, wi, wv = blk.forward(t, flags=pkg.MOE_FLAG_FORCE_DIRECT, residual_x=r0)
        names = blk.describe(blk.params(t, want, wi, wv))
        if 4 * n * K <= 5 * E:
            assert names["gate_up"] == "expert_small_kernel<%d, 0>" % (fmt == "mxfp4")
            assert (names["router"] == "router_scores_kernel") == (n <= 8 and n * K <= 64)
            tiny = names["router"] == "router_scores_kernel" and n * K <= (16 if fmt == "mxfp4" else 12)
            assert (names["down"] == "expert_tiny_down_kernel<%d>" % (fmt == "mxfp4")) == tiny
            assert names["combine"] == ("in the down kernel" if tiny else "combine_kernel")
        else:
            assert E == 4 and n > 1
        for _ in range(2):  # a second pass over the workspace that the first one left
            y, ti, tv = blk.forward(t)
            assert torch.equal(ti, wi) and torch.equal(tv, wv) and torch.equal(y, want)
        y, ti, tv = blk.forward(t, router_score=scores, residual_x=r1)
        assert torch.equal(ti, wi) and torch.equal(y, want) and torch.equal(r1, r0)
        top = scores.gather(1, ti.long())  # the chosen scores, in order, above all others
        assert (top[:, 1:] <= top[:, :-1]).all() and (scores >= top[:, -1:]).sum(1).le(K + 1).all()


@pytest.mark.parametrize("fmt", ["bf16", "mxfp4"])
@pytest.mark.parametrize("what", ["inf router weight", "nan router weight", "-nan bias", "inf bias", "inf row", "nan row", "inf expert bias", "nan expert bias"])
def test_few_tokens_non_finite(pkg, wl, dev, fmt, what):
    """Infinities and NaN in scores, rows and weights: the same experts, and they reach the same outputs and no others."""
    H, I, E, K = 320, 192, 48, 4
    shape = wl.MoeShape("tiny", T=8, H=H, I=I, E=E, K=K, fmt=fmt, seed=17)
    blk, raw = wl.make_device_layer(shape, pkg.normal_table(), dev)
    x = wl.make_device_input(shape, pkg.normal_table(), dev)
    v = float(what.split()[0])
    kind = what.split(" ", 1)[1]
    if kind == "router weight":
        raw["w_router"][5, 7] = v
    elif kind == "bias":
        raw["b_router"][[3, 40]] = v
    elif kind == "row":
        x[1, 9] = v
        x[5] = v
    else:
        raw["b_mlp2"][:, 11] = v
    bits = lambda t: t.nan_to_num(12345.0, 1e30, -1e30)  # noqa: E731
    for n in (1, 2, 3, 4, 8):
        print("few tokens, non-finite", fmt, what, n, flush=True)
        t = x[:n].contiguous()
        y, ti, tv = blk.forward(t)
        assert blk.describe(blk.params(t, y, ti, tv))["router"] == "router_scores_kernel"
        want, wi, wv = blk.forward(t, flags=pkg.MOE_FLAG_FORCE_DIRECT)
        assert torch.equal(ti, wi) and torch.equal(bits(tv), bits(wv)) and torch.equal(bits(y), bits(want))
        if kind == "row" and n > 1:
            assert bool(y[0].isfinite().all())
