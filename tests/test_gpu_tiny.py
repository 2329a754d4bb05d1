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
        for _ in range(2):  # a second pass over the workspace that the first one left
            y, ti, tv = blk.forward(t)
            assert torch.equal(ti, wi) and torch.equal(tv, wv) and torch.equal(y, want)
        y, ti, tv = blk.forward(t, router_score=scores, residual_x=r1)
        assert torch.equal(ti, wi) and torch.equal(y, want) and torch.equal(r1, r0)
        top = scores.gather(1, ti.long())  # the chosen scores, in order, above all others
        assert (top[:, 1:] <= top[:, :-1]).all() and (scores >= top[:, -1:]).sum(1).le(K + 1).all()
