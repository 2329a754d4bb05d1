"""The combine kernels for every number of experts per token and every number of columns a thread of the fused norm holds: rows by
assignment and by slot give the same bits, and so do the fused norm and the norm as a launch of its own; against the oracle."""
import hostgen
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", range(1, 9))
@pytest.mark.parametrize("H", [64, 1088, 2880, 4096])
def test_combine_of_every_top_k(pkg, wl, oracle, dev, H, K):
    T = 33
    shape = wl.MoeShape("combine", T=T, H=H, I=64, E=9, K=K, fmt="bf16", seed=H + K)
    blk, _ = wl.make_device_layer(shape, pkg.normal_table(), dev)
    t = wl.make_device_input(shape, pkg.normal_table(), dev)
    x0 = torch.randn((T, H), device=dev, generator=torch.Generator(device=dev).manual_seed(K))
    w = torch.rand(H, device=dev, generator=torch.Generator(device=dev).manual_seed(H)).bfloat16()
    print("combine", H, K, flush=True)
    got = []
    for flags in (pkg.MOE_FLAG_FORCE_STREAM | pkg.MOE_FLAG_FORCE_DIRECT, pkg.MOE_FLAG_FORCE_STREAM | pkg.MOE_FLAG_FORCE_BUCKET_LAUNCH):
        x = x0.clone()
        y, ti, _ = blk.forward(t, flags=flags, residual_x=x)
        norm, fused, xf = torch.empty_like(x), torch.full_like(x, float("nan")), x0.clone()
        pkg.rmsnorm(norm, x, w, T, H)
        yf, _, _ = blk.forward(t, flags=flags, residual_x=xf, next_norm_weight=w, next_norm_out=fused)
        assert torch.equal(y, yf) and torch.equal(x, xf) and torch.equal(norm, fused)
        assert torch.equal(x, x0 + y)
        got.append((y, ti))
    assert torch.equal(got[0][1], got[1][1]) and torch.equal(got[0][0], got[1][0])
    hw = hostgen.host_layer(oracle, wl, shape)
    ref, ref_i, _, _ = hostgen.oracle_block(oracle, shape, hw, hostgen.host_input(oracle, wl, shape))
    assert (got[0][1].cpu().numpy() == ref_i).all()
    assert hostgen.rel_err(got[0][0].cpu().numpy(), ref) <= 1e-2  # bf16 operands of both products, as in test_gpu_parity.py


@pytest.mark.parametrize("K,H", [(1, 4096), (4, 2880), (7, 3072), (8, 4096)])
def test_combine_of_more_rows_than_the_cache_holds(pkg, wl, dev, K, H):
    """Rows by slot past 256 MiB are read by other loads: the same bits as for parts of the batch, with and without the norm."""
    T = (256 << 20) // (4 * K * H) + 1
    shape = wl.MoeShape("combine", T=T, H=H, I=64, E=9, K=K, fmt="bf16", seed=H + K)
    blk, _ = wl.make_device_layer(shape, pkg.normal_table(), dev)
    t = wl.make_device_input(shape, pkg.normal_table(), dev)
    x = torch.randn((T, H), device=dev, generator=torch.Generator(device=dev).manual_seed(K))
    w = torch.rand(H, device=dev, generator=torch.Generator(device=dev).manual_seed(H)).bfloat16()
    print("combine, rows past the cache", H, K, T, flush=True)
    flags = pkg.MOE_FLAG_FORCE_STREAM | pkg.MOE_FLAG_FORCE_BUCKET_LAUNCH

    def run(a, b):
        xa, xn, norm = x[a:b].clone(), x[a:b].clone(), torch.empty_like(x[a:b])
        y, _, _ = blk.forward(t[a:b].contiguous(), flags=flags, residual_x=xa)
        yn, _, _ = blk.forward(t[a:b].contiguous(), flags=flags, residual_x=xn, next_norm_weight=w, next_norm_out=norm)
        assert torch.equal(y, yn) and torch.equal(xa, xn)
        return y, xa, norm
    whole = run(0, T)
    for a, b in ((0, 500), (T // 2, T // 2 + 500), (T - 500, T)):
        for got, want in zip(whole, run(a, b)):
            assert torch.equal(got[a:b], want), (a, b)
