"""Bucketing inside the MXFP4 streaming kernel with buckets of many token blocks: those from the third on are dealt out over further
blocks of the launch.  Bit-identical to the launch over a tile map, which adds in the same order."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,I", [(64, 64), (320, 192), (1088, 960), (2880, 2880)])  # one pass and two, 10 and 12 consumers
@pytest.mark.parametrize("T,E,K,zipf", [(200, 8, 1, 9.0), (1024, 1, 1, 0.0), (512, 32, 2, 2.0), (1000, 128, 4, 1.2), (2048, 65, 2, 1.0),
                                        (512, 300, 8, 1.5)])
def test_dealt_out_blocks(pkg, wl, dev, H, I, T, E, K, zipf):
    if H == 2880 and E > 128:
        E = 70
    table = pkg.normal_table()
    shape = wl.MoeShape("skew", T=T, H=H, I=I, E=E, K=K, fmt="mxfp4", zipf_s=zipf, seed=T + H)
    blk, _ = wl.make_device_layer(shape, table, dev)
    x = wl.make_device_input(shape, table, dev)
    print("dealt out", shape, flush=True)
    y, ti, tv = blk.forward(x, flags=pkg.MOE_FLAG_FORCE_STREAM | pkg.MOE_FLAG_FORCE_DIRECT)
    p = blk.params(x, y, ti, tv, flags=pkg.MOE_FLAG_FORCE_STREAM | pkg.MOE_FLAG_FORCE_DIRECT)
    assert "expert_stream_direct_kernel<1, 0" in blk.describe(p)["gate_up"]
    assert torch.bincount(ti.flatten().long(), minlength=E).max().item() > 128
    want, wi, _ = blk.forward(x, flags=pkg.MOE_FLAG_FORCE_STREAM | pkg.MOE_FLAG_FORCE_BUCKET_LAUNCH)
    assert torch.equal(ti, wi) and torch.equal(y, want)


def test_dealt_out_blocks_of_a_callers_list(pkg, wl, dev):
    """The down GEMM on its own takes the list from its caller: ids that name no expert are nobody's rows, and an expert may be
    named twice by one token."""
    H, I, E, K, T = 320, 192, 8, 4, 512
    table = pkg.normal_table()
    shape = wl.MoeShape("skew", T=T, H=H, I=I, E=E, K=K, fmt="mxfp4", seed=5)
    blk, _ = wl.make_device_layer(shape, table, dev)
    x = wl.make_device_input(shape, table, dev)
    g = torch.Generator(device="cpu").manual_seed(3)
    ids = torch.randint(0, 3, (T, K), generator=g, dtype=torch.int32).to(dev)
    ids[::7, 1], ids[::5, 2] = -1, E
    h = torch.randn(T * K, I, device=dev).bfloat16()
    y = torch.full((T * K, H), float("nan"), device=dev)
    tv = torch.zeros(T, K, device=dev)
    p = blk.params(x, torch.empty_like(x), ids, tv, flags=pkg.MOE_FLAG_FORCE_STREAM | pkg.MOE_FLAG_FORCE_DIRECT)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    print("dealt out, caller's list", flush=True)
    assert pkg.lib.moe_block_down_gemm(ctypes.byref(p), h.data_ptr(), y.data_ptr(), st) == 0
    # the same rows a few at a time, where no bucket has a third token block
    flat = ids.flatten()
    for t0 in range(0, T, 32):
        part = ids[t0:t0 + 32].contiguous()
        yp = torch.full((part.numel(), H), float("nan"), device=dev)
        q = blk.params(x[:32].contiguous(), torch.empty(32, H, device=dev), part, tv[:32].contiguous(),
                       flags=pkg.MOE_FLAG_FORCE_STREAM | pkg.MOE_FLAG_FORCE_DIRECT)
        hp = h[t0 * K:t0 * K + part.numel()].contiguous()
        assert pkg.lib.moe_block_down_gemm(ctypes.byref(q), hp.data_ptr(), yp.data_ptr(), st) == 0
        torch.cuda.synchronize()
        got = y[t0 * K:t0 * K + part.numel()]
        named = (part.flatten() >= 0) & (part.flatten() < E)
        assert torch.equal(got[named], yp[named])
        assert got[~named].isnan().all()
    assert (flat == 0).sum().item() > 128


@pytest.mark.parametrize("fmt", ["mxfp4", "bf16"])
@pytest.mark.parametrize("H,I", [(64, 64), (1088, 960)])
@pytest.mark.parametrize("often", [2047, 2049, 3000, 4096])
def test_an_expert_named_more_often_than_a_list_holds(pkg, wl, dev, H, I, fmt, often):
    """A caller's list with one expert in more than 2048 assignments: the first 2048 of them get their rows, the others' rows and
    what lies around the output stay as they are, and the other experts' rows are right."""
    E, K, T = 128, 4, 1024
    shape = wl.MoeShape("skew", T=T, H=H, I=I, E=E, K=K, fmt=fmt, seed=often)
    blk, _ = wl.make_device_layer(shape, pkg.normal_table(), dev)
    A = T * K
    ids = (torch.arange(A, dtype=torch.int32) % (E - 1)) + 1
    ids[torch.randperm(A, generator=torch.Generator().manual_seed(often))[:often]] = 0
    ids = ids.view(T, K).to(dev)
    h = torch.randn(A, I, device=dev).bfloat16()
    tv = torch.zeros(T, K, device=dev)
    st = torch.cuda.current_stream().cuda_stream
    guarded = torch.full((3 * A, H), 123.0, device=dev)
    y = guarded[A:2 * A]
    p = blk.params(None, None, ids, tv)
    assert blk.describe(p)["down"].startswith("expert_stream_direct")
    print("long list", H, I, fmt, often, flush=True)
    assert pkg.lib.moe_block_down_gemm(ctypes.byref(p), h.data_ptr(), y.data_ptr(), st) == 0
    want = torch.empty_like(y)
    for a in range(0, A, 512):  # the same rows, no expert named more than 512 times
        part = ids.view(-1)[a:a + 512].view(-1, K).contiguous()
        q = blk.params(None, None, part, tv[:part.shape[0]].contiguous(), flags=pkg.MOE_FLAG_FORCE_STREAM | pkg.MOE_FLAG_FORCE_DIRECT)
        assert pkg.lib.moe_block_down_gemm(ctypes.byref(q), h[a:].data_ptr(), want[a:].data_ptr(), st) == 0
    flat = ids.view(-1)
    past = (flat == 0) & ((flat == 0).cumsum(0) > 2048)
    assert int(past.sum()) == max(0, often - 2048)
    want[past] = 123.0
    assert torch.equal(y, want)
    assert (guarded[:A] == 123.0).all() and (guarded[2 * A:] == 123.0).all()
