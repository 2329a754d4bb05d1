"""The block index -> (token block, row block) map of the MXFP4 prefill kernel, launches of few and of many blocks: every output
row as the streaming kernels compute it (they add in the same order)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# one to five row blocks of 256 rows in the two launches, an odd last one among them; 2 to 694 token blocks; with the most of
# them either launch, both or neither has few blocks
@pytest.mark.parametrize("H,I", [(64, 64), (320, 192), (576, 640), (1088, 128), (64, 640)])
@pytest.mark.parametrize("T,E,K,zipf_s", [(1, 4, 2, 0.0), (700, 32, 4, 1.2), (1500, 6, 2, 3.0), (900, 130, 8, 0.0), (9000, 130, 8, 0.5)])
def test_prefill_blocks_cover_every_row(pkg, wl, dev, H, I, T, E, K, zipf_s):
    table = pkg.normal_table()
    shape = wl.MoeShape("prefill", T=T, H=H, I=I, E=E, K=K, fmt="mxfp4", zipf_s=zipf_s, seed=T + H)
    blk, _ = wl.make_device_layer(shape, table, dev)
    x = wl.make_device_input(shape, table, dev)
    print("prefill", shape, flush=True)
    y, ti, _ = blk.forward(x, flags=pkg.MOE_FLAG_FORCE_TILED)
    want, _, _ = blk.forward(x, flags=pkg.MOE_FLAG_FORCE_STREAM)
    assert torch.equal(y, want)


# MXFP4 blocks of up to 128 rows, bf16 of up to 256: buckets of up to 8 blocks, among them the first and the last length that is cut (into
# two equal ones, bf16 into three as well), and one row past whole blocks
@pytest.mark.parametrize("fmt,rows", [("mxfp4", [128, 129, 144, 145, 224, 225, 256, 257, 300, 336, 337, 385, 513, 769, 897]),
                                      ("bf16", [256, 257, 320, 384, 385, 512, 513, 576, 577, 769, 1025])])
def test_evenly_cut_buckets(pkg, wl, dev, fmt, rows):
    table = pkg.normal_table()
    # two row blocks and more in both launches; every token uses both experts
    shape = wl.MoeShape("prefill", T=max(rows), H=320, I=448, E=2, K=2, fmt=fmt, seed=len(rows))
    blk, _ = wl.make_device_layer(shape, table, dev)
    x = wl.make_device_input(shape, table, dev)
    for n in rows:
        print("evenly cut", fmt, n, flush=True)
        t = x[:n].contiguous()
        y, ti, tv = blk.forward(t, flags=pkg.MOE_FLAG_FORCE_TILED)
        p = blk.params(t, y, ti, tv, flags=pkg.MOE_FLAG_FORCE_TILED)
        assert blk.describe(p)["gate_up"].startswith("expert_tile" if fmt == "bf16" else "expert_prefill")
        want, _, _ = blk.forward(t, flags=pkg.MOE_FLAG_FORCE_STREAM)
        assert torch.equal(y, want), n
