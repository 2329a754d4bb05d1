"""The 256-token-block kernel of bf16 experts (experts_tile.hip) at the sizes where its block shapes, rings and last row
blocks change: bit-identical to the streaming kernels, which add in the same order (the oracle checks both families in
test_gpu_parity.py)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# contraction lengths of 1, 2, 3, 5, 7 and 9 stages of 64; last row blocks of one, two, three and four groups of 64 rows
DIMS = [(64, 64), (128, 192), (192, 576), (320, 448), (576, 320)]
# rows per bucket around the token-tile counts of every variant (2, 4, 6, 8 tiles a wave) and of one and two more blocks
ROWS = [1, 16, 17, 33, 64, 65, 128, 129, 192, 193, 255, 256, 257, 300, 513]


@pytest.mark.parametrize("H,I", DIMS)
def test_tile_kernel_equals_streaming_kernels(pkg, wl, dev, H, I):
    table = pkg.normal_table()
    shape = wl.MoeShape("tile", T=max(ROWS), H=H, I=I, E=4, K=4, fmt="bf16", seed=H + I)  # every token uses every expert
    blk, _ = wl.make_device_layer(shape, table, dev)
    x = wl.make_device_input(shape, table, dev)
    for n in ROWS:
        print("tile kernel", H, I, n, flush=True)
        t = x[:n].contiguous()
        p = blk.params(t, x, x, x, flags=pkg.MOE_FLAG_FORCE_TILED)
        assert blk.describe(p)["gate_up"] == "expert_tile_bf16_kernel<0>"
        y, ti, _ = blk.forward(t, flags=pkg.MOE_FLAG_FORCE_TILED)
        want, _, _ = blk.forward(t, flags=pkg.MOE_FLAG_FORCE_STREAM)
        assert torch.equal(y, want), (H, I, n)


@pytest.mark.parametrize("T,E,K,zipf_s", [(700, 32, 4, 1.2), (1500, 6, 2, 3.0), (260, 130, 8, 0.0)])
def test_tile_kernel_uneven_buckets(pkg, wl, dev, T, E, K, zipf_s):
    """Buckets of none, a few and many rows beside each other: the block index finds each expert's tiles."""
    table = pkg.normal_table()
    shape = wl.MoeShape("tile", T=T, H=320, I=448, E=E, K=K, fmt="bf16", zipf_s=zipf_s, seed=T)
    blk, _ = wl.make_device_layer(shape, table, dev)
    x = wl.make_device_input(shape, table, dev)
    print("tile kernel", shape, flush=True)
    y, ti, _ = blk.forward(x, flags=pkg.MOE_FLAG_FORCE_TILED)
    want, _, _ = blk.forward(x, flags=pkg.MOE_FLAG_FORCE_STREAM)
    assert torch.equal(y, want)


def test_tile_kernel_rows_past_4_gib(pkg, wl, dev):
    """The down GEMM's activation rows, by slot, end past byte 2^32."""
    T, H, I, E, K = 32800, 64, 8192, 8, 8
    assert T * K * I * 2 > 1 << 32
    table = pkg.normal_table()
    shape = wl.MoeShape("tile", T=T, H=H, I=I, E=E, K=K, fmt="bf16", seed=3)
    blk, _ = wl.make_device_layer(shape, table, dev)
    x = wl.make_device_input(shape, table, dev)
    print("tile kernel", shape, flush=True)
    y, ti, _ = blk.forward(x)
    assert blk.describe(blk.params(x, y, ti, y))["down"] == "expert_tile_bf16_kernel<1>"
    want, _, _ = blk.forward(x, flags=pkg.MOE_FLAG_FORCE_STREAM)
    assert torch.equal(y, want)
