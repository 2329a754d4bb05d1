"""Load-time conversions at the sizes where their waves run out: MX block counts per row around the quads and chunks that a
wave of the repack takes (16 and 4), and dequantisation lengths around the dwords that a wave takes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G", [1, 3, 4, 5, 15, 16, 17, 18, 31, 33])
def test_repack_layout(pkg, dev, G):
    """The tiled layout written out: tile, chunk, lane (blk % 4) * 16 + q; scale dword per lane and quad; 0 elsewhere."""
    E, rows = 3, 128
    rng = np.random.default_rng(G)
    blocks = rng.integers(0, 256, size=(E, rows, G, 16), dtype=np.uint8)
    scales = rng.integers(1, 256, size=(E, rows, G), dtype=np.uint8)
    db, ds = torch.from_numpy(blocks).to(dev), torch.from_numpy(scales).to(dev)
    bb, sb = pkg.mxfp4_tiled_bytes(rows, G * 32)
    out = (torch.full((E * bb,), 0xEE, dtype=torch.uint8, device=dev), torch.full((E * sb,), 0xEE, dtype=torch.uint8, device=dev))
    print("repack", G, flush=True)
    tb, ts = pkg.mxfp4_repack(db, ds, out=out)
    SQ = -(-(-(-G // 4)) // 4)
    want_b = np.zeros((E, rows // 16, G * 256), dtype=np.uint8)
    want_s = np.zeros((E, rows // 16, SQ, 64, 4), dtype=np.uint8)
    for t in range(rows // 16):
        for q in range(16):
            row = (t // 4) * 64 + (q // 4) * 16 + (t % 4) * 4 + q % 4
            for g in range(G):
                lane = (g % 4) * 16 + q
                want_b[:, t, (g // 4) * 1024 + lane * 16:][:, :16] = blocks[:, row, g]
                want_s[:, t, g // 16, lane, (g // 4) % 4] = scales[:, row, g]
    # a ragged last chunk holds only the lanes of the blocks that exist, i.e. its first bytes
    assert np.array_equal(tb.cpu().numpy(), want_b.reshape(-1))
    assert np.array_equal(ts.cpu().numpy(), want_s.reshape(-1))
    ub, us = pkg.mxfp4_unpack(tb, ts, E, rows, G * 32)
    assert torch.equal(ub, db) and torch.equal(us, ds)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 127, 128, 129, 511, 512, 513, 1027])
def test_dequant_lengths(pkg, oracle, dev, n):
    """Block counts around a lane group, a wave's run and a thread block's; every scale byte among them."""
    rng = np.random.default_rng(n)
    blocks = rng.integers(0, 256, size=(n, 16), dtype=np.uint8)
    scales = rng.integers(0, 256, size=(n,), dtype=np.uint8)
    scales[: n // 2] = rng.integers(1, 255, size=n // 2)  # waves with and without the bytes that take the integer routine
    print("dequant", n, flush=True)
    got = pkg.dequant_mxfp4(torch.from_numpy(blocks).to(dev), torch.from_numpy(scales).to(dev))
    want = oracle.dequant_mxfp4(blocks.reshape(1, n, 16), scales.reshape(1, n)).reshape(-1)
    assert np.array_equal(got.view(torch.int16).cpu().numpy().view(np.uint16).reshape(-1), want)
