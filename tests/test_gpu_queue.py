"""The work-queue entries (moe_mlp1_swiglu, moe_mlp2_scatter and their MXFP4 forms) over entries of every token-tile count, of
no rows and of many token blocks, few and many of them, against the same sums in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# rows per entry; up to 16 a tile of weight rows per wave; the last leaves compute units to shares of an entry's token blocks
ROWS = [[1, 0, 15, 16, 17, 33, 48, 63, 64, 65, 129, 200], [1, 0, 3, 4, 5, 8, 13, 16], [3], [700, 0]]


@pytest.mark.parametrize("fmt", ["bf16", "mxfp4"])
@pytest.mark.parametrize("H,I", [(64, 64), (320, 192), (576, 832)])
@pytest.mark.parametrize("rows", ROWS, ids=["mixed", "short", "few", "long"])
def test_queue_entries(pkg, wl, dev, H, I, rows, fmt):
    E, A = len(rows) + 1, sum(rows)
    shape = wl.MoeShape("queue", T=A, H=H, I=I, E=E, K=1, fmt=fmt, seed=H + I)
    blk, raw = wl.make_device_layer(shape, pkg.normal_table(), dev, keep_canonical=True)
    x = wl.make_device_input(shape, pkg.normal_table(), dev)
    w = blk.tensors
    if fmt == "bf16":
        w1, w2 = w["w_mlp1"].double().view(E, 2 * I, H), w["w_mlp2"].double().view(E, H, I)
    else:
        w1, w2 = (pkg.dequant_mxfp4(raw[n + "_blocks"], raw[n + "_scales"]).double().view(E, r, k)
                  for n, r, k in (("w_mlp1", 2 * I, H), ("w_mlp2", H, I)))
    b1, b2 = w["b_mlp1"].double().view(E, 2 * I), w["b_mlp2"].double().view(E, H)
    tokens = torch.randperm(A, device=dev).to(torch.int32)
    weights = torch.rand(A, device=dev)
    queue, off = [7, 7, 7], 0  # one triple in front that work_start leaves out
    gate_want = torch.zeros(A, I, dtype=torch.float64, device=dev)
    out_want = torch.zeros(A, H, dtype=torch.float64, device=dev)
    for i, n in enumerate(rows):
        e = E - 1 - i
        queue += [e, off, n]
        y = x[off:off + n].bfloat16().double() @ w1[e].T + b1[e]
        g, u = y[:, 0::2].clamp(max=7.0), y[:, 1::2].clamp(-7.0, 7.0)
        gate_want[off:off + n] = g * torch.sigmoid(1.702 * g) * (u + 1)
        off += n
    queue = torch.tensor(queue, dtype=torch.int32, device=dev)
    gate = torch.empty(A, I, device=dev)
    out = torch.zeros(A, H, device=dev)
    print("queue", H, I, rows, fmt, flush=True)
    n = len(rows)
    if fmt == "bf16":
        pkg.moe_mlp1_swiglu(queue, 1, n, x, gate, w["w_mlp1"], w["b_mlp1"], H, I, 2 * I * H, 2 * I, 1.702, 7.0, max(rows), 0)
        pkg.moe_mlp2_scatter(queue, 1, n, gate, tokens, weights, out, w["w_mlp2"], w["b_mlp2"], I, H, I * H, H, max(rows), 0)
    else:
        pkg.moe_mlp1_swiglu_mxfp4(queue, 1, n, x, gate, w["w_mlp1"], w["w_mlp1_scales"], w["b_mlp1"], H, I, 2 * I, 1.702, 7.0,
                                  max(rows), 0)
        pkg.moe_mlp2_scatter_mxfp4(queue, 1, n, gate, tokens, weights, out, w["w_mlp2"], w["w_mlp2_scales"], w["b_mlp2"], I, H,
                                   H, max(rows), 0)
    off = 0
    for i, n in enumerate(rows):
        e = E - 1 - i
        h = gate[off:off + n].bfloat16().double()
        out_want[tokens[off:off + n].long()] = (h @ w2[e].T + b2[e]) * weights[off:off + n, None].double()
        off += n
    # fp32 sums of at most 832 exact products: K / 2 roundings of 2^-24 on average, and 1e-6 of the fast exponential
    for got, want in ((gate, gate_want), (out, out_want)):
        assert ((got.double() - want).norm() / want.norm()).item() < 5e-5


def test_queue_rows_beyond_the_hint(pkg, wl, dev):
    """max rows is a hint: entries with more rows than it says take further passes."""
    shape = wl.MoeShape("queue", T=70, H=128, I=64, E=1, K=1, fmt="bf16", seed=1)
    blk, _ = wl.make_device_layer(shape, pkg.normal_table(), dev)
    x = wl.make_device_input(shape, pkg.normal_table(), dev)
    w = blk.tensors
    queue = torch.tensor([0, 0, 70], dtype=torch.int32, device=dev)
    got = [torch.empty(70, 64, device=dev) for _ in range(2)]
    for hint, gate in zip((5, 70), got):
        pkg.moe_mlp1_swiglu(queue, 0, 1, x, gate, w["w_mlp1"], w["b_mlp1"], 128, 64, 2 * 64 * 128, 128, 1.702, 7.0, hint, 0)
    assert torch.equal(*got)


@pytest.mark.parametrize("fmt", ["bf16", "mxfp4"])
@pytest.mark.parametrize("K", [64, 96, 320, 576])  # half, three quarters, half, half of the last stage of 128
def test_queue_non_finite_rows(pkg, wl, dev, K, fmt):
    """Infinities and NaN of a row reach what the sums in 64 bits say and no more: positions past the row's end, in the last
    stage of the contraction, count as zeros against them.  Rows up to 16 and more of them (either kernel)."""
    if fmt == "bf16" and K % 64:
        pytest.skip("bf16 experts take K % 64 == 0")
    H, rows = 128, [40, 9]
    A = sum(rows)
    if fmt == "bf16":
        w = (0.02 * torch.randn(2, H, K, device=dev)).bfloat16()
        args, wd = (w,), w.double()
    else:
        blocks = torch.randint(0, 256, (2, H, K // 32, 16), dtype=torch.uint8, device=dev)
        scales = torch.randint(119, 128, (2, H, K // 32), dtype=torch.uint8, device=dev)
        args, wd = pkg.mxfp4_repack(blocks, scales), pkg.dequant_mxfp4(blocks, scales).double().view(2, H, K)
    bias = torch.randn(2, H, device=dev).bfloat16()
    x = torch.randn(A, K, device=dev)
    for r, (c, v) in enumerate([(0, "inf"), (5, "-inf"), (31, "inf"), (K - 1, "inf"), (K - 32, "-inf"), (2, "nan"), (K - 2, "nan")]):
        x[5 * r + 1, c] = float(v)
        x[A - 1 - r, c] = float(v)
    want = torch.cat([x[:40].double() @ wd[0].T + bias[0].double(), x[40:].double() @ wd[1].T + bias[1].double()])
    tokens = torch.arange(A, dtype=torch.int32, device=dev)
    ones = torch.ones(A, device=dev)
    print("queue non-finite", K, fmt, flush=True)
    for queue, hint in (([0, 0, 40, 1, 40, 9], 40), ([1, 40, 9], 9)):
        n, first = len(queue) // 3, queue[1]
        q = torch.tensor(queue, dtype=torch.int32, device=dev)
        out = torch.zeros(A, H, device=dev)
        if fmt == "bf16":
            pkg.moe_mlp2_scatter(q, 0, n, x, tokens, ones, out, *args, bias, K, H, K * H, H, hint, 0)
        else:
            pkg.moe_mlp2_scatter_mxfp4(q, 0, n, x, tokens, ones, out, *args, bias, K, H, H, hint, 0)
        got, ref = out[first:].double(), want[first:]
        assert torch.equal(got.isnan(), ref.isnan())
        assert torch.equal(got.isposinf(), ref.isposinf()) and torch.equal(got.isneginf(), ref.isneginf())
        fin = ref.isfinite()
        # rows rounded to bf16: 2^-9 of each of K terms
        assert ((got[fin] - ref[fin]).norm() / ref[fin].norm()).item() < 2.0 ** -8
        assert ref[~fin].numel() > 0 and ref.isposinf().any() and ref.isneginf().any()


@pytest.mark.parametrize("fmt", ["bf16", "mxfp4"])
@pytest.mark.parametrize("rows", [[8] * 31 + [1000], [700] + [1] * 70 + [65, 64, 400] + [0] * 60 + [129], [300, 5], [500], [100] * 7,
                                  [3] * 1020 + [0, 200, 1, 64, 90, 7, 130]],
                         ids=["last", "spread", "two", "one", "seven", "parts"])
def test_queue_uneven_entries(pkg, wl, dev, rows, fmt):
    """Long entries among short ones, fewer entries than XCDs, and more of them than one launch takes: whole blocks of 64 rows
    are dealt out over all blocks of the launch, and every row is computed once."""
    H, I, E, A = 192, 320, 5, sum(rows)
    shape = wl.MoeShape("queue", T=1, H=H, I=I, E=E, K=1, fmt=fmt, seed=len(rows))
    blk, raw = wl.make_device_layer(shape, pkg.normal_table(), dev, keep_canonical=True)
    w = blk.tensors
    w2 = w["w_mlp2"].double() if fmt == "bf16" else pkg.dequant_mxfp4(raw["w_mlp2_blocks"], raw["w_mlp2_scales"]).double()
    w2 = w2.view(E, H, I)
    gate = torch.randn(A, I, device=dev)
    tokens = torch.randperm(A, device=dev).int()
    weights = torch.rand(A, device=dev) + 0.5
    expert = torch.tensor([i * 3 % E for i in range(len(rows))], device=dev)
    sizes = torch.tensor(rows, device=dev)
    queue = torch.stack([expert, sizes.cumsum(0) - sizes, sizes], 1).int().contiguous()
    want = torch.zeros(A, H, dtype=torch.float64, device=dev)
    of_row = expert.repeat_interleave(sizes)
    for e in range(E):
        m = of_row == e
        y = gate[m].bfloat16().double() @ w2[e].T + w["b_mlp2"].view(E, H)[e].double()
        want[tokens[m].long()] = y * weights[m, None].double()
    print("queue uneven", len(rows), max(rows), fmt, flush=True)
    for hint in (max(rows), 100):
        out = torch.zeros(A, H, device=dev)
        if fmt == "bf16":
            pkg.moe_mlp2_scatter(queue, 0, len(rows), gate, tokens, weights, out, w["w_mlp2"], w["b_mlp2"], I, H, I * H, H, hint, 0)
        else:
            pkg.moe_mlp2_scatter_mxfp4(queue, 0, len(rows), gate, tokens, weights, out, w["w_mlp2"], w["w_mlp2_scales"],
                                       w["b_mlp2"], I, H, H, hint, 0)
        # as in test_queue_entries; a row computed twice or not at all is off by its whole norm
        assert ((out.double() - want).norm(dim=1) / want.norm(dim=1)).max().item() < 5e-5


def queue_time(pkg, dev, w, H, I, rows, hint):
    """us of one gate/up call, the best of five."""
    queue, off = [], 0
    for i, n in enumerate(rows):
        queue += [i, off, n]
        off += n
    queue = torch.tensor(queue, dtype=torch.int32, device=dev)
    x, gate = torch.randn(off, H, device=dev), torch.empty(off, I, device=dev)
    us = []
    for _ in range(6):
        t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        t0.record()
        pkg.moe_mlp1_swiglu(queue, 0, len(rows), x, gate, w["w_mlp1"], w["b_mlp1"], H, I, 2 * I * H, 2 * I, 1.702, 7.0, hint, 0)
        t1.record()
        torch.cuda.synchronize()
        us.append(t0.elapsed_time(t1) * 1e3)
    return min(us[1:])


def test_queue_time_follows_the_rows_and_not_the_longest_entry(pkg, wl, dev):
    """The same number of rows and of experts takes about the same time however they are spread over the entries: with a share
    of the compute units to each entry the uneven queue took ten times as long."""
    H, I, E = 2880, 2880, 32
    shape = wl.MoeShape("queue", T=1, H=H, I=I, E=E, K=1, fmt="bf16", seed=1)
    blk, _ = wl.make_device_layer(shape, pkg.normal_table(), dev)
    even = queue_time(pkg, dev, blk.tensors, H, I, [128] * E, 128)
    uneven = queue_time(pkg, dev, blk.tensors, H, I, [8] * (E - 1) + [128 * E - 8 * (E - 1)], 128 * E)
    print("queue times", even, uneven, flush=True)
    assert uneven < 3 * even


@pytest.mark.parametrize("rows,hint,limit", [([40] * 32, 1, 3.5), ([8] * 31 + [2048], 0, 1.5)], ids=["low", "unknown"])
def test_queue_time_under_a_hint_that_is_too_low(pkg, wl, dev, rows, hint, limit):
    """A hint below the row counts costs further passes over the weights, 32 rows each (two of them here, where one is enough
    with the right hint), not a pass per few rows; a hint of 0 says nothing and costs nothing."""
    shape = wl.MoeShape("queue", T=1, H=2880, I=2880, E=32, K=1, fmt="bf16", seed=1)
    blk, _ = wl.make_device_layer(shape, pkg.normal_table(), dev)
    right = queue_time(pkg, dev, blk.tensors, 2880, 2880, rows, max(rows))
    low = queue_time(pkg, dev, blk.tensors, 2880, 2880, rows, hint)
    print("queue times", right, low, flush=True)
    assert low < limit * right
