"""moe_block_forward inside a captured HIP graph: the entry allocates nothing, never synchronises and clears
its counters with kernels, so a serving loop may capture one call and replay it.  Every replay must return
the eager call's bits: replayed several times, with eager work on the same buffers and synchronisations
between the replays, for each kernel family the size rule can pick."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# T, H, I, E, K, fmt -> a handful of rows per expert / bucketing inside the expert kernels / bucketing launch + 64-token
# blocks / 128-token blocks (MXFP4) and 256-token blocks (bf16) / the three routers
FUSED = 32  # MOE_FLAG_FUSED_GEMM_LAUNCH: both expert GEMMs in one launch (counters cleared by a kernel)
CASES = [
    (64, 256, 128, 8, 4, "mxfp4"),
    (64, 256, 128, 8, 4, "bf16"),
    (64, 256, 128, 8, 4, "mxfp4", FUSED),
    (96, 320, 192, 16, 4, "bf16", FUSED),
    (300, 192, 128, 8, 1, "mxfp4"),
    (260, 320, 192, 4, 1, "bf16"),      # 65 rows per expert: one partial token block each
    (700, 320, 192, 8, 4, "bf16"),      # 350 rows per expert: a full and a partial token block each
    (700, 320, 192, 8, 4, "mxfp4"),
    (2100, 128, 64, 32, 2, "mxfp4"),    # T x E >= 65536: the two-pass router
    (1200, 128, 64, 128, 4, "mxfp4"),   # 4800 assignments, 37 rows per expert: bucketing launch + 64-token blocks
    (1200, 128, 64, 128, 4, "bf16"),
    (5, 256, 128, 16, 2, "mxfp4"),      # under one row per expert: a tile of weight rows per wave
    (5, 256, 128, 16, 2, "bf16"),
    (20, 320, 192, 64, 4, "mxfp4"),     # the same behind partial sums and finalize
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in c))
def test_graph_replays_equal_the_eager_call(pkg, wl, oracle, dev, case):
    T, H, I, E, K, fmt = case[:6]
    flags = case[6] if len(case) > 6 else 0
    assert FUSED == pkg.MOE_FLAG_FUSED_GEMM_LAUNCH
    shape = wl.MoeShape("graph", T=T, H=H, I=I, E=E, K=K, fmt=fmt, seed=5 + T)
    table = oracle.normal_table()
    blk, raw = wl.make_device_layer(shape, table, dev)
    x = wl.make_device_input(shape, table, dev)
    x_alt = x.flip(0).contiguous()
    e_agg = torch.empty((T, H), dtype=torch.float32, device=dev)
    ti = torch.empty((T, K), dtype=torch.int32, device=dev)
    tv = torch.empty((T, K), dtype=torch.float32, device=dev)
    x_in = x.clone()
    p = blk.params(x_in, e_agg, ti, tv, flags=flags)
    stream = torch.cuda.current_stream().cuda_stream
    print("graph", shape, blk.describe(p), flush=True)

    def eager(inp):
        x_in.copy_(inp)
        blk.launch(p, stream)
        torch.cuda.synchronize()
        return e_agg.clone(), ti.clone(), tv.clone()

    want = eager(x)
    want_alt = eager(x_alt)
    assert not torch.equal(want[0], want_alt[0])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        blk.launch(p, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    for rep in range(4):
        inp, ref = (x, want) if rep % 2 == 0 else (x_alt, want_alt)
        x_in.copy_(inp)
        e_agg.fill_(float("nan"))
        ti.fill_(-1)
        tv.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(ti, ref[1]) and torch.equal(tv, ref[2]), rep
        assert torch.equal(e_agg, ref[0]), rep
        # eager work on the same buffers between the replays
        got = eager(inp)
        assert torch.equal(got[0], ref[0])


@pytest.mark.parametrize("cases", [((256, 256, 128, 8, 4, "mxfp4"), (700, 320, 192, 8, 4, "bf16")),
                                   ((5, 256, 128, 16, 2, "mxfp4"), (20, 320, 192, 64, 4, "bf16"))], ids=["large", "small"])
def test_two_streams_do_not_share_state(pkg, wl, oracle, dev, cases):
    """Two calls with their own workspaces on two streams at once (default priority) give the bits each gives
    alone: the library keeps nothing between or across calls."""
    table = oracle.normal_table()
    jobs = []
    for T, H, I, E, K, fmt in cases:
        shape = wl.MoeShape("streams", T=T, H=H, I=I, E=E, K=K, fmt=fmt, seed=T)
        blk, raw = wl.make_device_layer(shape, table, dev)
        x = wl.make_device_input(shape, table, dev)
        out = (torch.empty((T, H), dtype=torch.float32, device=dev), torch.empty((T, K), dtype=torch.int32, device=dev),
               torch.empty((T, K), dtype=torch.float32, device=dev))
        p = blk.params(x, *out)
        blk.launch(p, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        jobs.append((blk, raw, x, p, out, [o.clone() for o in out]))
    streams = [torch.cuda.Stream(device=dev), torch.cuda.Stream(device=dev)]
    torch.cuda.synchronize()
    for _ in range(20):
        for (blk, raw, x, p, out, alone), st in zip(jobs, streams):
            for o in out:
                o.zero_()
        torch.cuda.synchronize()
        for _ in range(3):
            for (blk, raw, x, p, out, alone), st in zip(jobs, streams):
                blk.launch(p, st.cuda_stream)
        torch.cuda.synchronize()
        for blk, raw, x, p, out, alone in jobs:
            assert all(torch.equal(o, a) for o, a in zip(out, alone))


@pytest.mark.parametrize("fmt", ["bf16", "mxfp4"])
@pytest.mark.parametrize("rows", [[3, 0, 1, 2], [100, 0, 17, 300]], ids=["short", "long"])
def test_graph_replays_of_the_queue_entries(pkg, wl, dev, rows, fmt):
    """The work-queue entries in a captured graph, one assignment to a token (the atomic sums then have one term): the queue is
    read on the device, so replays follow what it holds."""
    H, I, E, A = 320, 192, len(rows), sum(rows)
    shape = wl.MoeShape("queue", T=A, H=H, I=I, E=E, K=1, fmt=fmt, seed=A)
    blk, _ = wl.make_device_layer(shape, pkg.normal_table(), dev)
    w = blk.tensors
    x = wl.make_device_input(shape, pkg.normal_table(), dev)
    tokens = torch.randperm(A, device=dev).int()
    weights = torch.rand(A, device=dev)
    gate, out = torch.empty(A, I, device=dev), torch.empty(A, H, device=dev)
    queues = []
    for order in (rows, rows[::-1]):
        off, q = 0, []
        for e, n in enumerate(order):
            q += [e, off, n]
            off += n
        queues.append(torch.tensor(q, dtype=torch.int32, device=dev))
    queue = queues[0].clone()

    def calls(stream):
        out.zero_()
        if fmt == "bf16":
            pkg.moe_mlp1_swiglu(queue, 0, E, x, gate, w["w_mlp1"], w["b_mlp1"], H, I, 2 * I * H, 2 * I, 1.702, 7.0, max(rows), 0,
                                stream=stream)
            pkg.moe_mlp2_scatter(queue, 0, E, gate, tokens, weights, out, w["w_mlp2"], w["b_mlp2"], I, H, I * H, H, max(rows), 0,
                                 stream=stream)
        else:
            pkg.moe_mlp1_swiglu_mxfp4(queue, 0, E, x, gate, w["w_mlp1"], w["w_mlp1_scales"], w["b_mlp1"], H, I, 2 * I, 1.702, 7.0,
                                      max(rows), 0, stream=stream)
            pkg.moe_mlp2_scatter_mxfp4(queue, 0, E, gate, tokens, weights, out, w["w_mlp2"], w["w_mlp2_scales"], w["b_mlp2"], I, H,
                                       H, max(rows), 0, stream=stream)

    def eager(q):
        queue.copy_(q)
        calls(None)
        torch.cuda.synchronize()
        return gate.clone(), out.clone()

    print("queue graph", rows, fmt, flush=True)
    want = [eager(q) for q in queues]
    assert not torch.equal(want[0][1], want[1][1])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        calls(torch.cuda.current_stream())
    for rep in range(4):
        queue.copy_(queues[rep % 2])
        gate.fill_(float("nan"))
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(gate, want[rep % 2][0]) and torch.equal(out, want[rep % 2][1]), rep
        assert torch.equal(eager(queues[rep % 2])[1], want[rep % 2][1])
