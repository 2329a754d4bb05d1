"""The work that is timed: MoE blocks of the two model shapes this package exists for, through its public entry points.

Shapes are those of workloads.py: hidden = intermediate = 2880, top-4 of 32 experts ("20b") or of 128 ("120b"), MXFP4
experts as the checkpoints hold them or bf16 experts as the dense route holds them.  Values come from the package's own
generators (activations N(0,1) as an RMSNorm leaves them, weights N(0, 0.02), uniformly drawn MXFP4 codes with scale
exponents -8..0), all of them made from the seed on the device.  Four ways in:

  block    MoeBlock.forward: router, top-k, experts and combine of one layer
  stack    forward_layers: the MoE halves of consecutive layers, residual stream and norms between them included
  calls    one layer issued call by call under the reference-named entries, in the order of the layer loop they replace
  load     a layer's MXFP4 expert tensors from the checkpoint layout into a layout the kernels read
"""
import importlib

import torch

pkg = importlib.import_module("gpt-oss-amd_amd")
workloads = importlib.import_module("gpt-oss-amd_amd.workloads")

DIM, TOP = 2880, 4  # hidden size and expert intermediate size; experts per token


def case(kind, tokens=0, experts=32, fmt="mxfp4", zipf=0.0, layers=1, to="", name=None):
    c = {"kind": kind, "tokens": tokens, "experts": experts, "fmt": fmt, "zipf": zipf, "layers": layers, "to": to}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one user generating: a single token per step
        case("block", 1, name="decode1_mxfp4"),
        # a handful of concurrent users on the dense checkpoint route
        case("block", 7, fmt="bf16", name="decode7_bf16"),
        # a small ragged batch on the larger model: about one row per expert, some experts without any
        case("block", 33, experts=128, name="decode33_120b_mxfp4"),
        # a full decode batch, dense and MXFP4 experts (the benchmark's two decode blocks)
        case("block", 256, fmt="bf16", name="decode256_bf16"),
        case("block", 256, name="decode256_mxfp4"),
        # the larger model's layers one after the other at a large decode batch (the benchmark's stack, four of its layers)
        case("stack", 1024, experts=128, layers=4, name="stack1024_120b_mxfp4"),
        # one prompt of ordinary length, expert load skewed
        case("block", 1000, zipf=1.2, name="prefill1000_mxfp4"),
        # a prefill chunk with skewed expert load, and the same size on the dense route
        case("block", 4096, zipf=1.2, name="prefill4096_mxfp4"),
        case("block", 4096, fmt="bf16", name="prefill4096_bf16"),
        # the largest: prompts of several users prefilled together
        case("block", 16384, name="prefill16384_mxfp4"),
        # a host loop that keeps the reference's call sites, at its decode batch
        case("calls", 256, fmt="bf16", name="calls256_bf16"),
        # loading one layer of a MXFP4 checkpoint
        case("load", to="tiled", name="load_20b"),
    ]


def draw(rng):
    kind = rng.choice(["block"] * 6 + ["stack", "calls", "calls", "load"])
    experts = rng.choice([32, 32, 128])
    fmt = rng.choice(["mxfp4", "mxfp4", "bf16"])

    def tokens(most):  # spread over the logarithm of the range, any whole number (a single token is a listed case)
        return max(2, min(most, int(round(2 ** rng.uniform(0.6, most.bit_length() - 1 + 0.01)))))

    if kind == "block":
        return case("block", tokens(16384 if fmt == "mxfp4" else 4096), experts, fmt, rng.choice([0.0, 0.0, round(rng.uniform(0.5, 1.5), 2)]))
    if kind == "stack":
        return case("stack", tokens(1024), experts, fmt, layers=rng.randint(2, 4))
    if kind == "calls":
        return case("calls", tokens(2048), experts, fmt)
    # a shard of the layer's experts, or all of them
    return case("load", experts=rng.randint(2, 64), to=rng.choice(["tiled", "tiled", "bf16"]))


_table = None


def table():
    global _table
    if _table is None:
        _table = pkg.normal_table()
    return _table


def prepare(case, seed):
    dev = torch.device("cuda")
    T, E = case["tokens"], case["experts"]
    shape = workloads.MoeShape(case["kind"], T=T, H=DIM, I=DIM, E=E, K=TOP, fmt=case["fmt"], zipf_s=case["zipf"],
                               layers=case["layers"], seed=seed)
    s = {"case": case}
    if case["kind"] == "load":
        raw = {}
        for n, (dims, kind, args) in workloads.tensor_specs(shape).items():
            if n.endswith("_blocks") or n.endswith("_scales"):
                raw[n] = workloads.fill_device(dims, kind, args, seed, None, dev)
        s["raw"] = raw
        return s
    x = workloads.make_device_input(shape, table(), dev)
    if case["kind"] == "block":
        s["block"], _ = workloads.make_device_layer(shape, table(), dev)
        s["t"] = x
        return s
    # the residual stream, larger than what one layer adds to it, as between the layers of a deep model
    s["x0"], s["x"] = x * 4096.0, torch.empty_like(x)
    if case["kind"] == "stack":
        s["stack"] = workloads.DeviceStack(shape, table(), dev)
        s["stack"].prepare(s["x"])
        return s
    blk, s["raw"] = workloads.make_device_layer(shape, table(), dev)
    s["weights"] = blk.tensors
    # the buffers such a host loop holds for its largest batch
    A = T * TOP
    f32 = lambda *d: torch.empty(d, dtype=torch.float32, device=dev)  # noqa: E731
    i32 = lambda *d: torch.empty(d, dtype=torch.int32, device=dev)  # noqa: E731
    s.update(t=f32(T, DIM), rms=torch.ones(DIM, dtype=torch.bfloat16, device=dev), scores=f32(T, E), topk_v=f32(T, TOP),
             topk_i=i32(T, TOP), offsets=i32(E + 1), tokens_flat=i32(A), weights_flat=f32(A), by_expert=f32(A, DIM),
             gate=f32(A, DIM), queue=i32(3 * E), count=i32(1), e_agg=torch.zeros(T, DIM, device=dev),
             scratch=torch.empty(pkg.lib.moe_router_scratch_bytes(T, E), dtype=torch.uint8, device=dev))
    return s


def run(s):
    c = s["case"]
    if c["kind"] == "block":
        return s["block"].forward(s["t"])
    if c["kind"] == "stack":
        s["x"].copy_(s["x0"])  # the step's residual stream, updated in place by the layers
        s["stack"].forward()
        return s["x"], s["stack"].topk_i[0]
    if c["kind"] == "load":
        raw, out = s["raw"], []
        for n in ("w_mlp1", "w_mlp2"):
            if c["to"] == "tiled":
                out += pkg.mxfp4_repack(raw[n + "_blocks"], raw[n + "_scales"])
            else:
                out.append(pkg.dequant_mxfp4(raw[n + "_blocks"], raw[n + "_scales"]))
        return out
    return calls(s, c["tokens"], c["experts"], c["fmt"])


def calls(s, T, E, fmt):
    w, A = s["weights"], T * TOP
    s["x"].copy_(s["x0"])
    pkg.rmsnorm(s["t"], s["x"], s["rms"], T, DIM)
    pkg.gemm_router(s["scores"], s["t"], w["w_router"], w["b_router"], T, DIM, E, scratch=s["scratch"])
    pkg.topk(s["topk_v"], s["topk_i"], s["scores"], T, E, TOP)
    pkg.softmax(s["topk_v"], T, TOP)
    pkg.bucket_by_expert(s["topk_i"], s["topk_v"], T, TOP, E, s["offsets"], s["tokens_flat"], s["weights_flat"])
    pkg.gather_rows(s["t"], s["tokens_flat"], s["by_expert"], A, DIM)
    pkg.build_work_queue(s["offsets"], E, s["queue"], s["count"])
    n = int(s["count"].item())  # the layer loop reads the queue length back before it launches the experts
    if fmt == "bf16":
        pkg.moe_mlp1_swiglu(s["queue"], 0, n, s["by_expert"], s["gate"], w["w_mlp1"], w["b_mlp1"], DIM, DIM,
                            2 * DIM * DIM, 2 * DIM, 1.702, 7.0, T, 0)
        pkg.moe_mlp2_scatter(s["queue"], 0, n, s["gate"], s["tokens_flat"], s["weights_flat"], s["e_agg"], w["w_mlp2"],
                             w["b_mlp2"], DIM, DIM, DIM * DIM, DIM, T, 0)
    else:
        pkg.moe_mlp1_swiglu_mxfp4(s["queue"], 0, n, s["by_expert"], s["gate"], w["w_mlp1"], w["w_mlp1_scales"],
                                  w["b_mlp1"], DIM, DIM, 2 * DIM, 1.702, 7.0, T, 0)
        pkg.moe_mlp2_scatter_mxfp4(s["queue"], 0, n, s["gate"], s["tokens_flat"], s["weights_flat"], s["e_agg"],
                                   w["w_mlp2"], w["w_mlp2_scales"], w["b_mlp2"], DIM, DIM, DIM, T, 0)
    pkg.vecadd_and_zero(s["x"], s["e_agg"], 1.0, T, DIM)  # leaves e_agg zero for the next pass
    return s["x"], s["gate"], s["topk_i"], s["topk_v"]


def work(case):
    T, E, L = case["tokens"], case["experts"], case["layers"]
    elements = 3 * DIM * DIM  # expert weights of one expert
    packed = elements // 2 + elements // 32
    if case["kind"] == "load":
        return {"bytes": E * (packed + (packed if case["to"] == "tiled" else 2 * elements)), "flops": 0}
    per_expert = (packed if case["fmt"] == "mxfp4" else 2 * elements) + 3 * DIM * 2
    used = E * (1 - (1 - TOP / E) ** T)  # experts that get a row, on average
    router = E * DIM * 2 + E * 2
    # the block's input and output rows; a stack's residual stream is read and written as well
    return {"bytes": L * (used * per_expert + router + 2 * T * DIM * 4), "flops": L * 2 * T * (TOP * elements + E * DIM)}


def tolerance(case):
    if case["kind"] == "load":
        return "exact"
    # bf16 operands of both expert products (activations, SwiGLU outputs), fp32 sums: against the same block in 64 bits
    # 2.6e-3 (bf16 experts) and 6.3e-3 (MXFP4 experts), largest difference 0.017 and 0.047 of the rms; with the sums in
    # another order 4e-5 and 0.002.  Expert indices are whole numbers, decided by scores that every route computes exactly.
    if case["kind"] == "stack":
        # a layer's input carries the differences of the layers before it, so a token in a few thousand may take
        # another fourth expert there (inputs off by 1e-4: 2e-2)
        return {"rel": 2e-2, "max": 0.5}
    return {"rel": 1e-2, "max": 0.1}
