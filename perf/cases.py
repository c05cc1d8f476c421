"""Timed cases of the block-scaled FP8 path.

Each case is work that a program using this package has it do, called through
``akas_amd.ops`` and ``akas_amd.moe``: dense FP8 linears from one row to a
long prompt, the RMSNorm that feeds them, and the routed and shared-expert
MoE blocks from a few tokens to a long prompt.  Decode steps run as the HIP
graph that a decode program captures once and replays per token; prompts of
every length are called eagerly, since no two are alike.

A case names its kind:
- ``linear``: one ``fp8_linear`` on unquantized activations;
- ``decode``: the dense projections of several layers in one graph, each with
  its own weights (more than the last-level cache holds at the listed sizes)
  and its own activations;
- ``norm``: ``rms_quantize`` and the prequantized linear behind it;
- ``moe``: ``routed_moe``, eager or as a graph;
- ``shared``: ``shared_expert_moe``.
"""

import math

import torch

BLOCK = 128
_DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_SIZE = {"f32": 4, "f16": 2, "bf16": 2}


def listed():
    return [
        # A single small projection on one request, float32 in and out: what
        # one call costs when there is next to nothing to compute.
        dict(name="linear_small", kind="linear", m=3, k=2048, n=512, x="f32", out="f32",
             scales="f32"),
        # The dense projections of a single-stream decode step.
        dict(name="decode_1", kind="decode", m=1, h=2048, layers=6, out="bf16", scales="f32"),
        # The same for a batch of 40 streams, scales as checkpoints hold them.
        dict(name="decode_40", kind="decode", m=40, h=2048, layers=6, out="bf16", scales="bf16"),
        # A short prompt, or a chunk of a long one.
        dict(name="linear_chunk", kind="linear", m=300, k=2048, n=6144, x="bf16", out="bf16",
             scales="f32"),
        # A down projection (deep product) over a prompt of a thousand tokens.
        dict(name="linear_prompt", kind="linear", m=1000, k=8192, n=2048, x="bf16", out="bf16",
             scales="bf16"),
        # A batch of long prompts.
        dict(name="linear_prefill", kind="linear", m=8192, k=2048, n=8192, x="bf16", out="bf16",
             scales="f32"),
        # Norm, quantizer and input projection of a 2049-token prompt.
        dict(name="norm_prompt", kind="norm", m=2049, k=2048, n=6144, x="bf16", out="bf16",
             scales="bf16"),
        # The MoE block for a handful of streams: sigmoid router with bias,
        # float32 intermediates.
        dict(name="moe_few", kind="moe", t=5, h=2048, f=1536, e=64, top=4, router="sigmoid",
             policy="f32", zipf=False, packed=False, graph=False, scales="bf16"),
        # A decode step over 256 streams.
        dict(name="moe_decode", kind="moe", t=256, h=2048, f=1536, e=64, top=4, router="softmax",
             policy="bf16", zipf=False, packed=False, graph=True, scales="f32"),
        # A prompt of 1500 tokens.
        dict(name="moe_prompt", kind="moe", t=1500, h=2048, f=1536, e=64, top=4,
             router="softmax", policy="bf16", zipf=False, packed=False, graph=False,
             scales="bf16"),
        # Eight prompts of 2048 tokens with skewed routing.
        dict(name="moe_prefill", kind="moe", t=16384, h=2048, f=1536, e=64, top=4,
             router="softmax", policy="bf16", zipf=True, packed=False, graph=False,
             scales="f32"),
        # Many narrow experts and a shared one, 64 streams.
        dict(name="shared_decode", kind="shared", t=64, h=2048, f=512, e=256, top=8,
             scales="f32"),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more case of the listed ranges, no larger than the listed ones."""
    kind = rng.choice(["linear", "linear", "linear", "decode", "norm", "moe", "moe", "shared"])
    scales = rng.choice(["f32", "bf16"])
    if kind == "decode":
        return dict(kind=kind, m=_log(rng, 1, 256), h=rng.choice([1024, 1536, 2048]),
                    layers=rng.randint(2, 6), out=rng.choice(["bf16", "f16", "f32"]),
                    scales=scales)
    if kind == "shared":
        return dict(kind=kind, t=_log(rng, 1, 2048), h=rng.choice([1024, 2048]), f=512,
                    e=rng.choice([64, 128, 256]), top=rng.choice([4, 8]), scales=scales)
    if kind == "moe":
        h, f, e, top = rng.choice([(2048, 1536, 64, 4), (1024, 512, 32, 4), (1536, 768, 64, 2),
                                   (2048, 512, 128, 8)])
        packed = rng.random() < 0.25
        return dict(kind=kind, t=_log(rng, 1, 12000), h=h, f=f, e=e, top=top,
                    router=rng.choice(["sigmoid", "softmax"]),
                    policy=rng.choice(["f32", "bf16", "bf16"]), zipf=rng.random() < 0.5,
                    packed=packed, graph=rng.random() < 0.3, scales=scales)
    k = rng.choice([512, 1024, 1536, 2048, 2048, 4096, 8192, BLOCK * rng.randint(3, 64)])
    n = rng.choice([512, 2048, 2048, 6144, 8192, BLOCK * rng.randint(2, 64),
                    16 * rng.randint(16, 512)])
    m = min(_log(rng, 1, 8192), (1 << 37) // (k * n))
    if kind == "norm":
        return dict(kind=kind, m=m, k=k, n=n, x=rng.choice(["bf16", "f32"]),
                    out=rng.choice(["bf16", "f32"]), scales=scales)
    return dict(kind=kind, m=m, k=k, n=n, x=rng.choice(["bf16", "bf16", "f16", "f32"]),
                out=rng.choice(["bf16", "bf16", "f16", "f32"]), scales=scales)


# ---------------------------------------------------------------------------
# inputs: made from the seed alone, in plain torch
# ---------------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1_000_003 * int(seed) + 17)
    return g


def _weight(g, shape, scales):
    """Block-FP8 weights ``[..., n, k]`` ~N(0, 0.02): e4m3 codes (as bytes)
    and their 128x128 block scales."""
    *lead, n, k = shape
    nb = -(-n // BLOCK)
    codes = torch.empty(shape, dtype=torch.uint8, device="cuda")
    out = torch.empty((*lead, nb, k // BLOCK), dtype=_DT[scales], device="cuda")
    flat_c, flat_s = codes.view(-1, n, k), out.view(-1, nb, k // BLOCK)
    step = max(1, (1 << 27) // (n * k))
    for i in range(0, flat_c.shape[0], step):
        count = min(step, flat_c.shape[0] - i)
        w = torch.zeros((count, nb * BLOCK, k), device="cuda")
        w[:, :n] = torch.randn((count, n, k), generator=g, device="cuda") * 0.02
        blocks = w.view(count, nb, BLOCK, k // BLOCK, BLOCK)
        s = (blocks.abs().amax((2, 4)).clamp_min(1e-12) / 448.0).to(_DT[scales])
        q = (blocks / s.float()[:, :, None, :, None]).clamp_(-448.0, 448.0)
        q = q.to(torch.float8_e4m3fn).view(torch.uint8).view(count, nb * BLOCK, k)
        flat_c[i:i + count] = q[:, :n]
        flat_s[i:i + count] = s
    return codes, out


def _activations(g, shape, dtype):
    """~N(0, 1) with one value in a hundred twenty times as large."""
    x = torch.randn(shape, generator=g, device="cuda")
    x = torch.where(torch.rand(shape, generator=g, device="cuda") < 0.01, 20.0 * x, x)
    return x.to(_DT[dtype])


def _decode_shapes(h):
    """(k, n) of a layer's dense projections: input, output, up and down."""
    return [(h, 3 * h), (h, h), (h, 4 * h), (4 * h, h)]


def _inputs(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind == "linear":
        return dict(x=_activations(g, (case["m"], case["k"]), case["x"]),
                    w=_weight(g, (case["n"], case["k"]), case["scales"]))
    if kind == "norm":
        return dict(x=_activations(g, (case["m"], case["k"]), case["x"]),
                    norm=1.0 + 0.1 * torch.randn(case["k"], generator=g, device="cuda"),
                    w=_weight(g, (case["n"], case["k"]), case["scales"]))
    if kind == "decode":
        return dict(linears=[(_activations(g, (case["m"], k), "bf16"),
                              *_weight(g, (n, k), case["scales"]))
                             for _ in range(case["layers"]) for k, n in _decode_shapes(case["h"])])
    t, h, f, e = case["t"], case["h"], case["f"], case["e"]
    bank = [_weight(g, shape, case["scales"]) for shape in ((e, f, h), (e, f, h), (e, h, f))]
    x = torch.randn((t, h), generator=g, device="cuda").to(torch.bfloat16)
    logits = torch.randn((t, e), generator=g, device="cuda")
    if kind == "shared":
        own = [_weight(g, shape, case["scales"]) for shape in ((f, h), (f, h), (h, f))]
        gate = torch.randn(t, generator=g, device="cuda").to(torch.bfloat16)
        return dict(x=x, logits=logits, bank=bank, own=own, gate=gate)
    if case["zipf"]:
        rank = torch.randperm(e, generator=g, device="cuda").float()
        logits = logits - 1.1 * torch.log1p(rank)
    bias = None
    if case["router"] == "sigmoid":
        bias = 0.1 * torch.randn(e, generator=g, device="cuda")
    return dict(x=x, logits=logits, bank=bank, bias=bias)


# ---------------------------------------------------------------------------
# what a program holds, and one pass
# ---------------------------------------------------------------------------

def _captured(call):
    """``call`` as a graph (warmed up once on the capture's stream) and its
    outputs' buffers."""
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        call()
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        outputs = call()
    return graph, outputs


def prepare(case, seed):
    from akas_amd import moe, ops

    state = dict(case=case, **_inputs(case, seed))
    kind = case["kind"]
    if kind in ("moe", "shared"):
        (w1, s1), (w3, s3), (w2, s2) = state.pop("bank")
        state["experts"] = moe.ExpertWeights(w1, s1, w3, s3, w2, s2)
    if kind == "shared":
        (w1, s1), (w3, s3), (w2, s2) = state.pop("own")
        state["shared"] = moe.SharedExpert(w1, s1, w3, s3, w2, s2)
    if kind == "decode":
        # a decode program owns its activations' buffers and one workspace
        m, dtype = case["m"], _DT[case["out"]]
        outs = [torch.empty((m, w.shape[0]), dtype=dtype, device="cuda")
                for _, w, _ in state["linears"]]
        largest = max((ops.linear_workspace(m, w.shape[1], w.shape[0], "cuda").numel()
                       for _, w, _ in state["linears"]))
        state["workspace"] = torch.empty(largest, dtype=torch.uint8, device="cuda")

        def step():
            for (x, w, s), out in zip(state["linears"], outs):
                ops.fp8_linear(x, w, s, out=out, workspace=state["workspace"])
            return outs

        state["graph"] = _captured(step)
    if kind == "moe" and case["graph"]:
        state["graph"] = _captured(lambda: _block(state))
    return state


def _block(state):
    from akas_amd import moe

    case = state["case"]
    dtype = _DT[case["policy"]]
    return moe.routed_moe(
        state["x"], state["logits"], state["bias"], state["experts"], top=case["top"],
        router="biased_router" if case["router"] == "sigmoid" else "biased_softmax_router",
        packed=case["packed"], max_block_m=128 if case["packed"] else 64, product_dtype=dtype,
        activation_dtype=dtype, contribution_dtype=dtype)


def run(state):
    from akas_amd import moe, ops

    case = state["case"]
    if "graph" in state:
        graph, outputs = state["graph"]
        graph.replay()
        return outputs
    if case["kind"] == "linear":
        return ops.fp8_linear(state["x"], *state["w"], out_dtype=_DT[case["out"]])
    if case["kind"] == "norm":
        codes, scales, normalized = ops.rms_quantize(state["x"], state["norm"], eps=1e-5)
        y = ops.fp8_linear(codes, *state["w"], activation_scales=scales,
                           out_dtype=_DT[case["out"]])
        return codes, scales, normalized, y
    if case["kind"] == "moe":
        return _block(state)
    return moe.shared_expert_moe(state["x"], state["logits"], state["gate"], state["experts"],
                                 state["shared"], top=case["top"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _linear_bytes(m, k, n, case, x_bytes):
    weights = n * k + _SIZE[case["scales"]] * -(-n // BLOCK) * (k // BLOCK)
    return weights + x_bytes * m * k + _SIZE[case["out"]] * m * n


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=_linear_bytes(m, k, n, case, _SIZE[case["x"]]), flops=2 * m * k * n)
    if kind == "norm":
        # the codes, their scales and the normalized rows are outputs too
        m, k, n = case["m"], case["k"], case["n"]
        extra = m * k * (1 + 2) + 4 * m * (k // BLOCK) + 4 * k
        return dict(bytes=_linear_bytes(m, k, n, case, _SIZE[case["x"]]) + extra,
                    flops=2 * m * k * n)
    if kind == "decode":
        shapes, m = _decode_shapes(case["h"]), case["m"]
        return dict(bytes=case["layers"] * sum(_linear_bytes(m, k, n, case, 2) for k, n in shapes),
                    flops=case["layers"] * sum(2 * m * k * n for k, n in shapes))
    # MoE: the weights of the experts that the tokens reach (their expected
    # number under uniform routing), tokens and logits in, float32 rows out
    t, h, f, e, top = case["t"], case["h"], case["f"], case["e"], case["top"]
    reached = e * (1.0 - (1.0 - top / e) ** t) + (kind == "shared")
    per_expert = 3 * f * h * (1 + _SIZE[case["scales"]] / (BLOCK * BLOCK))
    ranks = top + (kind == "shared")
    return dict(bytes=int(reached * per_expert + t * (2 * h + 4 * e + 4 * h)),
                flops=6 * t * ranks * f * h)


def tolerance(case):
    """About four times the distance to the float64 result (``exact``)."""
    if case["kind"] in ("moe", "shared"):
        # a rounding that falls the other way in an intermediate (its dtype,
        # then its e4m3 code) reaches the output as one code step of one value
        return {"rel": 8e-3}
    if case["kind"] == "norm":
        # a normalized value on the other side of a bf16 rounding boundary
        # takes the neighbouring code
        return {"rel": 8e-3 if case["out"] == "bf16" else 7e-3, "differ": 2e-3}
    # f32: the FP8 matrix instruction's own sum of 128 products
    return {"rel": {"f32": 1.2e-4, "f16": 1e-3, "bf16": 7e-3}[case["out"]]}


# ---------------------------------------------------------------------------
# the same results in plain float64
# ---------------------------------------------------------------------------

def _codes(x):
    """1x128 e4m3 codes (as bytes) and float32 scales of ``x``: the format's
    float32 equations."""
    groups = x.float().view(*x.shape[:-1], -1, BLOCK)
    largest = groups.abs().amax(-1).clamp_min(1e-12)
    s = largest / torch.full_like(largest, 448.0)  # by a tensor: a true division
    q = (groups / s[..., None]).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn)
    return q.view(torch.uint8).view(x.shape), s


def _values(codes, s):
    q = codes.view(torch.float8_e4m3fn).float().double()
    return (q.view(*s.shape, BLOCK) * s.double()[..., None]).view(codes.shape)


def _weight_values(codes, s):
    n, k = codes.shape
    full = s.double().repeat_interleave(BLOCK, 0)[:n].repeat_interleave(BLOCK, 1)
    return codes.view(torch.float8_e4m3fn).float().double() * full


def _experts_exact(x, ids, bank, policy):
    """[t, top, h] contributions of the routed experts, intermediates rounded
    as the policy says."""
    dtype = _DT[policy]
    source = _values(*_codes(x))
    (w1, s1), (w3, s3), (w2, s2) = bank
    out = torch.zeros((*ids.shape, x.shape[1]), dtype=torch.float64, device="cuda")
    for e in range(w1.shape[0]):
        row, rank = torch.nonzero(ids == e, as_tuple=True)
        if not row.numel():
            continue
        rows = source[row]
        gate = (rows @ _weight_values(w1[e], s1[e]).T).float().to(dtype).double()
        up = (rows @ _weight_values(w3[e], s3[e]).T).float().to(dtype).double()
        act = (gate * torch.sigmoid(gate) * up).float().to(dtype)
        out[row, rank] = _values(*_codes(act)) @ _weight_values(w2[e], s2[e]).T
    return out


def exact(case, seed):
    given = _inputs(case, seed)
    kind = case["kind"]
    if kind == "linear":
        return _values(*_codes(given["x"])) @ _weight_values(*given["w"]).T
    if kind == "decode":
        return [_values(*_codes(x)) @ _weight_values(w, s).T for x, w, s in given["linears"]]
    if kind == "norm":
        x = given["x"].double()
        y = x / torch.sqrt(x.square().mean(-1, keepdim=True) + 1e-5) * given["norm"].double()
        codes, scales = _codes(y.float().to(torch.bfloat16))
        return codes, scales, y, _values(codes, scales) @ _weight_values(*given["w"]).T
    top, logits = case["top"], given["logits"]
    if kind == "shared":
        logits = logits.to(torch.bfloat16).double()
        picked, ids = logits.sort(dim=-1, descending=True, stable=True)
        picked, ids = picked[:, :top], ids[:, :top]
        p = torch.softmax(picked, -1)
        parts = _experts_exact(given["x"], ids, given["bank"], "f32")
        own = [(w[None], s[None]) for w, s in given["own"]]
        shared = _experts_exact(given["x"], torch.zeros_like(ids[:, :1]), own, "f32")[:, 0]
        parts, shared = (v.float().to(torch.bfloat16).double() for v in (parts, shared))
        gate = torch.sigmoid(given["gate"].double())[:, None]
        return (parts * p[..., None]).sum(1) + shared * gate
    if case["router"] == "sigmoid":
        score = torch.sigmoid(logits.double())
        ids = (score + given["bias"].double()).topk(top, -1).indices
        p = score.gather(1, ids)
        p = p / (p.sum(-1, keepdim=True) + 1e-6)
    else:
        ids = logits.topk(top, -1).indices
        p = torch.softmax(logits.double().gather(1, ids), -1)
    parts = _experts_exact(given["x"], ids, given["bank"], case["policy"])
    parts = parts.float().to(_DT[case["policy"]]).double()
    return (parts * p[..., None]).sum(1)
