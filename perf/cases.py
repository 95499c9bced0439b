"""The work whose speed counts: calls of the MoE layer's public entry points over the range that a serving
or prefill program makes them in, on one GPU that owns some of the 256 experts.

`listed()` names the cases, `draw(rng)` gives more of the same ranges; `prepare` makes what a program holds
before the call (packed weights, scales and the batch), `run` is one call.  Two kinds:

  forward   the routed-expert layer: `ops.moe_forward` on weights packed once, or `moe_layer.run_custom`, the
            drop-in call that takes the unpacked weights and keeps its own packed copy
  producer  `ops.router_quant`, which makes the layer's logits and FP8 activations from bf16 hidden states

Routing is "even" (no bias: each expert gets its share), "uneven" (a bias ~N(0, 0.1), which at these logits
makes some experts many times as busy as others) or "skewed" (+3 on the first four local experts, which then
take most picks).  Values are "normal" (e4m3 of N(0, 1); scales as in the benchmark's configurations) or
"uniform" (e4m3 of U(-1, 1) and the scales of the layer's own input builder).
"""

import importlib
import math

import torch

moe_layer = importlib.import_module("15642_moe_amd.moe_layer")
ops = importlib.import_module("15642_moe_amd.ops")

H, I, E_GLOBAL, TOP_K, GROUPS, TOP_GROUPS, BLK = 7168, 2048, 256, 8, 8, 4, 128
FLOPS_PER_ROUTE = 2 * H * 2 * I + 2 * I * H
BYTES_PER_EXPERT = 3 * I * H + 4 * (2 * I // BLK * (H // BLK) + H // BLK * (I // BLK))
#: Batches below this are redrawn until they hold the local picks that such a batch has on average (at least
#: two): a rank that a small batch does not route to has nothing to do.
REDRAW_BELOW = 16


def _forward(name, T, routing, e_local=32, offset=0, entry="moe_forward", values="normal"):
    return {"name": name, "kind": "forward", "T": T, "routing": routing, "e_local": e_local, "offset": offset,
            "entry": entry, "values": values}


def listed():
    return [
        # One sequence decoding a token at a time: latency and launches.
        _forward("decode_T1", 1, "even"),
        # A small serving batch through the drop-in call, an odd number of sequences.
        _forward("dropin_T19", 19, "even", offset=64, entry="run_custom", values="uniform"),
        # The decode configuration of the benchmark: weights of about half the experts are streamed.
        _forward("decode_T64", 64, "uneven"),
        # A full serving batch of odd size: every expert is hit by a few tokens.
        _forward("decode_T113", 113, "even", offset=224),
        # A short prompt on a rank that owns 16 experts.
        _forward("prefill_T421_E16", 421, "even", e_local=16, offset=48),
        # The mid-prefill configuration of the benchmark.
        _forward("prefill_T1024", 1024, "uneven", offset=96),
        # A prompt of a few thousand tokens, ragged against every tile.
        _forward("prefill_T3001", 3001, "even", offset=160),
        # The routing stress of the benchmark: four experts take most of the work.
        _forward("skewed_T4096", 4096, "skewed"),
        # The large-prefill configuration of the benchmark.
        _forward("prefill_T8192", 8192, "uneven"),
        # The largest batch of the reference's own sweep, through the drop-in call.
        _forward("dropin_T16384", 16384, "even", entry="run_custom", values="uniform"),
        # The producer in front of a decode step, and of a large prefill.
        {"name": "producer_T77", "kind": "producer", "T": 77},
        {"name": "producer_T8192", "kind": "producer", "T": 8192},
    ]


def draw(rng):
    def size(most):
        return min(most, int(math.exp(rng.uniform(0.0, math.log(most + 1)))))

    if rng.random() < 0.25:
        return {"kind": "producer", "T": size(16384)}
    routing = rng.choice(("even", "even", "uneven", "uneven", "skewed"))
    e_local = rng.choice((8, 16, 32, 32))
    c = _forward("", size({"even": 16384, "uneven": 6000, "skewed": 4096}[routing]), routing, e_local=e_local,
                 offset=e_local * rng.randrange(E_GLOBAL // e_local),
                 entry=rng.choice(("moe_forward", "moe_forward", "moe_forward", "run_custom")),
                 values=rng.choice(("normal", "uniform")))
    del c["name"]
    return c


def _scores(logits):
    """The sigmoid as the layer defines it (the exponential in 64 bits, rounded to 32; add and divide in 32):
    the picks are whole numbers that follow from these values' order."""
    return 1.0 / (1.0 + torch.exp(-logits.double()).float())


def _picks(logits, bias):
    """The eight experts of each token (ascending), on the host: the two best scores of each of 8 groups make
    the group's score, the four best groups stay, and their eight best experts are taken; ties go to the lower
    index."""
    T = logits.shape[0]
    v = _scores(logits) + bias.float()
    best2 = v.view(T, GROUPS, -1).topk(2, dim=2).values
    kept = torch.sort(best2[..., 0] + best2[..., 1], dim=1, descending=True, stable=True).indices[:, :TOP_GROUPS]
    mask = torch.zeros(T, GROUPS, dtype=torch.bool).scatter_(1, kept, True).repeat_interleave(E_GLOBAL // GROUPS, 1)
    order = torch.sort(v.masked_fill(~mask, -math.inf), dim=1, descending=True, stable=True).indices
    return order[:, :TOP_K].sort(dim=1).values


def _routing(case, seed):
    """(logits [T, 256] fp32, bias [256] bf16, picks) on the host."""
    g = torch.Generator().manual_seed(seed)
    T, lo, n = case["T"], case["offset"], case["e_local"]
    bias = torch.zeros(E_GLOBAL)
    if case["routing"] == "uneven":
        bias = torch.randn(E_GLOBAL, generator=g) * 0.1
    elif case["routing"] == "skewed":
        bias[lo:lo + 4] = 3.0
    bias = bias.bfloat16()
    want = max(2, round(T * TOP_K * n / E_GLOBAL))
    for _ in range(400):
        logits = torch.randn(T, E_GLOBAL, generator=g)
        picks = _picks(logits, bias)
        local = int(((picks >= lo) & (picks < lo + n)).sum())
        if T >= REDRAW_BELOW or local == want or (case["routing"] != "even" and local >= 2):
            break
    return logits, bias, picks


def _inputs(case, seed):
    """The layer's ten inputs, on the GPU, in the layouts of its drop-in call."""
    T, n = case["T"], case["e_local"]
    logits, bias, _ = _routing(case, seed)
    g = torch.Generator(device="cuda").manual_seed(seed)
    normal = case["values"] == "normal"

    def e4m3(*shape):
        if normal:
            return torch.randn(*shape, generator=g, device="cuda").to(torch.float8_e4m3fn)
        return (torch.rand(*shape, generator=g, device="cuda") * 2 - 1).to(torch.float8_e4m3fn)

    def scale(lo, hi, *shape):
        return torch.rand(*shape, generator=g, device="cuda") * (hi - lo) + lo

    w13 = torch.empty((n, 2 * I, H), dtype=torch.float8_e4m3fn, device="cuda")
    w2 = torch.empty((n, H, I), dtype=torch.float8_e4m3fn, device="cuda")
    for e in range(n):
        w13[e] = e4m3(2 * I, H)
        w2[e] = e4m3(H, I)
    ws = (0.001, 0.01) if normal else (0.01, 0.11)
    return {
        "routing_logits": logits.cuda(),
        "routing_bias": bias.cuda(),
        "hidden_states": e4m3(T, H),
        "hidden_states_scale": scale(*((0.01, 0.05) if normal else (0.01, 0.11)), H // BLK, T),
        "gemm1_weights": w13,
        "gemm1_weights_scale": scale(*ws, n, 2 * I // BLK, H // BLK),
        "gemm2_weights": w2,
        "gemm2_weights_scale": scale(*ws, n, H // BLK, I // BLK),
        "local_expert_offset": case["offset"],
        "routed_scaling_factor": 2.5 if normal else 1.0,
    }


def _producer_inputs(case, seed):
    """bf16 hidden states as a residual stream after its norm has them (a few columns run hot), and a router."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    hot = torch.where(torch.rand(H, generator=g, device="cuda") < 0.002, 20.0, 1.0)
    x = (torch.randn(case["T"], H, generator=g, device="cuda") * hot).bfloat16()
    w = (torch.randn(E_GLOBAL, H, generator=g, device="cuda") * H ** -0.5).bfloat16()
    return x, w


def prepare(case, seed):
    if case["kind"] == "producer":
        x, w = _producer_inputs(case, seed)
        return {"call": ops.router_quant, "args": (x, ops.pack_router(w))}
    x = _inputs(case, seed)
    if case["entry"] == "run_custom":
        return {"call": moe_layer.run_custom, "args": (moe_layer._load_custom_ops(), *x.values())}
    return {"call": ops.moe_forward, "args": (
        x["hidden_states"], x["hidden_states_scale"], ops.pack_w13(x["gemm1_weights"]), x["gemm1_weights_scale"],
        ops.pack_w2(x["gemm2_weights"]), x["gemm2_weights_scale"], x["routing_logits"], x["routing_bias"].float(),
        x["routed_scaling_factor"], x["local_expert_offset"])}


def run(state):
    out = state["call"](*state["args"])
    if isinstance(out, tuple):  # the producer: its FP8 codes as the bytes they are
        logits, codes, scales = out
        return {"logits": logits, "codes": codes.view(torch.uint8), "scales": scales}
    return out


def work(case):
    T = case["T"]
    if case["kind"] == "producer":
        return {"bytes": T * (2 * H + H + H // BLK * 4 + E_GLOBAL * 4) + 2 * E_GLOBAL * H, "flops": 2 * T * H * E_GLOBAL}
    picks = _routing(case, 0)[2] - case["offset"]  # the counts of one batch; others of the case are close to it
    local = picks[(picks >= 0) & (picks < case["e_local"])]
    return {
        "bytes": int(local.unique().numel()) * BYTES_PER_EXPERT + T * (H + H // BLK * 4 + E_GLOBAL * 4 + 2 * H) + 4 * E_GLOBAL,
        "flops": int(local.numel()) * FLOPS_PER_ROUTE,
    }


def tolerance(case):
    if case["kind"] == "producer":  # codes and scales follow from 32-bit operations; the logits are 32-bit sums
        return {"rel": 1e-5, "max": 1e-4, "differ": 1e-5}
    # bf16 results, 0.002 from the 64-bit ones: another order of the 32-bit sums in front of the FP8
    # requantisation moves a code in a thousand by one step.
    return {"rel": 8e-3, "max": 0.05}


def exact(case, seed):
    if case["kind"] == "producer":
        x, w = _producer_inputs(case, seed)
        blocks = x.float().view(-1, H // BLK, BLK)
        scale = (blocks.abs().amax(2) / 448.0).clamp_min(1e-8)
        codes = (blocks / scale[:, :, None]).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
        return {"logits": x.double() @ w.double().t(), "codes": codes.view(-1, H).view(torch.uint8),
                "scales": (blocks.double().abs().amax(2) / 448.0).clamp_min(1e-8).t().contiguous()}
    x = _inputs(case, seed)
    picks = _routing(case, seed)[2].cuda()
    s = _scores(x["routing_logits"].cpu()).cuda().double().gather(1, picks)
    weights = s / (s.sum(1, keepdim=True) + 1e-20) * x["routed_scaling_factor"]

    def rows(t, scale):  # [n, K] e4m3 with [n, K / 128] scales, in 64 bits
        return t.float().double() * scale.double().repeat_interleave(BLK, 1)

    out = torch.zeros((case["T"], H), dtype=torch.float64, device="cuda")
    for e in range(case["e_local"]):
        tok, k = torch.nonzero(picks == case["offset"] + e, as_tuple=True)
        if not tok.numel():
            continue
        w13 = rows(x["gemm1_weights"][e], x["gemm1_weights_scale"][e].repeat_interleave(BLK, 0))
        a = x["hidden_states"].view(torch.uint8)[tok].view(torch.float8_e4m3fn)
        g = rows(a, x["hidden_states_scale"].t()[tok]) @ w13.t()
        c = (g[:, I:] * torch.sigmoid(g[:, I:]) * g[:, :I]).view(-1, I // BLK, BLK)
        cs = (c.abs().amax(2) / 448.0).clamp_min(1e-8)  # the layer's own FP8 requantisation, a part of its result
        cq = (c / cs[:, :, None]).clamp(-448.0, 448.0).float().to(torch.float8_e4m3fn).view(-1, I)
        w2 = rows(x["gemm2_weights"][e], x["gemm2_weights_scale"][e].repeat_interleave(BLK, 0))
        out.index_add_(0, tok, (rows(cq, cs) @ w2.t()) * weights[tok, k][:, None])
    return out
