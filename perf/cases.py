"""Performance cases of the paged fused-MoE layer call.

A case is one shape of work a serving program has a MoE layer do through
``WispMoEState`` / ``WispMoEStateFP8``: ``steps`` layer calls of ``tokens``
tokens each, on a state whose expert masters sit in pinned host memory and
whose scratch holds ``cap`` experts.  ``cap == experts`` is a layer whose
experts are all in HBM; a smaller one pages.  Shapes are the ones of
``wisp_amd.workloads`` (the fp32 toy layer, a Qwen3-30B-A3B layer, a
Mixtral-8x7B layer, the block-FP8 Qwen3 layer).
"""
from __future__ import annotations

import math

import torch

from wisp.integrations.vllm.fused_moe import WispMoEState
from wisp.integrations.vllm.fused_moe_fp8 import Fp8SlabLayout, WispMoEStateFP8
from wisp_amd.workloads import FP8_BLOCK, SHAPES, block_quant_fp8, slab_views

WEIGHT_STD = 0.02


def _case(name, layer, dtype, tokens, cap, steps, routing, logits="bf16"):
    return {"name": name, "layer": layer, "dtype": dtype, "tokens": tokens, "cap": cap,
            "steps": steps, "routing": routing, "logits": logits}


def listed():
    return [
        # Smallest calls: one token through a small fp32 layer that pages
        # (launches and host work are all there is).
        _case("toy-f32-decode-paged", "toy", "f32", 1, 4, 16, "uniform", "f32"),
        # bs=1 generation with an 8-expert scratch, routing that repeats and
        # favours some experts: paging over the host link sets the rate.
        _case("qwen3-decode-paged", "qwen3", "bf16", 1, 8, 24, "trace", "f32"),
        # bs=1 generation with every expert in HBM.
        _case("qwen3-decode-resident", "qwen3", "bf16", 1, 128, 8, "uniform"),
        # The block-FP8 layer at its default cap, bs=1.
        _case("qwen3-fp8-decode-paged", "qwen3", "fp8", 1, 24, 24, "trace"),
        # A few users at once, a ragged number of them.
        _case("qwen3-batch7-resident", "qwen3", "bf16", 7, 128, 4, "uniform"),
        _case("mixtral-batch6-resident", "mixtral", "bf16", 6, 8, 1, "uniform"),
        # Batched generation.
        _case("qwen3-batch32-resident", "qwen3", "bf16", 32, 128, 2, "uniform"),
        # Prompt chunks: an ordinary one, large ones, one that pages.
        _case("qwen3-prefill512-resident", "qwen3", "bf16", 512, 128, 1, "uniform"),
        _case("qwen3-prefill8192-resident", "qwen3", "bf16", 8192, 128, 1, "uniform"),
        _case("mixtral-prefill1000-resident", "mixtral", "bf16", 1000, 8, 1, "uniform"),
        _case("qwen3-fp8-prefill4096-resident", "qwen3", "fp8", 4096, 128, 1, "uniform"),
        _case("qwen3-prefill96-paged", "qwen3", "bf16", 96, 24, 1, "uniform"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the listed ranges: the same layers, data types and
    modes at other token counts and caps."""
    kind = rng.choice(["toy", "decode-paged", "fp8-decode-paged", "batch", "batch", "fp8-batch",
                       "mixtral-batch", "prefill", "prefill", "fp8-prefill", "mixtral-prefill",
                       "prefill-paged"])
    logits = rng.choice(["bf16", "f32"])
    if kind == "toy":
        cap = rng.choice([4, 6, 16])
        tokens = _log_int(rng, 1, 64)
        c = _case("", "toy", "f32", tokens, cap, 8, "uniform", "f32")
    elif kind == "decode-paged":
        c = _case("", "qwen3", "bf16", 1, rng.randint(8, 32), rng.randint(12, 24), "trace", logits)
    elif kind == "fp8-decode-paged":
        c = _case("", "qwen3", "fp8", 1, rng.randint(8, 48), rng.randint(12, 24), "trace", logits)
    elif kind == "batch":
        c = _case("", "qwen3", "bf16", _log_int(rng, 1, 128), 128, 2, "uniform", logits)
    elif kind == "fp8-batch":
        c = _case("", "qwen3", "fp8", _log_int(rng, 1, 128), 128, 2, "uniform", logits)
    elif kind == "mixtral-batch":
        c = _case("", "mixtral", "bf16", _log_int(rng, 1, 64), 8, 1, "uniform", logits)
    elif kind == "prefill":
        c = _case("", "qwen3", "bf16", _log_int(rng, 129, 8192), 128, 1, "uniform", logits)
    elif kind == "fp8-prefill":
        c = _case("", "qwen3", "fp8", _log_int(rng, 129, 8192), 128, 1, "uniform", logits)
    elif kind == "mixtral-prefill":
        c = _case("", "mixtral", "bf16", _log_int(rng, 65, 1000), 8, 1, "uniform", logits)
    else:
        c = _case("", "qwen3", "bf16", rng.randint(8, 96), rng.randint(24, 64), 1, "uniform",
                  logits)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def _shape(case):
    s = SHAPES[case["layer"]]
    return s.hidden, s.inter, s.experts, s.top_k


def _inputs(case, seed):
    """Activations ``[steps, T, H]`` (as a normalisation leaves them: unit
    variance) and router logits ``[steps, T, E]``, on the GPU."""
    H, _, E, K = _shape(case)
    n, T = case["steps"], case["tokens"]
    g = torch.Generator(device="cuda").manual_seed(2 * seed + 1)
    x = torch.randn((n, T, H), generator=g, device="cuda")
    x = x if case["dtype"] == "f32" else x.to(torch.bfloat16)
    logits = torch.randn((n, T, E), generator=g, device="cuda")
    if case["routing"] == "trace":
        # experts of unequal popularity, and steps that mostly keep the
        # experts of the step before (60 % of them route to the same set)
        rank = torch.randperm(E, generator=g, device="cuda") + 1
        logits = 0.9 * logits - 1.1 * torch.log(rank.float())
        reuse = torch.rand((n,), generator=g, device="cuda").tolist()
        prev = None
        for t in range(n):
            if prev is not None and reuse[t] < 0.6:
                logits[t, 0, prev] += 20.0
            prev = torch.topk(logits[t, 0], K).indices
    return x, logits.to(torch.bfloat16) if case["logits"] == "bf16" else logits


def _expert_weights(case, seed):
    """Yields ``(expert, w13 [2I, H], w2 [H, I])`` float32 on the GPU."""
    H, I, E, _ = _shape(case)
    g = torch.Generator(device="cuda").manual_seed(2 * seed + 2)
    for e in range(E):
        yield (e, torch.randn((2 * I, H), generator=g, device="cuda") * WEIGHT_STD,
               torch.randn((H, I), generator=g, device="cuda") * WEIGHT_STD)


def prepare(case, seed):
    """The layer state a serving program keeps (masters in pinned host
    memory; a resident one primed) and the calls' device inputs."""
    H, I, E, K = _shape(case)
    dev = torch.device("cuda", torch.cuda.current_device())
    resident = case["cap"] == E
    if case["dtype"] == "fp8":
        lay = Fp8SlabLayout(H, I, FP8_BLOCK)
        buf = torch.empty((E, lay.slab), dtype=torch.uint8, pin_memory=True)
        views = lay.views(buf)
        for e, a, b in _expert_weights(case, seed):
            (q13, s13), (q2, s2) = block_quant_fp8(a), block_quant_fp8(b)
            for dst, src in zip(views, (q13, q2, s13, s2)):
                dst[e].copy_(src)
        st = WispMoEStateFP8(*views, case["cap"], dev, 0, block=FP8_BLOCK)
        if resident:
            st.ensure_resident(torch.arange(E, device=dev))
    else:
        dtype = torch.float32 if case["dtype"] == "f32" else torch.bfloat16
        slabs = torch.empty((E, 3 * I * H), dtype=dtype, pin_memory=True)
        w13, w2 = slab_views(slabs, SHAPES[case["layer"]])
        for e, a, b in _expert_weights(case, seed):
            w13[e].copy_(a.to(dtype))
            w2[e].copy_(b.to(dtype))
        st = WispMoEState(w13, w2, case["cap"], "resident" if resident else "paged", dev, 0)
        if resident:
            st.prime_identity()
    x, logits = _inputs(case, seed)
    torch.cuda.synchronize()
    return {"state": st, "x": list(x.unbind(0)), "logits": list(logits.unbind(0)), "k": K}


def run(state):
    st, k = state["state"], state["k"]
    return [st.forward(x, lg, k, True) for x, lg in zip(state["x"], state["logits"])]


# ---------------------------------------------------------------------------
# Cost and accuracy
# ---------------------------------------------------------------------------


def work(case):
    """Activations in and out, logits, and the weights of the experts each
    call routes to (their expected number), once each.  A paging case's
    copies from the host are not counted: how many there are depends on the
    trace."""
    H, I, E, K = _shape(case)
    n, T = case["steps"], case["tokens"]
    act = 4 if case["dtype"] == "f32" else 2
    per_expert = 3 * H * I * {"f32": 4, "bf16": 2, "fp8": 1}[case["dtype"]]
    if case["dtype"] == "fp8":
        per_expert += 4 * (3 * H * I) // (FP8_BLOCK[0] * FP8_BLOCK[1])
    experts = E * (1.0 - (1.0 - K / E) ** T)
    logits = T * E * (4 if case["logits"] == "f32" else 2)
    return {"bytes": int(n * (experts * per_expert + 2 * T * H * act + logits)),
            "flops": int(n * T * K * 6 * H * I)}


def tolerance(case):
    # f32: sums of 512 and 256 products in float32.  bf16: act and the output
    # are rounded to bf16 (2^-9 each).  fp8: bf16 roundings at h, silu, act,
    # y and the output, and groups of act whose largest value rounds to the
    # next bf16: a scale 2^-8 apart moves many of the group's e4m3 codes.
    # Seen against exact(): 1.7e-7, 2.5e-3 and 2.4e-2.
    return {"rel": {"f32": 1e-6, "bf16": 1e-2, "fp8": 6e-2}[case["dtype"]]}


def _quant_rows(v):
    """Per-row, per-128-group e4m3 quantisation and back (float64 values);
    the scale and the quotient are float32, as the operation defines them."""
    g = v.to(torch.float32).view(v.shape[0], -1, FP8_BLOCK[1])
    s = g.abs().amax(dim=2, keepdim=True).clamp_min(1e-10) / 448.0
    q = (g / s).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return (q.to(torch.float64) * s.to(torch.float64)).view(v.shape)


def _bf16(v):
    return v.to(torch.bfloat16).to(torch.float64)


def _expand(q, s):
    bn, bk = FP8_BLOCK
    w = q.to(torch.float64).view(s.shape[0], bn, s.shape[1], bk)
    return (w * s.to(torch.float64)[:, None, :, None]).view(q.shape)


def exact(case, seed):
    """The calls' outputs in float64: softmax, top-k (ties to the lower
    expert), renormalised weights, SwiGLU experts, weighted sum.  The
    block-FP8 layer's operation includes its quantisations and bf16
    intermediates; they are taken at float64 values."""
    H, I, E, K = _shape(case)
    x, logits = _inputs(case, seed)
    n, T = case["steps"], case["tokens"]
    xs = x.reshape(n * T, H).to(torch.float64)
    p = torch.softmax(logits.reshape(n * T, E).to(torch.float64), dim=1)
    order = torch.sort(logits.reshape(n * T, E).float(), dim=1, descending=True, stable=True)
    ids = order.indices[:, :K]
    w = p.gather(1, ids)
    w = w / w.sum(dim=1, keepdim=True)
    fp8 = case["dtype"] == "fp8"
    if fp8:
        xs = _quant_rows(xs)
    out = torch.zeros((n * T, H), dtype=torch.float64, device="cuda")
    for e, a, b in _expert_weights(case, seed):
        tok, kth = torch.nonzero(ids == e, as_tuple=True)
        if tok.numel() == 0:
            continue
        if fp8:
            a, b = _expand(*block_quant_fp8(a)), _expand(*block_quant_fp8(b))
        elif case["dtype"] == "bf16":
            a, b = _bf16(a), _bf16(b)
        else:
            a, b = a.to(torch.float64), b.to(torch.float64)
        h = xs[tok] @ a.t()
        if fp8:
            h = _bf16(h)
            act = _bf16(_bf16(torch.nn.functional.silu(h[:, :I])) * h[:, I:])
            y = _bf16((_quant_rows(act) @ b.t()) * w[tok, kth][:, None])
        else:
            y = ((torch.nn.functional.silu(h[:, :I]) * h[:, I:]) @ b.t()) * w[tok, kth][:, None]
        out.index_add_(0, tok, y)
    return list(out.view(n, T, H).unbind(0))
