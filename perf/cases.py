"""The work a user of this framework has it do, as timed cases.

Three kinds of case, each through the package's public entry points:

* "gemm": one grouped GEMM over the experts' rows (persistent_grouped_gemm),
  in bf16, fp16 or fp8 e4m3 with per-token and per-channel scales, weights
  stored [E, K, N] or as a linear layer's [E, N, K].  With routed counts the
  expert offsets are made from the received counts in the same pass, as a
  training or serving step does; with uniform counts they are in hand.
* "mlp": the routed expert MLP of a layer (expert_mlp_forward).
* "route": the row movement around the experts (dispatch_layout,
  permute_tokens, combine_tokens).

listed() names the cases; draw() gives others of the same ranges.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parent.parent / "moe-overlap_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import expert_mlp as mlp  # noqa: E402
import grouped_gemm as gg  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _gemm(name, experts, tokens, top_k, routing, k, n, dtype="bf16", weights="kn", atomic=True):
    case = dict(kind="gemm", experts=experts, tokens=tokens, top_k=top_k, routing=routing, k=k, n=n,
                dtype=dtype, weights=weights, atomic=atomic)
    return dict(case, name=name) if name else case


def _mlp(name, experts, tokens, top_k, hidden, ffn, activation, dtype="bf16", masked=0.0, atomic=True):
    case = dict(kind="mlp", experts=experts, tokens=tokens, top_k=top_k, routing="topk", hidden=hidden,
                ffn=ffn, activation=activation, dtype=dtype, masked=masked, atomic=atomic)
    return dict(case, name=name) if name else case


def _route(name, experts, tokens, top_k, hidden, dtype="bf16"):
    case = dict(kind="route", experts=experts, tokens=tokens, top_k=top_k, routing="topk", hidden=hidden,
                dtype=dtype)
    return dict(case, name=name) if name else case


def listed():
    return [
        # The smallest call: eight experts of a toy layer, where latency is all.
        _gemm("gemm_small", 8, 1024, 1, "uniform", 512, 1024),
        # The benchmark's main problem: a training micro-batch, balanced.
        _gemm("gemm_uniform", 16, 4096, 2, "uniform", 2048, 4096),
        # The same layer under heavily skewed routing.
        _gemm("gemm_skewed", 16, 8192, 2, "skewed", 2048, 4096),
        # The reference benchmark script's default problem, with its striped
        # schedule: 256 fine-grained experts of 128 rows.
        _gemm("gemm_reference_bench", 256, 4096, 8, "uniform", 7168, 2048, atomic=False),
        # A serving step on one rank's share of such a layer: 32 experts, a
        # few rows each.
        _gemm("gemm_decode", 32, 64, 8, "topk", 7168, 2048),
        # Weights as a linear layer keeps them, [out, in], with routed counts.
        _gemm("gemm_linear_weights", 16, 8192, 2, "topk", 2048, 4096, weights="nk"),
        # Sizes that fit no tile, in fp16.
        _gemm("gemm_odd_fp16", 12, 1111, 2, "topk", 1500, 2050, dtype="fp16"),
        # Fine-grained experts in fp8: prefill and decode of one layer.
        _gemm("fp8_prefill", 64, 4096, 6, "topk", 2048, 1408, dtype="fp8", weights="nk"),
        _gemm("fp8_decode", 64, 128, 6, "topk", 2048, 1408, dtype="fp8", weights="nk"),
        # A whole expert MLP: a training or prefill batch (SwiGLU), and a
        # decode step with the reference's GELU experts.
        _mlp("mlp_prefill", 16, 8192, 2, 2048, 4096, "swiglu"),
        _mlp("mlp_decode", 16, 32, 2, 2048, 4096, "gelu"),
        # Routing and row movement alone, at a large model's width.
        _route("route_rows", 256, 4096, 8, 7168),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _size(rng, lo, hi):
    """A matrix extent: mostly a multiple of 64, else of 8, else any number."""
    v = _log(rng, lo, hi)
    step = rng.choice((64, 64, 64, 64, 8, 1))
    return max(lo, v // step * step)


def draw(rng):
    """One more case of the ranges the listed ones stand for."""
    kind = rng.choice(("gemm", "gemm", "gemm", "fp8", "mlp", "mlp", "route"))
    while True:
        experts = _log(rng, 4, 256)
        top_k = rng.choice((1, 2, 4, 6, 8))
        top_k = min(top_k, experts)
        # 1 to 1024 rows an expert on average.
        tokens = max(1, int(experts * _log(rng, 1, 1024) / top_k))
        if tokens > 32768:
            continue
        rows = tokens * top_k
        atomic = rng.random() < 0.75
        if kind == "gemm":
            k, n = _size(rng, 256, 7168), _size(rng, 256, 7168)
            if experts * k * n > 256 * 7168 * 2048 or rows * k * n > 32768 * 7168 * 2048:
                continue
            routing = rng.choice(("uniform", "topk", "topk", "skewed"))
            if routing == "uniform":
                tokens = max(1, rows // experts) * experts
                top_k = 1
            return _gemm(None, experts, tokens, top_k, routing, k, n, dtype=rng.choice(("bf16", "bf16", "fp16")),
                         weights=rng.choice(("kn", "kn", "nk")), atomic=atomic)
        if kind == "fp8":
            k, n = _size(rng, 256, 7168), _size(rng, 256, 7168)
            if experts * k * n > 256 * 7168 * 2048 or rows * k * n > 32768 * 7168 * 2048:
                continue
            return _gemm(None, experts, tokens, top_k, rng.choice(("topk", "topk", "skewed")), k, n, dtype="fp8",
                         weights="nk", atomic=atomic)
        hidden = _log(rng, 512, 7168) // 64 * 64
        if kind == "mlp":
            ffn = _log(rng, 256, 4096) // 32 * 32
            activation = rng.choice(("gelu", "swiglu"))
            cols = 3 * ffn if activation == "swiglu" else 2 * ffn
            if experts * hidden * cols > 256 * 7168 * 2048 or rows * hidden * cols > 32768 * 7168 * 2048:
                continue
            return _mlp(None, experts, tokens, top_k, hidden, ffn, activation, dtype=rng.choice(("bf16", "bf16", "fp16")),
                        masked=rng.choice((0.0, 0.0, 0.25)), atomic=atomic)
        return _route(None, experts, tokens, top_k, hidden, dtype=rng.choice(("bf16", "fp16")))


# ---- inputs ------------------------------------------------------------------


def _routing(case, seed):
    """(topk_idx int64 [T, k], topk_weight fp32 [T, k]) on the CPU: top-k of
    N(0,1) router logits; "skewed" adds the log of a Zipf(1.2) draw per expert,
    the same for every seed."""
    gen = torch.Generator().manual_seed(seed)
    logits = torch.randn(case["tokens"], case["experts"], generator=gen)
    if case["routing"] == "skewed":
        zipf = np.random.default_rng(0).zipf(1.2, case["experts"])
        logits += torch.from_numpy(np.log(np.minimum(zipf, 10 ** 9).astype(np.float64))).float()
    weight, idx = torch.topk(torch.softmax(logits, dim=-1), case["top_k"], dim=1)
    if case.get("masked", 0.0) > 0:
        idx[torch.rand(idx.shape, generator=gen) < case["masked"]] = -1
    return idx, weight.float()


def _counts(case, seed):
    """Rows per expert, int32 [E] on the CPU."""
    experts, rows = case["experts"], case["tokens"] * case["top_k"]
    if case["routing"] == "uniform":
        return torch.full((experts,), rows // experts, dtype=torch.int32)
    idx, _ = _routing(case, seed)
    return torch.bincount(idx[idx >= 0].flatten(), minlength=experts).to(torch.int32)


def _weights(gen, experts, rows, cols, fan_in, dtype):
    """[experts, rows, cols] of N(0, 1/fan_in), made an expert at a time."""
    w = torch.empty(experts, rows, cols, device="cuda", dtype=dtype)
    for e in range(experts):
        w[e] = torch.randn(rows, cols, generator=gen, device="cuda").mul_(1.0 / math.sqrt(fan_in))
    return w


def _quantise(t):
    """(e4m3 values, fp32 scales) with one scale per row, amax / 448."""
    scale = t.abs().amax(dim=-1, keepdim=True).clamp_min(1e-12) / 448.0
    return (t / scale).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn), scale.squeeze(-1)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    experts = case["experts"]
    if case["kind"] == "gemm":
        counts = _counts(case, seed)
        m, k, n = int(counts.sum()), case["k"], case["n"]
        state = dict(kind="gemm", atomic=case["atomic"], scales={})
        if case["routing"] == "uniform":
            state["offsets"] = gg.expert_offsets_from_recv_counts(counts, device=torch.device("cuda"))
        else:
            state["counts"] = counts.cuda()
        a = torch.randn(m, k, generator=gen, device="cuda")
        if case["dtype"] == "fp8":
            state["a"], a_scale = _quantise(a)
            b = torch.empty(experts, n, k, device="cuda", dtype=torch.float8_e4m3fn)
            b_scale = torch.empty(experts, n, device="cuda")
            for e in range(experts):
                b[e], b_scale[e] = _quantise(torch.randn(n, k, generator=gen, device="cuda") / math.sqrt(k))
            state["scales"] = dict(a_scale=a_scale, b_scale=b_scale)
            state["b"] = b.transpose(1, 2)
            return state
        dtype = _DTYPES[case["dtype"]]
        state["a"] = a.to(dtype)
        if case["weights"] == "nk":
            state["b"] = _weights(gen, experts, n, k, k, dtype).transpose(1, 2)
        else:
            state["b"] = _weights(gen, experts, k, n, k, dtype)
        return state

    dtype, hidden = _DTYPES[case["dtype"]], case["hidden"]
    idx, weight = _routing(case, seed)
    state = dict(kind=case["kind"], idx=idx.cuda(), weight=weight.cuda(), experts=experts)
    state["x"] = torch.randn(case["tokens"], hidden, generator=gen, device="cuda").to(dtype)
    if case["kind"] == "route":
        state["y"] = torch.randn(case["tokens"] * case["top_k"], hidden, generator=gen, device="cuda").to(dtype)
        return state
    ffn = case["ffn"]
    state.update(activation=case["activation"], atomic=case["atomic"])
    w1 = _weights(gen, experts, hidden, ffn, hidden, dtype)
    if case["activation"] == "swiglu":
        w1 = mlp.interleave_gate_up(w1, _weights(gen, experts, hidden, ffn, hidden, dtype))
    state["w1"] = w1
    state["w2"] = _weights(gen, experts, ffn, hidden, ffn, dtype)
    return state


# ---- one pass ----------------------------------------------------------------


def run(state):
    if state["kind"] == "gemm":
        offsets = state.get("offsets")
        if offsets is None:
            offsets = gg.expert_offsets_from_recv_counts(state["counts"])
        return gg.persistent_grouped_gemm(state["a"], state["b"], offsets, use_atomic_queue=state["atomic"],
                                          **state["scales"])
    if state["kind"] == "mlp":
        return mlp.expert_mlp_forward(state["x"], state["idx"], state["weight"], state["w1"], state["w2"],
                                      state["activation"], use_atomic_queue=state["atomic"])
    layout = mlp.dispatch_layout(state["idx"], state["experts"])
    rows = mlp.permute_tokens(state["x"], layout)
    out = mlp.combine_tokens(state["y"], layout, state["weight"])
    return dict(counts=layout.counts, offsets=layout.offsets, slot_position=layout.slot_position,
                token_index=layout.token_index, row_assignment=layout.row_assignment, rows=rows, out=out)


# ---- what a pass cannot do without -------------------------------------------


def work(case):
    tokens, top_k = case["tokens"], case["top_k"]
    if case["kind"] == "route":
        row = 2 * case["hidden"]
        slots = tokens * top_k
        # Ids read, the layout written, rows gathered, rows and gates combined.
        return dict(bytes=slots * (8 + 12) + 8 * case["experts"] + (tokens + slots) * row
                    + slots * (row + 4) + tokens * row, flops=2 * slots * case["hidden"])
    counts = _counts(case, 0)
    m, busy = int(counts.sum()), int((counts > 0).sum())
    if case["kind"] == "gemm":
        k, n = case["k"], case["n"]
        elem = 1 if case["dtype"] == "fp8" else 2
        scales = 4 * (m + busy * n) if case["dtype"] == "fp8" else 0
        return dict(bytes=elem * (m * k + busy * k * n) + 2 * m * n + scales, flops=2 * m * k * n)
    hidden, ffn = case["hidden"], case["ffn"]
    cols = 2 * ffn if case["activation"] == "swiglu" else ffn
    return dict(bytes=2 * (2 * tokens * hidden + busy * hidden * (cols + ffn)) + 12 * tokens * top_k,
                flops=2 * m * hidden * (cols + ffn))


def tolerance(case):
    """Relative 2-norm error and largest error of another correct
    implementation: outputs are fp32 sums rounded once to 16 bits, so two sum
    orders differ by single roundings (2^-9 relative in bf16, 2^-12 in fp16)
    in a share of the values; the MLP's hidden layer is rounded to 16 bits as
    well."""
    unit = 4.0 if case["dtype"] == "fp16" else 1.0
    if case["kind"] == "mlp":
        return dict(rel=4e-3 / unit, max=4e-2 / unit)
    return dict(rel=2e-3 / unit, max=2e-2 / unit)


# ---- the same in 64 bits -----------------------------------------------------


def _mm(rows, w):
    return rows.double() @ w.double()


def exact(case, seed):
    state = prepare(case, seed)
    if case["kind"] == "gemm":
        counts = _counts(case, seed).tolist()
        a, b = state["a"], state["b"]
        out = torch.empty(a.shape[0], b.shape[2], dtype=torch.float64, device="cuda")
        at = 0
        for e, c in enumerate(counts):
            if c:
                if case["dtype"] == "fp8":
                    w = b[e].transpose(0, 1).float().double().transpose(0, 1).contiguous()
                    y = a[at:at + c].float().double() @ w
                    y *= state["scales"]["a_scale"][at:at + c, None].double()
                    y *= state["scales"]["b_scale"][e][None].double()
                    out[at:at + c] = y
                else:
                    out[at:at + c] = _mm(a[at:at + c], b[e].contiguous())
            at += c
        return out
    idx, weight = state["idx"].cpu(), state["weight"].double()
    flat = idx.flatten()
    order = torch.argsort(torch.where(flat >= 0, flat, case["experts"]), stable=True)[: int((flat >= 0).sum())]
    position = torch.full_like(flat, -1)
    position[order] = torch.arange(order.numel())
    if case["kind"] == "route":
        counts = torch.bincount(flat[flat >= 0], minlength=case["experts"])
        offsets = torch.cat([torch.zeros(1, dtype=torch.int64), counts.cumsum(0)])
        tokens = order // case["top_k"]
        gathered = state["y"].double()[position.cuda()].view(case["tokens"], case["top_k"], -1)
        i32 = torch.int32
        return dict(counts=counts.to(i32), offsets=offsets.to(i32), slot_position=position.to(i32),
                    token_index=tokens.to(i32), row_assignment=order.to(i32),
                    rows=state["x"].double()[tokens.cuda()], out=(gathered * weight[:, :, None]).sum(1))
    x = state["x"]
    out = torch.zeros(x.shape, dtype=torch.float64, device="cuda")
    for e in range(case["experts"]):
        slots = (flat == e).nonzero().flatten().cuda()
        if slots.numel() == 0:
            continue
        tokens = slots // case["top_k"]
        h = _mm(x[tokens], state["w1"][e])
        if case["activation"] == "swiglu":
            h = h.view(h.shape[0], -1, 2, 32)
            h = (torch.nn.functional.silu(h[:, :, 0]) * h[:, :, 1]).reshape(h.shape[0], -1)
        else:
            h = torch.nn.functional.gelu(h)
        y = h @ state["w2"][e].double()
        out.index_add_(0, tokens, y * weight.flatten()[slots, None])
    return out
