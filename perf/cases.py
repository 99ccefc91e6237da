"""The workloads that this repository's performance is measured on.

Each case is one call (or the short sequence of calls) that a serving program
makes through the public operators of ``q6moe``, on inputs drawn from a seed:

* ``proj``   one packed-Q6 projection (``q6_matmul``);
* ``moe``    the MoE half of a decoder layer: device router (``routes``) and
             routed SwiGLU experts (``expert_parallel``), with the always-on
             shared expert where the layer has one;
* ``attn``   the attention half of a decode step: the new token's key and value
             go into the paged INT8 cache (``write_paged``), then every
             sequence attends to its cached tokens (``paged_decode_attention``);
* ``kv``     a gather + dequant of cached tokens (``read_paged`` of a whole
             pool, ``read_quantized`` of selected tokens of the dense cache).

Expert tables are drawn as GGUF blocks with the code and scale distributions
that quantized N(0, 0.02) weights have, and packed once, as at load time.
"""

import math
import sys
from pathlib import Path

import torch

PACKAGE = str(Path(__file__).resolve().parents[1] / "data-synth-tpu_amd")
if PACKAGE not in sys.path:
    sys.path.insert(0, PACKAGE)

import q6moe  # noqa: E402

# The layers that configurations, tests and bench.py of this repository run
# (gate/up format, down format, experts, top-k, hidden, intermediate, shared
# intermediate, compute policy), and the most tokens that a drawn case gives it.
LAYERS = {
    "q6": ("Q6_K", "Q6_K", 128, 8, 2048, 768, 0, "bf16", 4096),
    "q4_shared": ("Q4_K", "Q4_K", 64, 6, 4096, 1024, 4096, "bf16", 1024),
    "wide": ("Q6_K", "Q8_0", 512, 10, 2560, 640, 0, "bf16", 2048),
    "q5": ("Q5_K", "Q8_0", 128, 8, 2048, 768, 0, "bf16", 1024),
    "w8a8": ("Q8_0", "Q8_0", 128, 8, 2048, 768, 0, "int8_q8", 1024),
}
BLOCK = {"Q6_K": (256, 210), "Q5_K": (256, 176), "Q4_K": (256, 144), "Q8_0": (32, 34)}
SIGMA = 0.02  # standard deviation of the weights


def listed():
    return [
        # the smallest call: one projection of a few tokens of a decode step
        dict(name="proj_step", kind="proj", tokens=4, inputs=2560, outputs=640),
        # the same operator over a prompt of odd length
        dict(name="proj_prompt", kind="proj", tokens=777, inputs=2560, outputs=1280),
        # the headline decode step: 8 sequences, 128 experts, top-8, Q6_K
        dict(name="q6_step", kind="moe", layer="q6", tokens=8, skew=0.0),
        # a long prompt (or many) through the same layer, experts unevenly loaded
        dict(name="q6_prompt", kind="moe", layer="q6", tokens=4096, skew=0.5),
        # Q4_K layer with a gated shared expert, decode step of 8 sequences
        dict(name="q4_shared_step", kind="moe", layer="q4_shared", tokens=8, skew=0.0),
        # and one prompt through it
        dict(name="q4_shared_prompt", kind="moe", layer="q4_shared", tokens=1024, skew=0.5),
        # the reference model's own layer (512 experts, top-10): one sequence decoding
        dict(name="wide_step", kind="moe", layer="wide", tokens=1, skew=0.0),
        # and a prompt of odd length through it
        dict(name="wide_prompt", kind="moe", layer="wide", tokens=2001, skew=0.5),
        # a Q5_K / Q8_0 checkpoint layer, a short prompt of odd length
        dict(name="q5_prompt", kind="moe", layer="q5", tokens=333, skew=0.5),
        # an all-Q8_0 layer under the W8A8 policy, a prompt
        dict(name="w8a8_prompt", kind="moe", layer="w8a8", tokens=1024, skew=0.5),
        # decode step of 8 sequences with ragged contexts of up to 32 K tokens
        dict(name="attn_step", kind="attn", batch=8, context=32768, page=256, kv_heads=4, heads_per_kv=8),
        # the whole paged cache of 8 such sequences, dequantized
        dict(name="kv_read", kind="kv", layout="paged", batch=8, context=32768, selected=32768, page=256,
             kv_heads=4, group=128),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choices(("proj", "moe", "attn", "kv"), (3, 10, 4, 2))[0]
    if kind == "proj":
        return dict(kind=kind, tokens=_log(rng, 1, 1024), inputs=32 * _log(rng, 16, 128),
                    outputs=8 * _log(rng, 40, 512))
    if kind == "moe":
        layer = rng.choice(sorted(LAYERS))
        return dict(kind=kind, layer=layer, tokens=_log(rng, 1, LAYERS[layer][8]), skew=rng.choice((0.0, 0.5)))
    if kind == "attn":
        page = rng.choice((64, 128, 256))
        kv_heads = rng.choice((2, 4, 8))
        return dict(kind=kind, batch=_log(rng, 1, 32 // kv_heads), context=page * _log(rng, 2, 32768 // page),
                    page=page, kv_heads=kv_heads, heads_per_kv=rng.choice((1, 4, 6, 8)))
    context = 256 * _log(rng, 2, 64)
    if rng.random() < 0.5:
        return dict(kind=kind, layout="paged", batch=_log(rng, 1, 8), context=context, selected=context, page=256,
                    kv_heads=4, group=128)
    return dict(kind=kind, layout="dense", batch=_log(rng, 1, 8), context=context,
                selected=_log(rng, 64, min(context, 4096)), page=0, kv_heads=4, group=rng.choice((32, 128)))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device="cuda")


def _codes(gen, shape, mean, sd, lo, hi):
    return (_randn(gen, *shape) * sd + mean).round_().clamp_(lo, hi).to(torch.int16)


def _small(gen, shape, lo, hi):
    return torch.randint(lo, hi + 1, shape, generator=gen, device="cuda", dtype=torch.int16)


def _fp16(gen, shape, center):
    """Block scales around ``center`` (+- 20 %), FP16."""
    return ((torch.rand(shape, generator=gen, device="cuda") * 0.4 + 0.8) * center).to(torch.float16)


def _as_bytes(t):
    return t.contiguous().view(torch.uint8)


def _k_scales(sc, mn):
    """The 12 bytes that hold 8 six-bit scales and 8 six-bit minima."""
    head = (sc[..., :4] & 63) | ((sc[..., 4:] >> 4) << 6)
    middle = (mn[..., :4] & 63) | ((mn[..., 4:] >> 4) << 6)
    tail = (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)
    return torch.cat((head, middle, tail), -1).to(torch.uint8)


def _quantized(gen, qtype, rows, width, raw=True, values=False):
    """One matrix (or a stack: ``rows`` a tuple) of GGUF blocks: its bytes
    [..., blocks, size], its values as FP64, or both. The weights are what the
    format's decoder gives in FP32."""
    rows = rows if isinstance(rows, tuple) else (rows,)
    per, _ = BLOCK[qtype]
    lead = (*rows, -(-width // per))
    got = []
    if qtype == "Q6_K":
        c = _codes(gen, (*lead, 2, 4, 32), 32, 10, 0, 63)
        sc = _small(gen, (*lead, 16), 60, 127) * (_small(gen, (*lead, 16), 0, 1) * 2 - 1)
        d = _fp16(gen, (*lead, 1), SIGMA / (10 * 94))
        if raw:
            low = c & 15
            ql = (low[..., :2, :] | (low[..., 2:, :] << 4)).to(torch.uint8).flatten(-3)
            high = c >> 4
            qh = (high[..., 0, :] | (high[..., 1, :] << 2) | (high[..., 2, :] << 4) | (high[..., 3, :] << 6))
            got.append(torch.cat((ql, qh.to(torch.uint8).flatten(-2), sc.to(torch.int8).view(torch.uint8),
                                  _as_bytes(d)), -1))
        if values:
            q = (c.double() - 32).flatten(-3).unflatten(-1, (16, 16))
            got.append((q * (sc.double() * d.double())[..., None]).flatten(-3))
    elif qtype in ("Q4_K", "Q5_K"):
        top = 15 if qtype == "Q4_K" else 31
        mid, sd = (top + 1) / 2, (top + 1) / 6
        c = _codes(gen, (*lead, 8, 32), mid, sd, 0, top)
        sc, mn = _small(gen, (*lead, 8), 32, 63), _small(gen, (*lead, 8), 32, 63)
        d = _fp16(gen, (*lead, 1), SIGMA / (sd * 47))
        dmin = (d.float() * mid).to(torch.float16)
        if raw:
            low = c & 15
            qs = (low[..., 0::2, :] | (low[..., 1::2, :] << 4)).to(torch.uint8).flatten(-2)
            parts = [_as_bytes(d), _as_bytes(dmin), _k_scales(sc, mn)]
            if qtype == "Q5_K":
                bit = torch.arange(8, device="cuda", dtype=torch.int16)[:, None]
                parts.append(((c >> 4) << bit).sum(-2).to(torch.uint8))
            got.append(torch.cat((*parts, qs), -1))
        if values:
            scale, low = sc.double() * d.double(), mn.double() * dmin.double()
            got.append((c.double() * scale[..., None] - low[..., None]).float().double().flatten(-3))
    else:  # Q8_0
        c = _codes(gen, (*lead, 32), 0, 45, -127, 127)
        d = _fp16(gen, (*lead, 1), SIGMA / 45)
        if raw:
            got.append(torch.cat((_as_bytes(d), c.to(torch.int8).view(torch.uint8)), -1))
        if values:
            got.append((c.double() * d.double()).flatten(-2))
    return got[0] if len(got) == 1 else got


def _experts(gen, experts, qtype, rows, width, **what):
    """The experts of one projection, a few at a time (bounded memory)."""
    step = max(1, (1 << 27) // (rows * width))
    for e in range(0, experts, step):
        yield _quantized(gen, qtype, (min(step, experts - e), rows), width, **what)


def _layer_inputs(case, seed):
    """The tokens, router logits, shared-expert gate and the generator that
    draws the weights next."""
    gate_up, down, experts, top_k, hidden, inter, shared, compute, _ = LAYERS[case["layer"]]
    gen = _generator(seed)
    x = _randn(gen, case["tokens"], hidden).to(torch.bfloat16)
    logits = _randn(gen, case["tokens"], experts) + _randn(gen, experts) * case["skew"]
    router = (_randn(gen, hidden) * SIGMA).to(torch.bfloat16) if shared else None
    return gen, x, logits, router


def _prepare_moe(case, seed):
    gate_up, down, experts, top_k, hidden, inter, shared, compute, _ = LAYERS[case["layer"]]
    gen, x, logits, router = _layer_inputs(case, seed)
    ffn = q6moe.expert_parallel(None, gate_type=gate_up, up_type=gate_up, down_type=down, hidden=hidden,
                                intermediate=inter, compute=compute)
    tables = []
    for qtype, rows, width in ((gate_up, inter, hidden), (gate_up, inter, hidden), (down, hidden, inter)):
        raw = torch.cat(list(_experts(gen, experts, qtype, rows, width)))
        tables.append(q6moe.pack_experts(raw.reshape(experts, -1), qtype, rows, width))
        del raw
    extra = None
    if shared:
        extra = dict(router=router, intermediate=shared)
        for name, qtype, rows, width in (("gate", gate_up, shared, hidden), ("up", gate_up, shared, hidden),
                                         ("down", down, hidden, shared)):
            extra[name] = q6moe.pack_experts(_quantized(gen, qtype, rows, width).reshape(1, -1), qtype, rows, width)
    return dict(kind="moe", ffn=ffn, tables=tables, x=x, logits=logits, top_k=top_k, shared=extra)


def _prepare_proj(case, seed):
    gen = _generator(seed)
    x = _randn(gen, case["tokens"], case["inputs"]).to(torch.bfloat16)
    raw = _quantized(gen, "Q6_K", case["outputs"], case["inputs"])
    packed, scales = q6moe.q6_pack(raw, case["inputs"])
    return dict(kind="proj", x=x, packed=packed, scales=scales, outputs=case["outputs"])


def _cache(gen, rows, groups, group):
    """INT8 codes [rows, groups * group] and scales [rows, groups] of N(0, 1) keys or values."""
    codes = (_randn(gen, rows, groups * group) * 45).round_().clamp_(-127, 127).to(torch.int8)
    return codes, torch.rand(rows, groups, generator=gen, device="cuda") * 0.008 + 0.018


def _attn_inputs(case, seed):
    gen = _generator(seed)
    batch, context, page, kvh = case["batch"], case["context"], case["page"], case["kv_heads"]
    per_seq = context // page
    pages = batch * per_seq
    state = dict(kind="attn", page=page, kv_heads=kvh)
    for name in ("k", "v"):
        codes, scales = _cache(gen, pages * page, kvh, 128)
        state[name] = codes.view(pages, page, kvh * 128)
        state[name + "_scales"] = scales.view(pages, page, kvh)
        state["new_" + name] = _randn(gen, batch, kvh * 128).to(torch.bfloat16)
    state["table"] = torch.randperm(pages, generator=gen, device="cuda").to(torch.int32).view(batch, per_seq)
    state["q"] = _randn(gen, batch, kvh * case["heads_per_kv"], 128).to(torch.bfloat16)
    # ragged contexts: a quarter to all of the capacity
    lengths = torch.rand(batch, generator=gen, device="cuda") * 0.75 + 0.25
    state["lengths"] = (lengths * context).ceil().to(torch.int32).clamp_(1, context)
    state["slots"] = state["lengths"] - 1  # the new token's place
    return state


def _kv_inputs(case, seed):
    gen = _generator(seed)
    batch, context, kvh, group = case["batch"], case["context"], case["kv_heads"], case["group"]
    groups = kvh * 128 // group
    state = dict(kind="kv", layout=case["layout"], kv_heads=kvh, group=group, page=case["page"])
    for name in ("k", "v"):
        codes, scales = _cache(gen, batch * context, groups, group)
        if case["layout"] == "paged":
            state[name] = codes.view(-1, case["page"], kvh * 128)
            state[name + "_scale"] = scales.view(-1, case["page"], groups)
        else:  # the dense cache keeps a BF16 scale plane [batch * groups, time]
            state[name] = codes.view(batch, context, kvh * 128)
            plane = scales.view(batch, context, groups).transpose(1, 2).reshape(batch * groups, context)
            state[name + "_scale"] = plane.to(torch.bfloat16)
    if case["layout"] == "paged":
        pages = batch * context // case["page"]
        table = torch.randperm(pages, generator=gen, device="cuda").to(torch.int32)
        state["table"] = table.view(batch, context // case["page"])
    else:
        state["indices"] = torch.randint(0, context, (batch, case["selected"]), generator=gen, device="cuda",
                                         dtype=torch.int32)
    return state


class _CacheShape:
    def __init__(self, kv_heads, group):
        self.kv_heads, self.head_dim, self.cache_group = kv_heads, 128, group


def prepare(case, seed):
    if case["kind"] == "proj":
        return _prepare_proj(case, seed)
    if case["kind"] == "moe":
        return _prepare_moe(case, seed)
    if case["kind"] == "attn":
        return _attn_inputs(case, seed)
    state = _kv_inputs(case, seed)
    state["shape"] = _CacheShape(case["kv_heads"], case["group"])
    return state


def run(s):
    if s["kind"] == "proj":
        return q6moe.q6_matmul(s["x"], s["packed"], s["scales"], output_features=s["outputs"])
    if s["kind"] == "moe":
        ids, weights = q6moe.routes(s["logits"], s["top_k"])
        return s["ffn"](*s["tables"], s["x"], ids, weights, shared=s["shared"])
    if s["kind"] == "attn":
        for name in ("k", "v"):
            q6moe.write_paged(s[name], s[name + "_scales"], s["table"], s["new_" + name], s["slots"],
                              page_size=s["page"], kv_heads=s["kv_heads"], head_dim=128)
        out = q6moe.paged_decode_attention(s["q"], s["k"], s["k_scales"], s["v"], s["v_scales"], s["table"],
                                           s["lengths"], page_size=s["page"], kv_heads=s["kv_heads"])
        return dict(out=out, k=s["k"], v=s["v"], k_scales=s["k_scales"], v_scales=s["v_scales"])
    if s["layout"] == "paged":
        return [q6moe.read_paged(s[n], s[n + "_scale"], s["table"], page_size=s["page"], kv_heads=s["kv_heads"],
                                 head_dim=128, group=s["group"]) for n in ("k", "v")]
    return [q6moe.read_quantized(s, n, s["indices"], s["shape"]) for n in ("k", "v")]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _bytes(qtype, rows, width):
    per, size = BLOCK[qtype]
    return rows * -(-width // per) * size


def work(case):
    if case["kind"] == "proj":
        m, k, n = case["tokens"], case["inputs"], case["outputs"]
        return dict(bytes=2 * m * k + _bytes("Q6_K", n, k) + 4 * m * n, flops=2 * m * n * k)
    if case["kind"] == "moe":
        gate_up, down, experts, top_k, hidden, inter, shared, _, _ = LAYERS[case["layer"]]
        m = case["tokens"]
        active = experts * (1 - (1 - top_k / experts) ** m)  # expected number of experts with a token
        expert = 2 * _bytes(gate_up, inter, hidden) + _bytes(down, hidden, inter)
        total = active * expert + m * (4 * experts + 2 * hidden + 2 * hidden)
        if shared:
            total += 2 * _bytes(gate_up, shared, hidden) + _bytes(down, hidden, shared) + 2 * hidden
        return dict(bytes=total, flops=6 * m * hidden * (top_k * inter + shared))
    kvh = case["kv_heads"]
    if case["kind"] == "attn":
        tokens = case["batch"] * case["context"] * 0.625  # mean of the ragged lengths
        heads = kvh * case["heads_per_kv"]
        return dict(bytes=tokens * kvh * 2 * (128 + 4) + case["batch"] * (4 * heads + 4 * kvh) * 128,
                    flops=4 * tokens * heads * 128)
    rows = case["batch"] * case["selected"]
    scale = 4 if case["layout"] == "paged" else 2
    return dict(bytes=2 * rows * (kvh * 128 * 3 + scale * kvh * 128 // case["group"]), flops=2 * rows * kvh * 128)


def tolerance(case):
    """About four times what the operators differ by from the same computation
    with the same rounding points and 64-bit sums, over sizes of the ranges."""
    if case["kind"] == "kv":
        return "exact"  # one product, rounded once
    if case["kind"] == "proj":
        return {"rel": 1e-5}  # FP32 sums of exact products
    if case["kind"] == "attn":
        return {"rel": 4e-4, "max": 0.03}
    if LAYERS[case["layer"]][7] == "int8_q8":
        return {"rel": 1.2e-2, "max": 0.12}  # another sum can move an activation's INT8 code
    return {"rel": 1.7e-3, "max": 0.07}


# ---------------------------------------------------------------------------
# The same results in 64 bits, from the BF16 (or INT8) operands on
# ---------------------------------------------------------------------------
def _bf16(v):
    return v.float().to(torch.bfloat16).double()


def _w8a8_operand(v):
    """Activations as the W8A8 policy defines them: per 32 values an INT8 code and an FP32 scale."""
    g = v.float().unflatten(-1, (-1, 32))
    scale = g.abs().amax(-1, keepdim=True) / 127
    codes = (g / torch.where(scale == 0, torch.ones_like(scale), scale)).round().clamp(-127, 127)
    return (codes.double() * scale.double()).flatten(-2)


def _ffn64(x, gate, up, down, w8):
    if not w8:
        g, u = x @ gate.T, x @ up.T
        return (g * torch.sigmoid(g) * u) @ down.T
    x = _w8a8_operand(x)
    g, u = _bf16(x @ gate.T), _bf16(x @ up.T)
    return _w8a8_operand(_bf16(_bf16(g * torch.sigmoid(g)) * u)) @ down.T


def _exact_moe(case, seed):
    gate_up, down, experts, top_k, hidden, inter, shared, compute, _ = LAYERS[case["layer"]]
    gen, x, logits, router = _layer_inputs(case, seed)
    w8 = compute == "int8_q8"
    operand = (lambda v: v) if w8 else _bf16
    x = x.double()
    order = torch.sort(logits, dim=-1, descending=True, stable=True).indices[:, :top_k]
    p = torch.softmax(logits.double(), -1).gather(-1, order)
    weights = _bf16(p / p.sum(-1, keepdim=True))
    mats = []  # gate, up and down of each expert as (chunks of) FP64; FP32 holds a BF16 weight exactly
    for qtype, rows, width in ((gate_up, inter, hidden), (gate_up, inter, hidden), (down, hidden, inter)):
        chunks = _experts(gen, experts, qtype, rows, width, raw=False, values=True)
        mats.append([operand(c[..., :width]).to(torch.float64 if w8 else torch.bfloat16) for c in chunks])
    out = torch.zeros(x.shape, dtype=torch.float64, device="cuda")

    def expert(i, e):
        for chunk in mats[i]:
            if e < chunk.shape[0]:
                return chunk[e].double()
            e -= chunk.shape[0]

    for e in range(experts):
        token, slot = torch.nonzero(order == e, as_tuple=True)
        if token.numel():
            y = _ffn64(x[token], expert(0, e), expert(1, e), expert(2, e), w8)
            out.index_add_(0, token, y * weights[token, slot][:, None])
    if shared:
        parts = [operand(_quantized(gen, q, rows, width, raw=False, values=True)[..., :width]) for q, rows, width in
                 ((gate_up, shared, hidden), (gate_up, shared, hidden), (down, hidden, shared))]
        out += _ffn64(x, *parts, w8) * torch.sigmoid(x @ router.double())[:, None]
    return out


def _exact_attn(case, seed):
    s = _attn_inputs(case, seed)
    page, kvh, r = case["page"], case["kv_heads"], case["heads_per_kv"]
    rows = []
    for b in range(case["batch"]):
        n = int(s["lengths"][b])
        at = torch.arange(n, device="cuda")
        at = s["table"][b].long()[at // page] * page + at % page
        kv = []
        for name in ("k", "v"):
            codes = s[name].view(-1, kvh, 128)[at].float()
            scales = s[name + "_scales"].view(-1, kvh)[at]
            new = s["new_" + name][b].float().view(kvh, 128)
            scales[-1] = new.abs().amax(-1) / 127
            codes[-1] = (new / scales[-1][:, None]).round().clamp(-127, 127)
            kv.append(_bf16(codes * scales[..., None]))
        q = s["q"][b].double().view(kvh, r, 128)
        scores = q @ kv[0].permute(1, 2, 0).contiguous() / math.sqrt(128)
        rows.append((torch.softmax(scores, -1) @ kv[1].transpose(0, 1).contiguous()).reshape(kvh * r, 128))
    return dict(out=torch.stack(rows), k=None, v=None, k_scales=None, v_scales=None)


def exact(case, seed):
    if case["kind"] == "proj":
        gen = _generator(seed)
        x = _randn(gen, case["tokens"], case["inputs"]).to(torch.bfloat16).double()
        w = _quantized(gen, "Q6_K", case["outputs"], case["inputs"], raw=False, values=True)
        return x @ _bf16(w[:, : case["inputs"]]).T
    if case["kind"] == "moe":
        return _exact_moe(case, seed)
    if case["kind"] == "attn":
        return _exact_attn(case, seed)
    s = _kv_inputs(case, seed)
    kvh, group = case["kv_heads"], case["group"]
    outs = []
    for name in ("k", "v"):
        if case["layout"] == "paged":
            codes, scales = s[name][s["table"].long()], s[name + "_scale"][s["table"].long()]
        else:
            at = s["indices"].long()
            codes = torch.stack([c[i] for c, i in zip(s[name], at)])
            plane = s[name + "_scale"].view(case["batch"], -1, case["context"])
            scales = torch.stack([p[:, i].T for p, i in zip(plane, at)])
        v = codes.reshape(-1, group).double() * scales.reshape(-1, 1).double()
        outs.append(_bf16(v).view(case["batch"], case["selected"], kvh, 128))
    return outs
