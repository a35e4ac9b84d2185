"""The work a user of this library has it do, as cases that can be timed.

A block is loaded from a checkpoint (ISQ: f32 rows quantised to GGUF on the
device), then serves one-token and batched decode steps, prompt chunks of the
512 tokens the daemon cuts prompts into, and whole prompts. Sizes are the
80B-A3B layer's (hidden 2048, 512 experts, top-10, intermediate 512, a shared
expert of 512), the small f32 block of the parity tests, and for drawn cases
other expert counts (an expert-parallel rank's share among them) and widths.

Weights are N(0, 0.02) drawn from the seed and packed to GGUF here with plain
torch; tokens are N(0, 1), with a direction all tokens share where `skew` is
set, which makes some experts popular, as trained routers do.
"""
from __future__ import annotations

import math

import torch

from helexa_amd import moe

Q8_0, Q4_K, Q6_K, BF16, F32 = moe.Q8_0, moe.Q4_K, moe.Q6_K, moe.BF16, moe.F32
# format of (gate and up, down), and of the router rows
MIXES = {"q8_0": (Q8_0, Q8_0, BF16), "q4_k_m": (Q4_K, Q6_K, BF16), "bf16": (BF16, BF16, BF16), "f32": (F32, F32, F32)}
QUANT = {"q8_0": Q8_0, "q4_k": Q4_K, "q6_k": Q6_K}
BLOCK_BYTES = {Q8_0: 34 / 32, Q4_K: 144 / 256, Q6_K: 210 / 256, BF16: 2.0, F32: 4.0}
EPS = 1e-6
QUANT_M = 64   # rows of an expert call up to which activations are quantised to the weights' vec_dot type


# ---------------------------------------------------------------- the cases
def _block(name, op, mix, tokens, layers=1, skew=0.0, hidden=2048, experts=512, topk=10, inter=512):
    c = dict(op=op, mix=mix, tokens=tokens, layers=layers, skew=skew, hidden=hidden, experts=experts, topk=topk,
             inter=inter)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # the smallest block anyone runs: the f32 parity configuration, a few tokens
        _block("tiny_f32_4", "forward", "f32", 4, hidden=256, experts=16, topk=4, inter=128),
        # one sequence generating: one token through one layer, 8-bit experts
        _block("decode1_q8", "forward", "q8_0", 1),
        # one sequence through consecutive decoder layers (norm, block, residual), the 4-bit mix
        _block("decode1_stack_q4km", "decoder", "q4_k_m", 1, layers=4),
        # eight sequences generating together
        _block("decode8_stack_q4km", "decoder", "q4_k_m", 8, layers=4),
        # one sequence on the checkpoint's own bf16 weights (no ISQ)
        _block("decode1_bf16", "forward", "bf16", 1),
        # a serving batch past the decode kernels, or a short prompt
        _block("batch27_q4km", "decoder", "q4_k_m", 27),
        # the daemon's prompt chunk, 4-bit mix, uneven experts
        _block("chunk512_q4km", "decoder", "q4_k_m", 512, skew=1.0),
        # the same chunk with 8-bit experts
        _block("chunk512_q8", "forward", "q8_0", 512, skew=1.0),
        # a prompt tail of odd length on bf16 weights
        _block("prompt301_bf16", "forward", "bf16", 301, skew=1.0),
        # a whole prompt in one call, 4-bit mix and 8-bit
        _block("prompt3001_q4km", "forward", "q4_k_m", 3001, skew=1.0),
        _block("prompt2048_q8", "forward", "q8_0", 2048, skew=1.0),
        # ISQ at load: a slice of an expert stack (64 experts of 512 x 2048) to 4 bits
        dict(name="isq_q4k", op="quantize", to="q4_k", rows=64 * 512, cols=2048),
    ]


def draw(rng):
    r = rng.random()
    if r < 0.2:   # ISQ of a projection stack
        cols = rng.choice([256, 512, 768, 1024, 2048, 4096])
        elems = math.exp(rng.uniform(math.log(1 << 16), math.log(64 * 512 * 2048)))
        return dict(op="quantize", to=rng.choice(sorted(QUANT)), rows=max(1, int(elems / cols)), cols=cols)
    if r < 0.3:   # small f32 blocks
        return _block(None, "forward", "f32", int(math.exp(rng.uniform(0, math.log(256)))),
                      hidden=rng.choice([128, 256, 512]), experts=rng.choice([8, 16, 32]), topk=rng.choice([2, 4]),
                      inter=rng.choice([64, 128, 256]))
    mix = rng.choice(["q4_k_m", "q4_k_m", "q8_0", "q8_0", "bf16"])
    tokens = int(math.exp(rng.uniform(0, math.log(500 if mix == "bf16" else 3000))))
    hidden, experts, topk, inter = 2048, 512, 10, 512
    if rng.random() < 0.5:
        hidden, inter = rng.choice([1024, 1536, 2048]), rng.choice([256, 512, 768, 1024])
        experts, topk = rng.choice([64, 128, 256]), rng.choice([4, 6, 8, 10])
    return _block(None, rng.choice(["forward", "decoder"]), mix, tokens, skew=rng.choice([0.0, 1.0]), hidden=hidden,
                  experts=experts, topk=topk, inter=inter)


# ---------------------------------------------------------------- GGUF packing
def _u8(t):
    return t.contiguous().view(torch.uint8)


def _rows(blocks, rows):
    return blocks.reshape(rows, -1)


def _pack_q8_0(w):
    x = w.reshape(-1, 32)
    d = (x.abs().amax(1, keepdim=True) / 127).half()
    q = torch.round(x / d.float().clamp_min(1e-12)).clamp_(-127, 127).to(torch.int8)
    return _rows(torch.cat([_u8(d), _u8(q)], 1), w.shape[0])


def _unpack_q8_0(b):
    b = b.reshape(-1, 34)
    return _u8(b[:, :2]).view(torch.float16).double() * _u8(b[:, 2:]).view(torch.int8).double()


def _pack_q4_k(w):
    x = w.reshape(-1, 8, 32)
    lo = x.amin(2).clamp_max(0)
    scale = (x.amax(2) - lo) / 15
    d = (scale.amax(1, keepdim=True) / 63).half()
    dm = ((-lo).amax(1, keepdim=True) / 63).half()
    df, dmf = d.float().clamp_min(1e-12), dm.float().clamp_min(1e-12)
    sc = torch.round(scale / df).clamp_(0, 63)
    mn = torch.round(-lo / dmf).clamp_(0, 63)
    q = torch.round((x + (dmf * mn)[:, :, None]) / (df * sc).clamp_min(1e-12)[:, :, None]).clamp_(0, 15).to(torch.uint8)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    s = torch.cat([sc[:, :4] | ((sc[:, 4:] >> 4) << 6), mn[:, :4] | ((mn[:, 4:] >> 4) << 6),
                   (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)
    qs = (q[:, 0::2] | (q[:, 1::2] << 4)).reshape(-1, 128)
    return _rows(torch.cat([_u8(d), _u8(dm), s, qs], 1), w.shape[0])


def _unpack_q4_k(b):
    b = b.reshape(-1, 144)
    d, dm = _u8(b[:, :2]).view(torch.float16).double(), _u8(b[:, 2:4]).view(torch.float16).double()
    s, qs = b[:, 4:16], b[:, 16:].reshape(-1, 4, 32)
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
    return (d * sc)[:, :, None] * q - (dm * mn)[:, :, None]


def _pack_q6_k(w):
    x = w.reshape(-1, 16, 16)
    scale = x.abs().amax(2) / 31
    d = (scale.amax(1, keepdim=True) / 127).half()
    df = d.float().clamp_min(1e-12)
    sc = torch.round(scale / df).clamp_(0, 127)
    q = (torch.round(x / (df * sc).clamp_min(1e-12)[:, :, None]).clamp_(-32, 31) + 32).to(torch.uint8)
    q = q.reshape(-1, 2, 4, 32)   # halves, quarters
    ql = torch.cat([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
    qh = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
    return _rows(torch.cat([ql.reshape(-1, 128), qh.reshape(-1, 64), _u8(sc.to(torch.int8)), _u8(d)], 1), w.shape[0])


def _unpack_q6_k(b):
    b = b.reshape(-1, 210)
    ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
    sc, d = _u8(b[:, 192:208]).view(torch.int8).double(), _u8(b[:, 208:]).view(torch.float16).double()
    q = torch.stack([(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                     (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 1] >> 4) | ((qh >> 6) << 4)], 2)
    return (d * sc)[:, :, None] * (q.reshape(-1, 16, 16).double() - 32)


_PACK = {Q8_0: _pack_q8_0, Q4_K: _pack_q4_k, Q6_K: _pack_q6_k, BF16: lambda w: w.bfloat16(), F32: lambda w: w}
_UNPACK = {Q8_0: _unpack_q8_0, Q4_K: _unpack_q4_k, Q6_K: _unpack_q6_k, BF16: lambda b: b.double(),
           F32: lambda b: b.double()}


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _stack(g, fmt, count, rows, cols):
    parts = []
    step = max(1, (1 << 26) // (rows * cols))   # matrices packed at a time
    for at in range(0, count, step):
        n = min(step, count - at)
        w = torch.randn((n * rows, cols), generator=g, device="cuda").mul_(0.02)
        parts.append(_PACK[fmt](w).reshape(n, rows, -1))
    return torch.cat(parts) if len(parts) > 1 else parts[0]


def _layer(c, seed):
    H, E, I = c["hidden"], c["experts"], c["inter"]
    gu, dn, rt = MIXES[c["mix"]]
    g = _gen(seed)
    w = {"router": (rt, _stack(g, rt, 1, E, H)[0]), "seg": (rt, _stack(g, rt, 1, 1, H)[0])}
    for key, fmt, n, r, k in (("gate", gu, E, I, H), ("up", gu, E, I, H), ("down", dn, E, H, I), ("sgate", gu, 1, I, H),
                              ("sup", gu, 1, I, H), ("sdown", dn, 1, H, I)):
        w[key] = (fmt, _stack(g, fmt, n, r, k))
    w["norm"] = torch.randn(H, generator=g, device="cuda") * 0.1   # the norm multiplies by 1 + this
    return w


def _tokens(c, seed):
    g = _gen(seed + 1)
    x = torch.randn((c["tokens"], c["hidden"]), generator=g, device="cuda")
    if c["skew"]:
        x += c["skew"] * torch.randn(c["hidden"], generator=g, device="cuda")
    return x if c["mix"] == "f32" else x.bfloat16()


def _weight_seed(seed, layer):
    return seed * 64 + 7 + layer


def _floats(c, seed):
    return torch.randn((c["rows"], c["cols"]), generator=_gen(seed), device="cuda").mul_(0.02)


def prepare(case, seed):
    c = case
    if c["op"] == "quantize":
        return {"case": c, "src": _floats(c, seed)}
    cfg = moe.TextConfig(hidden_size=c["hidden"], num_experts=c["experts"], num_experts_per_tok=c["topk"],
                         moe_intermediate_size=c["inter"], shared_expert_intermediate_size=c["inter"],
                         norm_topk_prob=True, num_hidden_layers=c["layers"], rms_norm_eps=EPS)
    blocks, norms = [], []
    for i in range(c["layers"]):
        w = _layer(c, _weight_seed(seed, i))
        norms.append(w.pop("norm"))
        blocks.append(moe.Qwen3_5MoeBlock.load(cfg, w, act_dtype=F32 if c["mix"] == "f32" else BF16))
        del w
    x = _tokens(c, seed)
    ws = torch.empty(max(1, blocks[0].workspace_size(c["tokens"])), dtype=torch.uint8, device="cuda")
    return {"case": c, "blocks": blocks, "norms": norms, "x": x, "ws": ws, "out": torch.empty_like(x)}


def run(state):
    c = state["case"]
    if c["op"] == "quantize":
        return moe.quantize(QUANT[c["to"]], state["src"])
    if c["op"] == "forward":
        return state["blocks"][0].forward(state["x"], workspace=state["ws"], out=state["out"])
    h = state["out"].copy_(state["x"])   # the residual stream the attention half leaves
    for b, nw in zip(state["blocks"], state["norms"]):
        b.decoder_mlp_(h, nw, EPS, workspace=state["ws"])
    return h


# ---------------------------------------------------------------- what it needs
def _touched(c):
    """experts at least one token chooses, on average: a logit is N(0, 1) plus the shared direction's
    part, N(0, skew); the top-k threshold follows from the mean popularity k / E"""
    E, T, p = c["experts"], c["tokens"], c["topk"] / c["experts"]
    if not c["skew"]:
        return E * (1 - (1 - p) ** T)
    n = 201
    zs = [-5 + 10 * i / (n - 1) for i in range(n)]
    ws = [math.exp(-z * z / 2) for z in zs]
    tot = sum(ws)
    pop = lambda thr: [0.5 * math.erfc((thr - c["skew"] * z) / math.sqrt(2)) for z in zs]
    lo, hi = -10.0, 10.0
    for _ in range(60):
        mid = (lo + hi) / 2
        mean = sum(w * q for w, q in zip(ws, pop(mid))) / tot
        lo, hi = (mid, hi) if mean > p else (lo, mid)
    return E * sum(w * (1 - (1 - q) ** T) for w, q in zip(ws, pop(lo))) / tot


def work(case):
    c = case
    if c["op"] == "quantize":
        n = c["rows"] * c["cols"]   # a magnitude or range search, a scaling and a rounding each
        return {"bytes": n * (4 + BLOCK_BYTES[QUANT[c["to"]]]), "flops": 4 * n}
    H, E, I, T, k = c["hidden"], c["experts"], c["inter"], c["tokens"], c["topk"]
    gu, dn, rt = MIXES[c["mix"]]
    expert = 2 * H * I * BLOCK_BYTES[gu] + H * I * BLOCK_BYTES[dn]
    act = BLOCK_BYTES[F32 if c["mix"] == "f32" else BF16]
    per_layer = (_touched(c) + 1) * expert + (E + 1) * H * BLOCK_BYTES[rt] + (4 * H if c["op"] == "decoder" else 0)
    return {"bytes": c["layers"] * (per_layer + 2 * T * H * act),
            "flops": c["layers"] * (6 * T * (k + 1) * H * I + 2 * T * (E + 1) * H)}


# ---------------------------------------------------------------- how close
# about four times the distance between the library's results and exact()
def tolerance(case):
    c = case
    if c["op"] == "quantize":
        return "exact"        # bytes
    if c["mix"] == "f32":
        return {"rel": 1e-6}   # 1.5e-7 seen, sums of up to 512 terms
    # bf16 outputs: 0.16 % to 0.28 % seen for one block, 0.38 % for a small one; 0.53 % over four layers
    return {"rel": 2e-2 if c["layers"] > 1 else 1e-2}


def _round_away(v):
    return torch.trunc(v + torch.copysign(torch.full_like(v, 0.5), v))


def _codes(x, wfmt):
    """rows quantised as a GGUF linear of wfmt weights quantises its activations, dequantised again"""
    x = x.float()
    if wfmt == Q8_0:
        b = x.reshape(x.shape[0], -1, 32)
        d = b.abs().amax(2, keepdim=True) / 127
        q = _round_away((b * torch.where(d != 0, 1 / d, torch.zeros_like(d))).double())
        return (q * d.half().double()).reshape(x.shape)
    b = x.reshape(x.shape[0], -1, 256)
    mx = torch.gather(b, 2, b.abs().argmax(2, keepdim=True))
    isc = -128 / mx
    q = _round_away((b * isc).double()).clamp_max(127)
    return torch.where(mx != 0, q / isc.double(), torch.zeros_like(q)).reshape(x.shape)


def _expert(c, x, gate, up, down):
    """silu(x Wg^T) * (x Wu^T), times Wd^T, for the rows of one expert call"""
    gu, dn, _ = MIXES[c["mix"]]
    G, U = (_UNPACK[gu](w).reshape(c["inter"], c["hidden"]) for w in (gate, up))
    D = _UNPACK[dn](down).reshape(c["hidden"], c["inter"])
    f16 = lambda t: t.half().double()
    silu = torch.nn.functional.silu
    if gu in (BF16, F32):
        return (silu(x @ G.T) * (x @ U.T)) @ D.T
    if x.shape[0] <= QUANT_M:
        xq = _codes(x, gu)
        return _codes(silu(xq @ G.T) * (xq @ U.T), dn) @ D.T
    xh = f16(x)
    h = f16(silu(f16(xh @ f16(G).T)) * f16(xh @ f16(U).T))
    return f16(h @ f16(D).T)


def _exact_block(c, w, x):
    """x [T, H] f64 holding act-dtype values -> the block's output in f64"""
    act = torch.float32 if c["mix"] == "f32" else torch.bfloat16
    logits = (x @ w["router"][1].double().T).to(act).double()
    top, idx = torch.sort(logits, dim=1, descending=True, stable=True)   # ties to the lower expert
    k = c["topk"]
    p = torch.softmax(top, 1)[:, :k]
    p = p / p.sum(1, keepdim=True)
    idx = idx[:, :k]
    y = torch.zeros_like(x)
    for e in torch.unique(idx).tolist():
        t, j = torch.nonzero(idx == e, as_tuple=True)
        y[t] += p[t, j, None] * _expert(c, x[t], w["gate"][1][e], w["up"][1][e], w["down"][1][e])
    sg = torch.sigmoid((x @ w["seg"][1].double().T).to(act).double())
    return y + sg * _expert(c, x, w["sgate"][1][0], w["sup"][1][0], w["sdown"][1][0])


def exact(case, seed):
    c = case
    if c["op"] == "quantize":
        return None   # bytes: compared as they are
    x = _tokens(c, seed)
    act = x.dtype
    h = x.double()
    for i in range(c["layers"]):
        w = _layer(c, _weight_seed(seed, i))
        if c["op"] == "forward":
            return _exact_block(c, w, h)
        n = h * torch.rsqrt((h * h).mean(1, keepdim=True) + EPS) * (1 + w["norm"].double())
        # the block sees activations of the stream's type and adds its output to it
        h = h + _exact_block(c, w, n.to(act).double())
        if i + 1 < c["layers"]:
            h = h.to(act).double()
    return h
