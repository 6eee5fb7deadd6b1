"""The calls whose time counts: the packed-prefill path as its host program runs it.

Three kinds of case, each through the package's public entry points:

  attn   one attention layer's hot path: K1 (QK RMSNorm + RoPE) then K2
         (packed attention over a cached prefix, the prefix's tail and the
         question blocks, or bidirectional rows), with the d3 readout of the
         last position where the case asks for it;
  gdn    one Gated DeltaNet layer core, from zero state (a prefix's prefill)
         or continuing a state that every row shares (question rows);
  stack  a packed pass through layers of a Qwen3-1.7B-shaped decoder stack:
         embedding, projections, norms, K1 / K2 over the device caches, SwiGLU
         and the code head (two layers: in 16 bits a rounding change grows with
         depth, and every layer is the same work).

Host programs keep the plan, the rotary table, the weights and the caches
between calls, so prepare() makes them; the per-pass block table of a stack
is built inside the pass, as the engine does.
"""
import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rust-cev_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import cev_hip  # noqa: E402
from cev_hip import configs  # noqa: E402
from cev_hip.qwen3 import Qwen3Stack  # noqa: E402

EPS = 1e-6
HIDDEN, CODES, TEMPERATURE = 2048, 255, 0.8  # the d3 readout


# ---------------------------------------------------------------------------
# The cases


def _attn(hq, hkv, d, bf16, past, tail, blocks, lo, hi, gated=False, rows=0, row_t=0, readout=False):
    """blocks question blocks of lo..hi tokens after `past` cached and `tail`
    new prefix tokens; rows > 0: bidirectional rows padded to row_t instead,
    lo..hi of their tokens real."""
    return dict(kind="attn", hq=hq, hkv=hkv, d=d, bf16=bf16, past=past, tail=tail, blocks=blocks, lo=lo, hi=hi, gated=gated, rows=rows,
                row_t=row_t, readout=readout)


def _gdn(bf16, batch, t, state):
    return dict(kind="gdn", bf16=bf16, batch=batch, t=t, nk=16, nv=32, state=state)


def _stack(bf16, layers, past, tail, questions, lo, hi):
    return dict(kind="stack", bf16=bf16, layers=layers, past=past, tail=tail, questions=questions, lo=lo, hi=hi)


def listed():
    return [
        # a single short question on a small model's layer: all latency
        dict(_attn(16, 8, 128, True, 301, 0, 1, 19, 19), name="attn_one_question"),
        # an f32 Qwen3-0.6B-shaped layer, 4 questions x 3 rotations
        dict(_attn(16, 8, 128, False, 256, 0, 12, 32, 32), name="attn_f32_rotations"),
        # a Qwen3-8B-shaped layer with a long cached prefix, a full batch of questions
        dict(_attn(32, 8, 128, True, 32768, 0, 64, 64, 64), name="attn_long_prefix"),
        # the same prefix asked one short question: streaming the K/V cache
        dict(_attn(32, 8, 128, True, 32768, 0, 1, 16, 16), name="attn_kv_stream"),
        # a Qwen3.5 gated layer, 32 question rows padded to 64 after a 4096-token prefix
        dict(_attn(16, 4, 256, True, 4096, 0, 32, 64, 64, gated=True), name="attn_gated_rows"),
        # a Qwen3.5 bidirectional row read out at its last position (d3)
        dict(_attn(16, 4, 256, True, 0, 0, 0, 8192, 8192, gated=True, rows=1, row_t=8192, readout=True), name="attn_bidirectional"),
        # the GDN layer over a 4096-token prefix
        dict(_gdn(True, 1, 4096, False), name="gdn_prefix"),
        # the GDN layer over 32 question rows that continue the prefix's state
        dict(_gdn(True, 32, 64, True), name="gdn_rows"),
        # an f32 model's GDN layer over a few rows of an odd length
        dict(_gdn(False, 3, 333, True), name="gdn_f32_odd"),
        # one question of a cached state through two layers and the code head: launches and weight reads
        dict(_stack(True, 2, 2048, 0, 1, 41, 41), name="stack_one_question"),
        # a full packed pass: the state's 512-token tail and 64 questions
        dict(_stack(True, 2, 1536, 512, 64, 48, 48), name="stack_pass"),
        # an f32 model's decoder layers over a ragged batch of questions
        dict(_stack(False, 2, 1000, 133, 20, 17, 64), name="stack_f32_layers"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attn", "attn", "attn", "gdn", "gdn", "stack"])
    if kind == "gdn":
        batch = _log(rng, 1, 32)
        return _gdn(rng.random() < 0.7, batch, _log(rng, 1, 4096 // batch), rng.random() < 0.6)
    if kind == "stack":
        bf16 = rng.random() < 0.7
        hi = rng.randint(16, 64)
        return _stack(bf16, rng.choice([1, 2]), _log(rng, 64, 2048), rng.choice([0, rng.randint(1, 512)]), _log(rng, 1, 64 if bf16 else 32),
                      rng.randint(9, hi), hi)
    form = rng.choice(["small", "f32", "large", "gated", "bidirectional"])
    hi = rng.randint(12, 96)
    lo = rng.randint(8, hi)
    tail = rng.choice([0, 0, rng.randint(1, 512)])
    if form == "small":
        return _attn(16, 8, 128, True, _log(rng, 32, 8192), tail, _log(rng, 1, 64), lo, hi)
    if form == "f32":
        return _attn(16, 8, 128, False, _log(rng, 32, 4096), tail, _log(rng, 1, 32), lo, hi)
    if form == "large":
        return _attn(32, 8, 128, True, _log(rng, 512, 32768), tail, _log(rng, 1, 48), lo, hi)
    if form == "gated":
        return _attn(16, 4, 256, True, _log(rng, 64, 8192), tail, _log(rng, 1, 48), lo, hi, gated=True)
    rows = _log(rng, 1, 16)
    t = _log(rng, 33, 8192 // rows)
    return _attn(16, 4, 256, True, 0, 0, 0, max(1, t // 2), t, gated=True, rows=rows, row_t=t, readout=rng.random() < 0.5)


# ---------------------------------------------------------------------------
# Shapes of a case


def _lengths(case, n):
    """n lengths of lo..hi, always the same for one case."""
    r = random.Random(n * 1000003 + case["lo"] * 1009 + case["hi"])
    return [r.randint(case["lo"], case["hi"]) for _ in range(n)]


def _questions(case):
    return _lengths(case, case["blocks"] if case["kind"] == "attn" else case["questions"])


def _tokens(case):
    if case["kind"] == "gdn":
        return case["batch"] * case["t"]
    if case.get("rows"):
        return case["rows"] * case["row_t"]
    return case["tail"] + sum(_questions(case))


def _pairs(case):
    """Visible (query row, key) pairs of one query head."""
    if case.get("rows"):
        t = case["row_t"]
        return sum(t * v + (t - v) for v in _lengths(case, case["rows"]))
    past, tail = case["past"], case["tail"]
    n = tail * past + tail * (tail + 1) // 2
    return n + sum(q * (past + tail) + q * (q + 1) // 2 for q in _questions(case))


def _dtype(case):
    return torch.bfloat16 if case["bf16"] else torch.float32


def work(case):
    e, t = (2 if case["bf16"] else 4), _tokens(case)
    if case["kind"] == "attn":
        hq, hkv, d = case["hq"], case["hkv"], case["d"]
        n = t * hq * d * (3 if case["gated"] else 2)      # q (and its gate) in, attention out
        n += t * hkv * d * 3 + case["past"] * hkv * d * 2  # k and v in, k out, the cached K/V
        flops = 4.0 * d * hq * _pairs(case)
        b = n * e
        if case["readout"]:
            b += HIDDEN * hq * d * e + CODES * HIDDEN * 4
            flops += 2.0 * HIDDEN * (hq * d + CODES)
        return dict(bytes=b, flops=flops)
    if case["kind"] == "gdn":
        nk, nv, dk = case["nk"], case["nv"], 128
        conv = (2 * nk + nv) * dk
        b = t * (conv + 2 * nv * dk + 2 * nv) * e + case["batch"] * (nv * dk * dk * 4 + conv * 3 * e)
        if case["state"]:
            b += nv * dk * dk * 4 + conv * 3 * e
        # the token recurrence: k S, the outer product and q S
        return dict(bytes=b, flops=6.0 * dk * dk * nv * t + 2.0 * 4 * conv * t)
    w = _stack_workload(case)
    H, inter, hq, hkv, d, L = w.hidden, w.inter, w.hq, w.hkv, w.d, w.n_layers
    per = H * (hq + 2 * hkv) * d + hq * d * H + 3 * H * inter
    b = L * (per * e + 2 * hkv * d * (case["past"] + t) * e) + t * H * e * 3
    return dict(bytes=b, flops=float(L) * (2.0 * per * t + 4.0 * d * hq * _pairs(case)))


# About four times the distance from 64 bits that the path shows.  bf16 results
# are rounded once per op (2^-9 relative each): attention is 0.5-0.8 % off, the
# GDN layer 0.6 % (its gated norm divides by the row, so single values of a
# small row are further off), two stack layers 1.2-1.8 %.
def tolerance(case):
    bf16 = case["bf16"]
    if case["kind"] == "stack":
        return {"rel": 0.03, "max": 0.4} if bf16 else {"rel": 2e-5, "max": 1e-4}
    if case["kind"] == "gdn":
        return {"rel": 0.025, "max": 0.9} if bf16 else {"rel": 6e-6, "max": 2e-4}
    if case["gated"]:
        return {"rel": 0.03, "max": 0.45}
    return {"rel": 0.02, "max": 0.15} if bf16 else {"rel": 2e-6, "max": 3e-5}


# ---------------------------------------------------------------------------
# Inputs


class _Draws:
    """Seeded tensors on the GPU."""

    def __init__(self, seed, dtype):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))
        self.dtype = dtype

    def normal(self, *shape, scale=1.0, offset=0.0, dtype=None):
        x = torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32)
        return x.mul_(scale).add_(offset).to(dtype or self.dtype)

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.g, device="cuda", dtype=torch.float32)


def _table(case):
    if case["rows"]:
        table = cev_hip.BlockTable.from_rows(case["rows"], case["row_t"], 0, causal=False, lengths=_lengths(case, case["rows"]))
        return table, torch.arange(case["row_t"], dtype=torch.int32).repeat(case["rows"])
    prefix = case["past"] + case["tail"]
    table, pos, _ = cev_hip.BlockTable.from_plans([(case["past"], prefix, case["past"])], [(0, n) for n in _questions(case)])
    return table, torch.from_numpy(pos)


def _rotary(case):
    """(theta, rotary dimensions): the Qwen3.5 layers rotate a quarter of each head."""
    return (1e7, case["d"] // 4) if case["gated"] else (1e6, case["d"])


def _attn_inputs(case, seed):
    r, hq, hkv, d, t = _Draws(seed, _dtype(case)), case["hq"], case["hkv"], case["d"], _tokens(case)
    x = dict(proj=r.normal(t, hq, 2 * d if case["gated"] else d), k=r.normal(t, hkv, d), v=r.normal(t, hkv, d))
    # Qwen3.5 stores its norm weights around zero and applies 1 + w
    off = 0.0 if case["gated"] else 1.0
    x.update(wq=r.normal(d, scale=0.1, offset=off), wk=r.normal(d, scale=0.1, offset=off))
    if case["past"]:
        x.update(pk=r.normal(hkv, case["past"], d), pv=r.normal(hkv, case["past"], d))
    if case["readout"]:
        x.update(wo=r.normal(HIDDEN, hq * d, scale=0.02), wr=r.normal(CODES, HIDDEN, scale=0.02, dtype=torch.float32))
    return x


def _gdn_inputs(case, seed):
    r, B, T, nk, nv, dk = _Draws(seed, _dtype(case)), case["batch"], case["t"], case["nk"], case["nv"], 128
    conv = (2 * nk + nv) * dk
    x = dict(mixed=r.normal(B, T, conv), z=r.normal(B, T, nv * dk))
    u = r.uniform(B, T, nv).clamp_(1e-4, 1 - 1e-4)
    x["b"] = torch.log(u / (1 - u)).to(r.dtype)                 # beta = sigmoid(b) uniform
    g = -math.log(1e-3) * r.uniform(B, T, nv)
    x["a"] = torch.log(torch.expm1(g.clamp_(min=1e-6))).to(r.dtype)  # decay e^-softplus(a) log-uniform in [1e-3, 1]
    x["conv_w"] = r.normal(conv, 4, scale=0.5)
    x["neg_a"] = -torch.ones(nv, device="cuda")
    x["dt_bias"] = torch.zeros(nv, device="cuda")
    x["norm_w"] = r.normal(dk, scale=0.1, offset=1.0, dtype=torch.float32)
    x["conv_in"] = x["s_in"] = None
    if case["state"]:  # one prefix's state, shared by every row
        x["conv_in"] = r.normal(1, conv, 3).expand(B, conv, 3)
        x["s_in"] = r.normal(1, nv, dk, dk, scale=0.1, dtype=torch.float32).expand(B, nv, dk, dk)
    return x


def _stack_workload(case):
    return configs.c2(bf16=case["bf16"], n_layers=case["layers"], state_tokens=case["past"] + case["tail"], questions=case["questions"],
                      q_len=case["hi"])


def _stack_inputs(case, seed):
    r, w = _Draws(seed, _dtype(case)), _stack_workload(case)
    weights = {name: r.normal(*shape, scale=w.std) for name, _, shape in w.weight_specs()}
    weights.update({name: r.normal(n, scale=0.1, offset=1.0) for name, n in w.norm_specs()})
    ids = torch.randint(0, w.vocab, (case["past"] + _tokens(case) + w.n_codes,), generator=torch.Generator().manual_seed(int(seed))).numpy()
    n = case["past"] + _tokens(case)
    return w, weights, ids[:n], ids[n:]


def prepare(case, seed):
    if case["kind"] == "attn":
        return _prepare_attn(case, seed)
    if case["kind"] == "gdn":
        x = _gdn_inputs(case, seed)
        layer = cev_hip.GatedDeltaNet(case["batch"], case["t"], case["nk"], case["nv"], eps=EPS, dtype=_dtype(case), device="cuda")
        return dict(kind="gdn", layer=layer, x=x)
    w, weights, ids, codes = _stack_inputs(case, seed)
    past, prefix = case["past"], case["past"] + case["tail"]
    lens = _questions(case)
    stack = Qwen3Stack(w, weights, torch.device("cuda"), capacity=prefix + sum(lens))
    stack.prefill(0, ids[:past], 512)
    items, slot = [], prefix
    for n in lens:
        items.append((0, n, slot))
        slot += n
    return dict(kind="stack", stack=stack, plans=[(0, prefix, past)], items=items, tokens=ids[past:], codes=codes)


def _prepare_attn(case, seed):
    x, d, t = _attn_inputs(case, seed), case["d"], _tokens(case)
    table, pos = _table(case)
    theta, rotary = _rotary(case)
    s = dict(kind="attn", x=x, pos=pos.cuda(), plus_one=case["gated"], q_in=x["proj"][:, :, :d],
             gate=x["proj"][:, :, d:] if case["gated"] else None, pk=x.get("pk"), pv=x.get("pv"))
    s["rot"] = cev_hip.Rotary(theta, rotary, int(pos.max()) + 1, _dtype(case), "cuda")
    s["q"], s["out"] = (torch.empty(t, case["hq"], d, dtype=_dtype(case), device="cuda") for _ in range(2))
    s["k"] = torch.empty_like(x["k"])
    s["attn"] = cev_hip.PackedAttention(s["q"], s["k"], table, k_cache=s["pk"], s_cache=case["past"], has_gate=case["gated"], out=s["out"],
                                        gate=s["gate"], v_new=x["v"], v_cache=s["pv"])
    s["readout"] = None
    if case["readout"]:
        s["readout"] = cev_hip.D3Readout(x["wo"].float().cpu().numpy(), x["wr"].cpu().numpy(), TEMPERATURE, "cuda", _dtype(case))
    return s


def run(s):
    x = s.get("x")
    if s["kind"] == "attn":
        cev_hip.qknorm_rope(s["q_in"], x["k"], x["wq"], x["wk"], s["pos"], s["rot"], EPS, plus_one=s["plus_one"], q_out=s["q"], k_out=s["k"])
        out = s["attn"](s["q"], s["k"], x["v"], s["pk"], s["pv"], s["gate"], s["out"])
        if s["readout"] is None:
            return dict(out=out, k=s["k"])
        return dict(out=out, k=s["k"], logits=s["readout"](out[-1:].view(1, -1)))
    if s["kind"] == "gdn":
        y, conv_out, s_out = s["layer"](x["mixed"], x["z"], x["b"], x["a"], x["conv_w"], x["neg_a"], x["dt_bias"], x["norm_w"],
                                        x["conv_in"], x["s_in"])
        return dict(y=y, conv_out=conv_out, s_out=s_out)
    stack = s["stack"]
    table, pos, slots, gather = cev_hip.BlockTable.from_slots(s["plans"], s["items"], stack.capacity)
    xh = stack.run(s["tokens"], pos, slots, table)
    hidden = stack.hidden(xh, gather)
    return dict(x=xh[0], h=xh[1], hidden=hidden, logits=stack.code_logits(hidden, s["codes"]))


# ---------------------------------------------------------------------------
# The same in 64 bits


def _rms(x, w):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w


def _rope(x, pos, theta, rotary):
    """Rotate-half over the first `rotary` of (t, heads, d); frequencies and
    angles in f32, which is how the model's table defines them."""
    half = rotary // 2
    inv = 1.0 / (torch.tensor(theta, dtype=torch.float64) ** (torch.arange(half, dtype=torch.float64) * 2 / rotary)).float()
    ang = (pos.float().cpu()[:, None] * inv).double().to(x.device)[:, None, :]
    a, b = x[..., :half], x[..., half:rotary]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin(), x[..., rotary:]], -1)


def _attend(q, k, v, pieces):
    """q (t, hq, d) over k, v (keys, hkv, d).  pieces: (rows, full key ranges,
    local key range, local mask or None)."""
    t, hq, d = q.shape
    hkv = k.shape[1]
    out = torch.zeros_like(q)
    for rows, spans, local, mask in pieces:
        n = rows.stop - rows.start
        at = torch.cat([torch.arange(a, b, device=q.device) for a, b in spans + [local]])
        m = local[1] - local[0]
        for h in range(hkv):
            qs = q[rows, h * (hq // hkv):(h + 1) * (hq // hkv)].reshape(-1, d)
            s = qs @ k[at, h].t().contiguous() / math.sqrt(d)
            if mask is not None:
                s.view(n, hq // hkv, -1)[:, :, at.numel() - m:].masked_fill_(~mask[:, None, :], -math.inf)
            out[rows, h * (hq // hkv):(h + 1) * (hq // hkv)] = (torch.softmax(s, -1) @ v[at, h]).view(n, -1, d)
    return out


def _pieces(case, key0):
    """_attend's pieces of a packed pass; new token i is key key0 + i."""
    dev = "cuda"
    out = []
    if case.get("rows"):
        t = case["row_t"]
        for i, n in enumerate(_lengths(case, case["rows"])):
            j = torch.arange(t, device=dev)
            mask = (j < n)[None, :] | ((j[:, None] >= n) & (j[None, :] == j[:, None]))
            for a in range(0, t, 2048):
                b = min(t, a + 2048)
                out.append((slice(i * t + a, i * t + b), [], (i * t, i * t + t), mask[a:b]))
        return out
    past, tail = case["past"], case["tail"]
    tri = lambda n: torch.ones(n, n, dtype=torch.bool, device=dev).tril()  # noqa: E731
    at = 0
    if tail:
        out.append((slice(0, tail), [(0, past)], (key0, key0 + tail), tri(tail)))
        at = tail
    for n in _questions(case):
        spans = [(0, past)] + ([(key0, key0 + tail)] if tail else [])
        out.append((slice(at, at + n), spans, (key0 + at, key0 + at + n), tri(n)))
        at += n
    return out


def _exact_attn(case, seed):
    x = {n: v.double() for n, v in _attn_inputs(case, seed).items()}
    d, t = case["d"], _tokens(case)
    _, pos = _table(case)
    theta, rotary = _rotary(case)
    plus = 1.0 if case["gated"] else 0.0
    q = _rope(_rms(x["proj"][:, :, :d], x["wq"] + plus), pos, theta, rotary)
    k = _rope(_rms(x["k"], x["wk"] + plus), pos, theta, rotary)
    ks, vs = k, x["v"]
    if case["past"]:
        ks, vs = torch.cat([x["pk"].transpose(0, 1), k]), torch.cat([x["pv"].transpose(0, 1), x["v"]])
    out = _attend(q, ks, vs, _pieces(case, case["past"]))
    if case["gated"]:
        out = out * torch.sigmoid(x["proj"][:, :, d:])
    got = dict(out=out, k=k)
    if case["readout"]:
        got["logits"] = out[t - 1].reshape(1, -1) @ x["wo"].t().contiguous() @ x["wr"].t().contiguous() / TEMPERATURE
    return got


def _exact_gdn(case, seed):
    x = _gdn_inputs(case, seed)
    x = {n: None if v is None else v.double() for n, v in x.items()}
    B, T, nk, nv, dk = case["batch"], case["t"], case["nk"], case["nv"], 128
    mixed = x["mixed"].transpose(1, 2)  # (B, channels, T)
    tail = torch.zeros(B, mixed.shape[1], 3, dtype=torch.float64, device="cuda") if x["conv_in"] is None else x["conv_in"]
    seq = torch.cat([tail, mixed], 2)
    c = sum(seq[:, :, u:u + T] * x["conv_w"][None, :, u, None] for u in range(4))
    c = (c * torch.sigmoid(c)).transpose(1, 2)
    unit = lambda y: y / (y.square().sum(-1, keepdim=True) + 1e-6).sqrt()  # noqa: E731
    rep = nv // nk
    q = unit(c[:, :, :nk * dk].reshape(B, T, nk, dk)).repeat_interleave(rep, 2) * dk ** -0.5
    k = unit(c[:, :, nk * dk:2 * nk * dk].reshape(B, T, nk, dk)).repeat_interleave(rep, 2)
    v = c[:, :, 2 * nk * dk:].reshape(B, T, nv, dk)
    beta = torch.sigmoid(x["b"])
    decay = torch.exp(x["neg_a"] * torch.nn.functional.softplus(x["a"] + x["dt_bias"]))
    S = torch.zeros(B, nv, dk, dk, dtype=torch.float64, device="cuda") if x["s_in"] is None else x["s_in"].clone()
    core = torch.empty(B, T, nv, dk, dtype=torch.float64, device="cuda")
    for i in range(T):  # the token recurrence
        S = S * decay[:, i, :, None, None]
        ki = k[:, i, :, :, None]
        dv = (v[:, i] - (ki * S).sum(2)) * beta[:, i, :, None]
        S = S + ki * dv[:, :, None, :]
        core[:, i] = (q[:, i, :, :, None] * S).sum(2)
    z = x["z"].view(B, T, nv, dk)
    y = _rms(core, x["norm_w"]) * z * torch.sigmoid(z)
    return dict(y=y.reshape(B, T, nv * dk), conv_out=seq[:, :, T:], s_out=S)


def _exact_stack(case, seed):
    """Every token of the state and of the questions in one pass: the cached
    part as a first, causal block."""
    w, weights, ids, codes = _stack_inputs(case, seed)
    past, prefix, lens = case["past"], case["past"] + case["tail"], _questions(case)
    dev, hq, hkv, d = "cuda", w.hq, w.hkv, w.d
    pos = torch.cat([torch.arange(prefix)] + [prefix + torch.arange(n) for n in lens])
    tri = torch.ones(past, past, dtype=torch.bool, device=dev).tril()
    pieces = [(slice(0, past), [], (0, past), tri)]
    for rows, spans, local, mask in _pieces(case, past):
        pieces.append((slice(rows.start + past, rows.stop + past), spans, local, mask))
    W = lambda name: weights[name].double()  # noqa: E731
    mul = lambda y, name: y @ W(name).t().contiguous()  # noqa: E731
    embed = weights["embed"]
    x = embed[torch.from_numpy(ids).to(dev)].double()
    for i in range(w.n_layers):
        p = f"l{i}."
        y = _rms(x, W(p + "ln1"))
        q, k, v = mul(y, p + "wq").view(-1, hq, d), mul(y, p + "wk").view(-1, hkv, d), mul(y, p + "wv").view(-1, hkv, d)
        q, k = (_rope(_rms(a, W(p + n)), pos, w.theta, d) for a, n in ((q, "q_norm"), (k, "k_norm")))
        x = x + mul(_attend(q, k, v, pieces).reshape(-1, hq * d), p + "wo")
        y = _rms(x, W(p + "ln2"))
        g = mul(y, p + "gate")
        h = mul(g * torch.sigmoid(g) * mul(y, p + "up"), p + "down")
        if i + 1 < w.n_layers:
            x = x + h
    last = torch.tensor(lens).cumsum(0) + prefix - 1
    hidden = _rms((x + h)[last.to(dev)], W("norm"))
    head = embed[torch.from_numpy(codes).to(dev)].double()
    return dict(x=x[past:], h=h[past:], hidden=hidden, logits=hidden @ head.t().contiguous())


def exact(case, seed):
    return {"attn": _exact_attn, "gdn": _exact_gdn, "stack": _exact_stack}[case["kind"]](case, seed)
