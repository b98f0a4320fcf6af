"""The workloads that stand for this framework's use, and how their results are checked.

Two engines, as a program of a user drives them:

* `llama_step` / `llama_prompt`: the W4A8KV4 path (qserve_amd.decode.DecodeEngine: packed 4-bit weights, int8 activations, 4- or
  8-bit paged cache) on a stack of Llama-shaped layers with that shape's own widths.  A step is one token per sequence, replayed
  from the engine's graph; a prompt is the whole prompt phase up to the first sampled token.
* `serve_prompt` / `serve_decode`: served models (qserve_amd.serving.Engine, bfloat16) at the sizes of the repository's benchmark.
  A prompt is one `execute` over whole prompts whose last positions are scored; a decode case opens its sequences, runs their
  prompts and then one token per sequence and step, and closes them.

The layers of a stack are alike, so a few of them stand for a model of any depth: four where each step has to stream weights that no
cache still holds, one for a prompt, whose products hide them.
"""
import math

import torch

from qserve_amd.decode import LLAMA2_7B, LLAMA3_8B, DecodeEngine
from qserve_amd.serving import bench as designs
from qserve_amd.serving.engine import Engine
from qserve_amd.serving.registry import resolve_model

F64 = torch.float64
DEV = "cuda:0"
LAYERS = {"llama_step": 4, "llama_prompt": 1, "serve_prompt": designs.LAYERS, "serve_decode": designs.LAYERS}
SCORED = 64                       # positions at the end of a prompt whose logits are asked for
SHAPES = {"llama3_8b": LLAMA3_8B, "llama2_7b": LLAMA2_7B}
DESIGNS = ("Vekalorn", "Mumelix", "Rivolix")


def listed():
    return [
        # one user at the keyboard: nothing but launches and the weights' stream
        dict(name="llama_step_1", kind="llama_step", shape="llama3_8b", batch=1, context=333, spread=0.0, group=-1, kv_bits=4),
        # the reference's serving batch in the middle of a generation, per-channel weights
        dict(name="llama_step_64", kind="llama_step", shape="llama3_8b", batch=64, context=1281, spread=0.2, group=-1, kv_bits=4),
        # the large batch with group-quantised weights
        dict(name="llama_step_128_g128", kind="llama_step", shape="llama3_8b", batch=128, context=1037, spread=0.1, group=128, kv_bits=4),
        # few long conversations over an 8-bit cache
        dict(name="llama_step_8_kv8_long", kind="llama_step", shape="llama3_8b", batch=8, context=7700, spread=0.1, group=-1, kv_bits=8),
        # prompt phase of a batch
        dict(name="llama_prompt_8x1024", kind="llama_prompt", shape="llama3_8b", batch=8, tokens=1024, group=-1, kv_bits=4),
        # odd prompts, group-quantised weights, one key / value head per query head, 8-bit cache
        dict(name="llama_prompt_3x1777_g128", kind="llama_prompt", shape="llama2_7b", batch=3, tokens=1777, group=128, kv_bits=8),
        # latent attention and small experts: a batch of prompts in one step
        dict(name="vekalorn_prompt_8x1024", kind="serve_prompt", design="Vekalorn", size="w2048", seqs=8, tokens=1024, spread=0.0),
        # the same model answering 64 short requests
        dict(name="vekalorn_decode_64", kind="serve_decode", design="Vekalorn", size="w2048", seqs=64, tokens=100, spread=0.5, steps=24),
        # recurrent and attention mixers on two streams, the wide size, prompts of different lengths
        dict(name="mumelix_prompt_8x1024_wide", kind="serve_prompt", design="Mumelix", size="w4096", seqs=8, tokens=1024, spread=0.3),
        # the same layers at the small size, a medium batch
        dict(name="mumelix_decode_16", kind="serve_decode", design="Mumelix", size="w2048", seqs=16, tokens=200, spread=0.5, steps=24),
        # one long odd prompt through differential and tied attention, weighted expert inputs and a shared expert
        dict(name="rivolix_prompt_1x2047", kind="serve_prompt", design="Rivolix", size="w2048", seqs=1, tokens=2047, spread=0.0),
        # one user's answer: every step is launches and the chosen experts' weights
        dict(name="rivolix_decode_1", kind="serve_decode", design="Rivolix", size="w2048", seqs=1, tokens=333, spread=0.0, steps=24),
    ]


def _between(rng, lo, hi):
    """An integer from [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("llama_step", "llama_prompt", "serve_prompt", "serve_decode"))
    if kind.startswith("llama"):
        shape, group, bits = rng.choice(("llama3_8b", "llama2_7b")), rng.choice((-1, 128)), rng.choice((4, 8))
        if kind == "llama_step":
            batch = _between(rng, 1, 128)
            context = _between(rng, 40, min(7900, 160000 // batch if shape == "llama3_8b" else 50000 // batch))
            return dict(kind=kind, shape=shape, batch=batch, context=context, spread=round(rng.uniform(0.0, 0.6), 2), group=group, kv_bits=bits)
        tokens = _between(rng, 33, 4100)
        return dict(kind=kind, shape=shape, batch=_between(rng, 1, max(1, 8000 // tokens)) if tokens > 125 else rng.randint(1, 64),
                    tokens=tokens, group=group, kv_bits=bits)
    design, size = rng.choice(DESIGNS), rng.choice(("w2048", "w2048", "w4096"))
    if kind == "serve_prompt":
        tokens = _between(rng, 65, 4100)
        return dict(kind=kind, design=design, size=size, seqs=_between(rng, 1, min(64, max(1, 8000 // tokens))), tokens=tokens,
                    spread=round(rng.uniform(0.0, 0.5), 2))
    return dict(kind=kind, design=design, size="w2048", seqs=_between(rng, 1, 64), tokens=_between(rng, 20, 105), spread=round(rng.uniform(0.0, 0.5), 2),
                steps=rng.randint(8, 20))


def _lengths(n, top, spread):
    """n lengths from `top` down to about (1 - spread) top."""
    return [max(2, top - int(spread * top * i / n)) for i in range(n)]


# ---- the W4A8KV4 stack -------------------------------------------------------------------------------------------------------

def _shape(case):
    return dict(SHAPES[case["shape"]], layers=LAYERS[case["kind"]])


def _llama_gen(seed):
    return torch.Generator(device=DEV).manual_seed(1000003 * seed + 17)


def _llama_linear(g, n, k, group, size=1.0):
    """A quantised projection as a checkpoint holds it: random nibbles, zero points near the middle, scales that keep outputs of
    the order of `size`."""
    d = {"qweight": torch.randint(-128, 128, (n, k // 2), dtype=torch.int8, device=DEV, generator=g)}
    unit = size / (4.6 * math.sqrt(k))
    if group == -1:
        d["s1_scales"] = ((torch.rand((n,), device=DEV, generator=g) + 0.5) * unit).half()
        d["s1_szeros"] = (torch.randint(7, 9, (n,), device=DEV, generator=g).half() * d["s1_scales"]).half()
    else:
        d["s1_scales"] = ((torch.rand((n,), device=DEV, generator=g) + 0.5) * unit / 6.0).half()
        d["s2_scales"] = torch.randint(3, 10, (k // 128, n), dtype=torch.int8, device=DEV, generator=g)
        zero = torch.randint(7, 9, (k // 128, n), dtype=torch.int8, device=DEV, generator=g)
        d["s2_zeros"] = (-(zero.int() * d["s2_scales"].int())).to(torch.int8)
    return d


def _llama_weights(case, seed, with_head):
    c, g = _shape(case), _llama_gen(seed)
    D, I, H, G = c["hidden"], c["inter"], c["heads"], c["kv_heads"]
    gain = lambda: (torch.rand((D,), device=DEV, generator=g) * 0.5 + 0.75).half()      # noqa: E731
    lin = lambda n, k, size=1.0: _llama_linear(g, n, k, case["group"], size)            # noqa: E731
    # (a layer adds less to the residual stream than the stream holds)
    W = {"layers": [dict(ln1=gain(), ln2=gain(), qkv=lin((H + 2 * G) * 128, D), o=lin(D, H * 128, 0.2), gate_up=lin(2 * I, D), down=lin(D, I, 0.2))
                    for _ in range(c["layers"])], "norm": gain()}
    if with_head:
        W["embed"] = torch.randn((c["vocab"], D), dtype=torch.float16, device=DEV, generator=g)
        W["lm_head"] = torch.randn((c["vocab"], D), dtype=torch.float16, device=DEV, generator=g) * (1.0 / math.sqrt(D))
    return W


def _llama_step_inputs(case, seed):
    """-> lengths (the new token included), hidden states [B, D], per layer the projections [sum of (length - 1), qkv] whose keys and
    values fill the cache."""
    c, g = _shape(case), _llama_gen(seed + 500009)
    lens = _lengths(case["batch"], case["context"], case["spread"])
    n = (c["heads"] + 2 * c["kv_heads"]) * 128
    hidden = torch.randn((case["batch"], c["hidden"]), dtype=torch.float16, device=DEV, generator=g)
    past = (torch.randn((sum(lens) - len(lens), n), dtype=torch.float16, device=DEV, generator=g) for _ in range(c["layers"]))
    return lens, hidden, past


def _prepare_llama_step(case, seed):
    import qserve_backend.fused_attention as fa
    c, B = _shape(case), case["batch"]
    lens, hidden, past = _llama_step_inputs(case, seed)
    eng = DecodeEngine(c, B, max(lens), 1, case["group"], case["kv_bits"] == 4, DEV, seed, with_lm_head=False, weights=_llama_weights(case, seed, False))
    held = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device=DEV)
    cu = torch.cat([held.new_zeros(1), held.cumsum(0, dtype=torch.int32)])
    top = max(lens) - 1
    pad = fa.compute_padding_offsets(cu, top, int(sum(lens) - B))
    for li, rows in enumerate(past):
        fa.apply_bias_rope_update_kv_cache(rows, held, pad, eng.tables[li], eng.H, eng.Hkv, top, 64, eng.size_per_token, 128, c["rope_theta"], 8192,
                                           True, eng.int4, True)
    eng.lengths.copy_(held + 1)
    eng.hidden.copy_(hidden)
    eng.capture()
    return dict(case=case, engine=eng, hidden=hidden, lengths=held + 1)


def _run_llama_step(st):
    eng = st["engine"]
    eng.hidden.copy_(st["hidden"])
    eng.lengths.copy_(st["lengths"])
    eng.run()
    return {"final": eng.final, "hidden": eng.hidden, "cache": [p for pools in eng.pools for p in pools]}


def _llama_prompt_tokens(case, seed):
    return torch.randint(0, _shape(case)["vocab"], (case["batch"] * case["tokens"],), device=DEV, generator=_llama_gen(seed + 500009))


def _prepare_llama_prompt(case, seed):
    eng = DecodeEngine(_shape(case), case["batch"], case["tokens"], 1, case["group"], case["kv_bits"] == 4, DEV, seed,
                       weights=_llama_weights(case, seed, True))
    return dict(case=case, engine=eng, tokens=_llama_prompt_tokens(case, seed))


def _run_llama_prompt(st):
    eng = st["engine"]
    eng.prefill(st["case"]["tokens"], st["tokens"])
    return {"final": eng.final, "hidden": eng.hidden, "cache": [p for pools in eng.pools for p in pools]}


# the same in 64 bits: the path's own integers (weights, per-token activations, cache) are part of what it computes

def _nibbles(q):
    """Packed [N, K / 2] -> the 4-bit values [N, K]: bytes run over (32 rows, 32 columns), c, e, d, b, f with row = 16 a + 8 b + c and
    column = 16 d + 4 e + f, a in the nibble."""
    N, K = q.size(0), q.size(1) * 2
    p = q.view(torch.uint8).reshape(N // 32, K // 32, 8, 4, 2, 2, 4)
    both = torch.stack([p & 15, p >> 4], 1)                                  # n32 a k32 c e d b f
    return both.permute(0, 1, 6, 3, 2, 5, 4, 7).reshape(N, K)                # n32 a b c | k32 d e f


def _linear64(x, w, group):
    """x [T, K] -> its product with a quantised projection: x quantised per token to int8 with a 16-bit scale and row sum, weights as
    stored."""
    amax = x.abs().amax(-1, keepdim=True)
    xq, scale = torch.round(x * (127.0 / amax)), (amax / 127.0).half().double()
    q = _nibbles(w["qweight"])
    if group == -1:
        y = _chunked(xq, q) * w["s1_scales"].double() * scale
        return y - w["s1_szeros"].double() * x.sum(-1, keepdim=True).half().double()
    k, n = q.size(1), q.size(0)

    def per_channel(m):                                                      # stored in the order (c, j) of channel 8 j + c in every 32
        return m.reshape(k // 128, n // 32, 8, 4).transpose(2, 3).reshape(k // 128, n).t().repeat_interleave(128, 1)

    w8 = (q.int() * per_channel(w["s2_scales"]).int() + per_channel(w["s2_zeros"]).int()).to(torch.int8)
    return _chunked(xq, w8) * w["s1_scales"].double() * scale


def _chunked(x, w):
    """x @ w^T in 64 bits, the weights widened piece by piece."""
    return torch.cat([x @ p.double().t() for p in w.split(4096)], -1)


def _rms64(x, w, eps, centred):
    u = x - x.mean(-1, keepdim=True) if centred else x
    return u / torch.sqrt((u * u).mean(-1, keepdim=True) + eps) * w.double()


def _rope64(x, pos, base):
    """x [T, heads, 128]: dimensions i and i + 64 turn by pos * base^(-i / 64)."""
    a = pos.double()[:, None, None] * base ** (-torch.arange(64, dtype=F64, device=x.device) / 64.0)
    u, v = x[..., :64], x[..., 64:]
    return torch.cat([u * torch.cos(a) - v * torch.sin(a), v * torch.cos(a) + u * torch.sin(a)], -1)


def _cache64(x, bits):
    """What the cache gives back for x [T, heads, 128]: per token and head a 16-bit scale and zero point and `bits`-bit values."""
    levels, hi, lo = 2.0 ** bits - 1.0, x.amax(-1, keepdim=True), x.amin(-1, keepdim=True)
    scale, zero = ((hi - lo) / levels).half().double(), (-levels * lo / (hi - lo)).half().double()
    return scale * (torch.round(x / scale + zero).clamp(0.0, levels) - zero)


def _attend64(q, k, v, scale, mask=None):
    """q [T, H, d], k [n, G, d], v [n, G, dv]; mask [T, n] of the visible keys (None: all)."""
    T, H, _ = q.shape
    G = k.size(1)
    out = []
    for h in range(H):
        s = q[:, h] @ k[:, h // (H // G)].t() * scale
        if mask is not None:
            s = s.masked_fill(~mask, -math.inf)
        out.append(torch.softmax(s, -1) @ v[:, h // (H // G)])
    return torch.stack(out, 1)


def _llama64(case, W, h, attend):
    """The stack: h [T, D] -> h behind the last layer; attend(layer, q, k, v) is the attention over un-rotated heads."""
    c, group = _shape(case), case["group"]
    H, G = c["heads"], c["kv_heads"]
    for li, L in enumerate(W["layers"]):
        qkv = _linear64(_rms64(h, L["ln1"], c["eps"], True), L["qkv"], group)
        q, k, v = qkv.view(h.size(0), -1, 128).split([H, G, G], 1)
        h = h + _linear64(attend(li, q, k, v).reshape(h.size(0), -1), L["o"], group)
        a, b = _linear64(_rms64(h, L["ln2"], c["eps"], True), L["gate_up"], group).chunk(2, -1)
        h = h + _linear64(a * torch.sigmoid(a) * b, L["down"], group)
    return h


def _exact_llama_step(case, seed):
    c, bits = _shape(case), case["kv_bits"]
    W = _llama_weights(case, seed, False)
    lens, hidden, past = _llama_step_inputs(case, seed)
    H, G, base = c["heads"], c["kv_heads"], c["rope_theta"]

    def attend(li, q, k, v):
        rows, at, out = next(past).view(-1, H + 2 * G, 128), 0, []
        for b, n in enumerate(lens):
            old, pos = rows[at:at + n - 1].double(), torch.arange(n, device=DEV)
            at += n - 1
            keys = torch.cat([_cache64(_rope64(old[:, H:H + G], pos[:-1], base), bits), _rope64(k[b:b + 1], pos[-1:], base)])
            values = torch.cat([_cache64(old[:, H + G:], bits), v[b:b + 1]])
            qb, out_b = _rope64(q[b:b + 1], pos[-1:], base)[0].view(G, H // G, 128), []
            s = torch.softmax(torch.matmul(qb, keys.permute(1, 2, 0).contiguous()) / math.sqrt(128.0), -1)
            out_b = torch.matmul(s, values.transpose(0, 1).contiguous())
            out.append(out_b.reshape(1, H, 128))
        return torch.cat(out)

    h = _llama64(case, W, hidden.double(), attend)
    return {"final": _rms64(h, W["norm"], c["eps"], False), "hidden": h, "cache": [None] * (2 * c["layers"])}


def _exact_llama_prompt(case, seed):
    c, B, L = _shape(case), case["batch"], case["tokens"]
    W = _llama_weights(case, seed, True)
    tokens, pos = _llama_prompt_tokens(case, seed), torch.arange(L, device=DEV)
    mask = pos[None, :] <= pos[:, None]

    def attend(li, q, k, v):
        out = []
        for b in range(B):
            r = slice(b * L, (b + 1) * L)
            out.append(_attend64(_rope64(q[r], pos, c["rope_theta"]), _rope64(k[r], pos, c["rope_theta"]), v[r], 1.0 / math.sqrt(128.0), mask))
        return torch.cat(out)

    h = _llama64(case, W, W["embed"][tokens].double(), attend)[L - 1::L]
    return {"final": _rms64(h, W["norm"], c["eps"], False), "hidden": h, "cache": [None] * (2 * c["layers"])}


def _llama_work(case):
    c = _shape(case)
    D, I, H, G, n = c["hidden"], c["inter"], c["heads"], c["kv_heads"], c["layers"]
    params = (H + 2 * G) * 128 * D + D * H * 128 + 3 * D * I
    weights = n * (params / 2 + (2 * params / 128 if case["group"] != -1 else 0) + 8 * D)
    row = G * 2 * (128 * case["kv_bits"] / 8 + 4)                            # cache bytes per token and layer
    if case["kind"] == "llama_step":
        lens = _lengths(case["batch"], case["context"], case["spread"])
        T, keys = case["batch"], sum(lens)
        return {"bytes": weights + n * keys * row + 6.0 * T * D, "flops": n * (2.0 * T * params + 4.0 * keys * H * 128)}
    B, L = case["batch"], case["tokens"]
    head = c["vocab"] * D
    return {"bytes": weights + n * B * L * row + 2.0 * B * L * D + 2.0 * head + 2.0 * B * c["vocab"],
            "flops": n * (2.0 * B * L * params + 4.0 * B * L * (L + 1) / 2 * H * 128) + 2.0 * B * head}


# ---- the served models -------------------------------------------------------------------------------------------------------

def _design(case, seed):
    """-> (configuration, checkpoint tensors) at the benchmark's sizes."""
    s, d = designs.SIZES[case["size"]], case["design"]
    m = designs.MUMELIX[case["size"]]
    if d == "Vekalorn":
        cfg = designs.vekalorn_config(s)
        W = designs.random_weights(cfg, DEV, seed)
        for n in W:
            if n.endswith(".norm2"):
                W[n] = W[n] * 0.15                                           # (gains as training leaves them: the experts add to the stream)
        return cfg, W
    if d == "Mumelix":
        cfg = designs.mumelix_config(s, m)
        return cfg, designs.mumelix_weights(cfg, m, DEV, seed)
    cfg = designs.rivolix_config(s, m)
    W = designs.rivolix_weights(cfg, DEV, seed)
    for n in W:
        if n.endswith((".ls1", ".ls2")):
            W[n] = W[n] * (0.4 if n.endswith(".ls1") else 0.08)              # (layer scales as training leaves them: well below one)
    return cfg, W


def _serve_tokens(case, seed):
    """-> per sequence the prompt and the tokens of the later steps (a replayed generation)."""
    g = torch.Generator().manual_seed(7919 * seed + 5)
    return [(torch.randint(0, designs.VOCAB, (n,), generator=g).tolist(), torch.randint(0, designs.VOCAB, (case.get("steps", 0),), generator=g).tolist())
            for n in _lengths(case["seqs"], case["tokens"], case["spread"])]


def _prepare_serve(case, seed):
    cfg, W = _design(case, seed)
    seqs = _serve_tokens(case, seed)
    pages = sum((len(p) + len(t) + 63) // 64 for p, t in seqs)
    eng = Engine(resolve_model(cfg)[0], cfg, W, dtype="bfloat16", device=DEV, max_tokens=64 * pages, max_seqs=len(seqs),
                 decode_graphs=case["kind"] == "serve_decode")
    want, at = [], 0
    for p, _ in seqs:
        at += len(p)
        want += range(at - (min(SCORED, len(p)) if case["kind"] == "serve_prompt" else 1), at)
    return dict(case=case, engine=eng, seqs=seqs, want=want)


def _run_serve(st):
    eng, seqs = st["engine"], st["seqs"]
    slots = [eng.open_sequence() for _ in seqs]
    out = [eng.execute([(s, p) for s, (p, _) in zip(slots, seqs)], st["want"])]
    rows = list(range(len(slots)))
    for i in range(st["case"].get("steps", 0)):
        out.append(eng.execute([(s, t[i:i + 1]) for s, (_, t) in zip(slots, seqs)], rows))
    for s in reversed(slots):
        eng.close_sequence(s)
    return torch.cat(out)


# the same in 64 bits: whole sequences, no cache, no state hand-over

def _mm(x, w):
    return x @ w.double().t()


def _silu(x):
    return x * torch.sigmoid(x)


def _experts64(h, idx, wt, count, unit):
    """sum over a token's experts of wt * unit(e, rows); unit(e, x, w) is given the weight too."""
    y = torch.zeros_like(h)
    for e in range(count):
        t, j = (idx == e).nonzero(as_tuple=True)
        if t.numel():
            y.index_add_(0, t, unit(e, h[t], wt[t, j][:, None]))
    return y


def _pairs(x, c, s, interleaved):
    """Turn the pairs (2 i, 2 i + 1) or (i, i + n / 2) of x [T, heads, n]; c, s [T, n / 2]."""
    c, s = c[:, None], s[:, None]
    u, v = (x[..., 0::2], x[..., 1::2]) if interleaved else x.chunk(2, -1)
    a, b = u * c - v * s, v * c + u * s
    return torch.stack([a, b], -1).flatten(-2) if interleaved else torch.cat([a, b], -1)


def _angles(pos, rot):
    """-> cos, sin [T, dims / 2] of the (scaled) rotary embedding."""
    n, base, sc = int(rot["dims"]), float(rot["base"]), rot.get("scaling")
    f, mag = [base ** (-2.0 * i / n) for i in range(n // 2)], 1.0
    if sc and "fast" in sc:                                                  # interpolation by dimension, with a magnitude
        dim = lambda turns: n * math.log(sc["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))       # noqa: E731
        lo, hi = max(math.floor(dim(sc["fast"])), 0), min(math.ceil(dim(sc["slow"])), n - 1)
        ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(n // 2)]
        f, mag = [x / sc["factor"] * r + x * (1.0 - r) for x, r in zip(f, ramp)], 0.1 * math.log(sc["factor"]) + 1.0
    elif sc:                                                                 # by wavelength
        def scaled(x):
            turns = sc["original"] * x / (2.0 * math.pi)
            r = min(max((turns - sc["low"]) / (sc["high"] - sc["low"]), 0.0), 1.0)
            return (1.0 - r) * x / sc["factor"] + r * x
        f = [scaled(x) for x in f]
    a = pos.double()[:, None] * torch.tensor(f, dtype=F64, device=pos.device)
    return torch.cos(a) * mag, torch.sin(a) * mag


def _causal(T, window=None):
    i = torch.arange(T, device=DEV)
    d = i[:, None] - i[None, :]
    return (d >= 0) & (d < window) if window else d >= 0


def _conv64(x, w):
    """Causal convolution over time of x [T, C] with taps w [C, n], the last tap on the token itself."""
    n = w.size(1)
    p = torch.cat([x.new_zeros(n - 1, x.size(1)), x])
    return sum(p[j:j + x.size(0)] * w[:, j].double() for j in range(n))


def _layer_norm64(x, w, eps):
    return _rms64(x, w, eps, True)


def _vekalorn64(cfg, W, runs, x):
    eps = cfg["norm"]["eps"]
    x = W["embed"][x].double()
    for i, L in enumerate(cfg["layers"]):
        p, m, r = f"l{i}.mix.", L["mixer"], L["mlp"]["router"]
        H, d, dv, rank = m["heads"], m["dim"], m["vdim"], m["kv_rank"]
        q = _mm(_rms64(_mm(x, W[p + "dq"]), W[p + "dq.norm"], eps, False), W[p + "uq"]).view(x.size(0), H, -1)
        down = _mm(x, W[p + "dkv"])
        c = _rms64(down[:, :rank], W[p + "dkv.norm"], eps, False)
        k, v = _mm(c, W[p + "uk"]).view(-1, H, d), _mm(c, W[p + "uv"]).view(-1, H, dv)
        o = []
        for a, n in runs:
            qs, ks = q[a:a + n], k[a:a + n]
            if "rot" in m:
                cs, sn = _angles(torch.arange(n, device=DEV), m["rot"])
                kr = _pairs(down[a:a + n, None, rank:], cs, sn, True).expand(n, H, -1)
                qs, ks = torch.cat([qs[..., :d], _pairs(qs[..., d:], cs, sn, True)], -1), torch.cat([ks, kr], -1)
            o.append(_attend64(qs, ks, v[a:a + n], m["scale"], _causal(n, (m.get("mask") or {}).get("size"))))
        o = torch.cat(o).flatten(1)
        if p + "g" in W:
            o = o * torch.sigmoid(_mm(x, W[p + "g"]))
        x = x + _layer_norm64(_mm(o, W[p + "o"]), W[f"l{i}.norm1"], eps)
        q = f"l{i}.mlp."
        s = torch.softmax(_mm(x, W[q + "router"]), -1)
        groups = s.view(x.size(0), r["groups"]["count"], -1)
        best = groups.amax(-1).topk(r["groups"]["keep"], -1).indices
        open_ = torch.zeros(groups.shape[:2], dtype=torch.bool, device=DEV).scatter_(1, best, True)
        idx = groups.masked_fill(~open_[..., None], -1.0).flatten(1).topk(r["top"], -1).indices
        y = _experts64(x, idx, s.gather(1, idx), r["experts"],
                       lambda e, h, w: w * _mm(torch.relu(_mm(h, W[f"{q}e{e}.up"])) ** 2, W[f"{q}e{e}.down"]))
        x = x + _layer_norm64(y, W[f"l{i}.norm2"], eps)
    return lambda rows: _mm(_layer_norm64(x[rows], W["final.norm"], eps), W["head"])


def _recurrence64(q, k, v, decay, beta, runs):
    """q, k, decay [T, H, d], v [T, H, dv], beta [T, H] (delta rule) or None; every sequence from a zero state, side by side."""
    o, n = torch.zeros_like(v), max(r[1] for r in runs)
    first = torch.tensor([a for a, _ in runs], device=DEV)
    count = torch.tensor([c for _, c in runs], device=DEV)
    S = v.new_zeros(len(runs), v.size(1), q.size(2), v.size(2))
    for t in range(n):
        live = count > t
        at = first[live] + t
        s = decay[at][..., None] * S[live]
        u = v[at]
        if beta is not None:
            u = beta[at][..., None] * (u - (k[at][..., None] * s).sum(-2))
        s = s + k[at][..., None] * u[..., None, :]
        o[at] = (q[at][..., None] * s).sum(-2)
        S[live] = s
    return o


def _mumelix64(cfg, W, runs, x):
    eps, S = cfg["norm"]["eps"], cfg["streams"]
    dyt = lambda u, n: torch.tanh(float(W[n + ".alpha"]) * u) * W[n].double() + W[n + ".b"].double()       # noqa: E731
    x = W["embed"][x].double() * cfg["embedding"]["scale"]
    T, starts = x.size(0), torch.tensor([a for a, _ in runs], device=DEV)
    pos = torch.cat([torch.arange(n, device=DEV) for _, n in runs])
    xs = x[:, None].expand(T, S, -1).clone()

    def read(p, n):
        return dyt((xs * W[p + "in"].double()[None, :, None]).sum(1), n)

    def write(p, y):
        mixed = torch.matmul(W[p + "mix"].double().t().contiguous(), xs)
        return mixed + W[p + "out"].double()[None, :, None] * y[:, None]

    def convolved(h, n):
        return torch.cat([_silu(_conv64(h[a:a + c], W[n])) for a, c in runs])

    for i, L in enumerate(cfg["layers"]):
        p, m = f"l{i}.mix.", L["mixer"]
        h = read(f"l{i}.hc1.", f"l{i}.norm1")
        before = h.roll(1, 0).index_fill(0, starts, 0.0)
        h = h + (before - h) * W[f"l{i}.shift"].double()
        if L["type"] == "gla":
            H, d, dv = m["heads"], m["dim"], m["vdim"]
            q, k, v = (_mm(h, W[p + n]).view(T, H, -1) for n in "qkv")
            z = _mm(_mm(h, W[p + "a1"]), W[p + "a2"]) + W[p + "a2.b"].double()
            o = _recurrence64(q * d ** -0.5, k, v, (torch.sigmoid(z) ** (1.0 / m["tau"])).view(T, H, d), None, runs)
            y = _mm(_rms64(o, W[p + "norm"], eps, False).flatten(1) * _silu(_mm(h, W[p + "g"])), W[p + "o"])
        else:
            a, b, q = m["left"], m["right"], p + "left."
            H, G, n, dv = a["heads"], a["kv_heads"], a["rot"]["dims"], a["vdim"]
            qh, kh, vh = (_mm(h, W[q + s]).view(T, -1, a["vdim"] if s == "v" else a["dim"]) for s in "qkv")
            ck, cv = _angles(pos, a["rot"]), _angles(pos, {"dims": dv, "base": a["rot"]["base"]})
            qh, kh = (torch.cat([_pairs(u[..., :n], *ck, False), u[..., n:]], -1) for u in (qh, kh))
            vh = _pairs(vh, *cv, False)
            o = torch.cat([_attend64(qh[s:s + c], kh[s:s + c], vh[s:s + c], a["scale"], _causal(c)) for s, c in runs])
            left = _mm(_pairs(o, cv[0], -cv[1], False).flatten(1), W[q + "o"])
            q = p + "right."
            H, G, d, dv = b["heads"], b["kv_heads"], b["dim"], b["vdim"]
            qh, kh, vh = (convolved(_mm(h, W[q + s]), q + s + ".conv").view(T, -1, dv if s == "v" else d) for s in "qkv")
            qh, kh = ((u / torch.sqrt((u * u).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 1) for u in (qh, kh))
            dt = torch.nn.functional.softplus(_mm(_mm(h, W[q + "a1"]), W[q + "a2"]) + W[q + "dt_bias"].double()).view(T, H, d)
            decay = torch.exp(-torch.exp(W[q + "A_log"].double())[:, None] * dt)
            o = _recurrence64(qh * d ** -0.5, kh, vh, decay, torch.sigmoid(_mm(h, W[q + "b"])), runs)
            gate = torch.sigmoid(_mm(_mm(h, W[q + "g1"]), W[q + "g2"])).view(T, H, dv)
            right = _mm((_rms64(o, W[q + "norm"], eps, False) * gate).flatten(1), W[q + "o"])
            y = 0.5 * (_rms64(left, W[p + "left.out"], eps, False) + _rms64(right, W[q + "out"], eps, False))
        xs = write(f"l{i}.hc1.", y)
        h, q, r = read(f"l{i}.hc2.", f"l{i}.norm2"), f"l{i}.mlp.", L["mlp"]["router"]
        z, idx = (_mm(h, W[q + "router"]) + W[q + "router.b"].double()).topk(r["top"], -1)
        y = _experts64(h, idx, torch.softmax(z, -1), r["experts"],
                       lambda e, u, w: w * _mm(_silu(_mm(u, W[f"{q}e{e}.gate"])) * _mm(u, W[f"{q}e{e}.up"]), W[f"{q}e{e}.down"]))
        xs = write(f"l{i}.hc2.", y)
    return lambda rows: _mm(dyt(xs[rows].sum(1), "final.norm"), W["head"])


def _rivolix64(cfg, W, runs, x):
    eps = cfg["norm"]["eps"]
    norm = lambda u, w=None: u / torch.sqrt((u * u).mean(-1, keepdim=True) + eps) * (1.0 if w is None else 1.0 + W[w].double())      # noqa: E731
    unit = lambda h, p: _mm(_silu(_mm(h, W[p + "gate"])) * _mm(h, W[p + "up"]), W[p + "down"])                                       # noqa: E731
    x, T, held = W["embed"][x].double(), x.numel(), {}
    pos = torch.cat([torch.arange(n, device=DEV) for _, n in runs])

    def convolved(h, n):
        return torch.cat([_conv64(h[a:a + c], W[n]) for a, c in runs])

    def attend(q, k, v, scale):
        return torch.cat([_attend64(q[a:a + c], k[a:a + c], v[a:a + c], scale, _causal(c)) for a, c in runs])

    for i, L in enumerate(cfg["layers"]):
        p, m = f"l{i}.mix.", L["mixer"]
        H, G, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        h = norm(x, f"l{i}.norm1")
        if L["type"] == "attention":
            if m.get("kv_from") is None:
                held[i] = (convolved(_mm(h, W[p + "k"]), p + "k.conv").view(T, G, 2, d), convolved(_mm(h, W[p + "v"]), p + "v.conv").view(T, G, dv))
            k, v = held[i if m.get("kv_from") is None else m["kv_from"]]
            warm = 1.0 + m["q_temp"]["coef"] * torch.log(torch.floor((pos.double() + 1.0) / m["q_temp"]["every"]) + 1.0)
            q = convolved(_mm(h, W[p + "q"]), p + "q.conv").view(T, H, 2, d) * warm[:, None, None, None]
            l1, l2 = (math.exp(float((W[p + "lq" + s].double() * W[p + "lk" + s].double()).sum())) for s in "12")
            one, two = (attend(q[:, :, j], k[:, :, j], v, m["scale"]) for j in (0, 1))
            o = norm(one - (l1 - l2 + m["diff"]) * two) * (1.0 - m["diff"])
            y = _mm(o.flatten(1) * torch.sigmoid(_mm(h, W[p + "g"])), W[p + "o"])
        else:
            cs = _angles(pos, m["rot"])
            q, k = _mm(h, W[p + "q"]).view(T, H, d), _mm(h, W[p + "k"]).view(T, G, d)
            y = _mm(attend(norm(_pairs(q, *cs, False)), norm(_pairs(k, *cs, False)), k, m["scale"]).flatten(1), W[p + "o"])
        g, q, r = norm(x, f"l{i}.norm2"), f"l{i}.mlp.", L["mlp"]["router"]
        s, idx = torch.sigmoid(_mm(g, W[q + "router"])).topk(r["top"], -1)
        ff = _experts64(g, idx, s, r["experts"], lambda e, u, w: unit(w * u, f"{q}e{e}.")) + unit(g, q + "shared.")
        x = x + (y * W[f"l{i}.ls1"].double() + ff * W[f"l{i}.ls2"].double())
    return lambda rows: _mm(norm(x[rows], "final.norm"), W["embed"])


def _exact_serve(case, seed):
    cfg, W = _design(case, seed)
    seqs, runs, at = _serve_tokens(case, seed), [], 0
    for p, t in seqs:
        runs.append((at, len(p) + len(t)))
        at += len(p) + len(t)
    tokens = torch.tensor([v for p, t in seqs for v in p + t], device=DEV)
    forward = {"Vekalorn": _vekalorn64, "Mumelix": _mumelix64, "Rivolix": _rivolix64}[case["design"]]
    logits = forward(cfg, W, runs, tokens)
    ends = [a + len(p) for (a, _), (p, _) in zip(runs, seqs)]
    keep = [min(SCORED, len(p)) if case["kind"] == "serve_prompt" else 1 for p, _ in seqs]
    out = [logits(torch.tensor([j for e, k in zip(ends, keep) for j in range(e - k, e)], device=DEV))]
    for i in range(case.get("steps", 0)):
        out.append(logits(torch.tensor([e + i for e in ends], device=DEV)))
    return torch.cat(out)


def _serve_work(case):
    s, m, d = designs.SIZES[case["size"]], designs.MUMELIX[case["size"]], case["design"]
    D, E, top, V, ff = s["width"], s["experts"], s["top"], designs.VOCAB, s["ff"]
    expert = (2 if d == "Vekalorn" else 3) * ff * D
    aw = m["a_heads"] * m["a_dim"]
    kv = m["a_kv"] * (m["a_dim"] + m["a_vdim"])
    if d == "Vekalorn":                                                      # a layer's mixer weights, its cached row, work per visible pair
        mixer = s["q_rank"] * (D + s["heads"] * (s["dim"] + s["rot_dim"] / 2)) + s["kv_rank"] * (D + 2 * s["heads"] * s["dim"]) + 1.5 * D * s["heads"] * s["vdim"]
        row, pair, state = s["kv_rank"] + s["rot_dim"] / 2, 2.0 * s["heads"] * (s["dim"] + s["rot_dim"] / 2 + s["vdim"]), 0
    elif d == "Mumelix":                                                     # half the layers have attention, all a recurrence
        gla = D * m["g_heads"] * (2 * m["g_dim"] + 3 * m["g_vdim"])
        delta = D * (2 * m["d_kv"] * m["d_dim"] + 2 * m["d_heads"] * m["d_vdim"])
        mixer = (gla + delta + D * (2 * aw + kv)) / 2
        row, pair, state = kv / 2, aw * 2.0, m["g_heads"] * m["g_dim"] * m["g_vdim"]
    else:
        mixer, row, pair, state = D * (3 * aw + kv), kv * 0.75, 2.5 * m["a_heads"] * 2 * m["a_dim"], 0
    shared, layers = expert if d == "Rivolix" else 0, LAYERS[case["kind"]]
    per_token = mixer + top * expert + shared

    def step(T, keys_read, pairs, rows, seqs):
        experts = E * (1.0 - (1.0 - top / E) ** T)
        return (layers * (2.0 * (mixer + shared + experts * expert) + 2.0 * row * (keys_read + T) + 8.0 * state * seqs) + 2.0 * V * D
                + 2.0 * T * D + 4.0 * rows * V,
                layers * (2.0 * T * per_token + pairs * pair + 7.0 * state * T) + 2.0 * rows * V * D)

    lens = _lengths(case["seqs"], case["tokens"], case["spread"])
    n = len(lens)
    rows = sum(min(SCORED, k) for k in lens) if case["kind"] == "serve_prompt" else n
    parts = [step(sum(lens), 0, sum(k * (k + 1) / 2.0 for k in lens), rows, n)]
    parts += [step(n, sum(lens) + n * i, sum(lens) + n * (i + 1), n, n) for i in range(case.get("steps", 0))]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


# ---- the contract ------------------------------------------------------------------------------------------------------------

def prepare(case, seed):
    return {"llama_step": _prepare_llama_step, "llama_prompt": _prepare_llama_prompt, "serve_prompt": _prepare_serve,
            "serve_decode": _prepare_serve}[case["kind"]](case, seed)


@torch.no_grad()
def run(state):
    return {"llama_step": _run_llama_step, "llama_prompt": _run_llama_prompt, "serve_prompt": _run_serve,
            "serve_decode": _run_serve}[state["case"]["kind"]](state)


def work(case):
    return _llama_work(case) if case["kind"].startswith("llama") else _serve_work(case)


def tolerance(case):
    """Measured against `exact` and against the same path with another order of the attention's sums or other expert products.  A
    quantised stack: activations and cache values that round to the other integer.  A served model: bfloat16 between its operations,
    and tokens whose last chosen expert is a near tie ("max": one of those)."""
    if case["kind"].startswith("llama"):
        return {"rel": 0.03, "max": 0.3, "differ": 0.01}
    return {"rel": 0.03, "max": 0.95}


@torch.no_grad()
def exact(case, seed):
    return {"llama_step": _exact_llama_step, "llama_prompt": _exact_llama_prompt, "serve_prompt": _exact_serve,
            "serve_decode": _exact_serve}[case["kind"]](case, seed)
