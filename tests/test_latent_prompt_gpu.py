"""Latent attention of prompts over written-out keys and values: tile edges, later portions, windows, neighbours that hold no numbers, against float64."""
import math

import pytest
import torch

from qserve_amd.layers.ops import make_ops
from qserve_amd.serving.engine import StepBatch

pytestmark = pytest.mark.gpu


# runs: (context, new tokens)
@pytest.mark.parametrize("H, rank, rot_dim, rot_n", [(16, 512, 64, 64), (3, 256, 64, 22), (8, 128, 0, 0)])
@pytest.mark.parametrize("runs, window, gated", [(((65, 65), (1, 1), (128, 128), (129, 129)), None, False), (((191, 191), (64, 64), (63, 63), (8, 7)), None, True),
                                                 (((200, 130), (385, 128), (70, 1)), None, True), (((300, 300), (257, 129)), 37, False),
                                                 (((700, 257), (64, 64)), 64, True), (((333, 333),), 300, False)])
def test_prompt(H, rank, rot_dim, rot_n, runs, window, gated):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    dev = torch.device("cuda:0")
    ops = make_ops("hip", torch.bfloat16, dev)
    g = torch.Generator().manual_seed(rank + H + len(runs))
    R, pages, scale = rank + rot_dim, sum((c + 63) // 64 for c, _ in runs), 1.0 / math.sqrt(128 + rot_dim)
    order = torch.randperm(pages + 1, generator=g).tolist()
    table = torch.full((len(runs), pages), order.pop(), dtype=torch.int32)           # (unused entries: a page of nothing)
    pool = torch.full(((pages + 1) * 64, R), float("nan"))                           # rows that nobody wrote must not reach a result
    keys, items, starts, pos, at = [], [], [], [], 0
    for b, (ctx, n) in enumerate(runs):
        rows = torch.randn(ctx, R, generator=g).bfloat16()
        if b == 1:
            rows[...] = float("nan")                                                 # a neighbour without numbers stays by itself
        for i in range((ctx + 63) // 64):
            table[b, i] = order.pop()
            part = rows[64 * i:64 * i + 64]
            pool[table[b, i] * 64:table[b, i] * 64 + part.size(0)] = part.float()
        keys.append(rows.double())
        items.append((b, at, n))
        starts.append(ctx - n)
        pos += range(ctx - n, ctx)
        at += n
    # every key and value is an element of its latent row times a power of two, so that the products with these weights are exact
    pick = lambda: torch.stack([torch.zeros(128, rank).scatter_(1, torch.randint(0, rank, (128, 1), generator=g),       # noqa: E731
                                                               2.0 ** torch.randint(-1, 2, (128, 1), generator=g)) for _ in range(H)])
    uk, uv = pick(), pick()
    q = (torch.randn(at, H, 128 + rot_dim, generator=g) * 1.5).bfloat16()
    gate = torch.randn(at, 5 + H * 128, generator=g).bfloat16()[:, 5:] if gated else None      # (a column slice off the alignment)
    angle = torch.rand(max(pos) + 1, max(rot_n // 2, 1), generator=g) * 6.0
    rope = torch.stack([torch.cos(angle), torch.sin(angle)], 1).contiguous() if rot_n else None
    batch = StepBatch(tokens=None, seq=None, pos=torch.tensor(pos, dtype=torch.int32, device=dev), slot=None, block_table=table.to(dev), max_pos=max(pos),
                      n_tokens=at, items=items, starts=starts)
    plan = batch.key_runs(window, ops.L.qsv_latent_prompt_tile_tokens())
    to = lambda t: None if t is None else t.to(dev)                                  # noqa: E731
    out = ops.latent_prompt(to(q.view(at, -1)), to(pool.bfloat16()), batch, plan, to(uk.view(-1, rank).bfloat16()), to(uv.view(-1, rank).bfloat16()), to(rope), scale,
                            H, rot_dim, rot_n, rank, 64, window, to(gate))
    out = out.view(at, H, 128).double().cpu()
    qr = q.double()
    if rot_n:
        c, s = (rope[pos, i].double()[:, None] for i in (0, 1))
        u, v = qr[..., 128:128 + rot_n:2].clone(), qr[..., 129:128 + rot_n:2].clone()
        qr[..., 128:128 + rot_n:2], qr[..., 129:128 + rot_n:2] = (u * c - v * s).bfloat16().double(), (v * c + u * s).bfloat16().double()
    for b, first, n in items:
        if b == 1:
            continue
        rows, p = keys[b], torch.tensor(pos[first:first + n])
        j = torch.arange(rows.size(0))
        seen = (j[None] <= p[:, None]) & (j[None] > p[:, None] - (window or 1 << 30))
        for h in range(H):
            k = torch.cat([rows[:, :rank] @ uk[h].double().t(), rows[:, rank:]], 1)
            v = rows[:, :rank] @ uv[h].double().t()
            w = torch.softmax((qr[first:first + n, h] @ k.t() * scale).masked_fill(~seen, -math.inf), 1)
            ref, spread = w @ v, ((w * w) @ (v * v)).sqrt()
            if gated:
                f = torch.sigmoid(gate[first:first + n, 128 * h:128 * h + 128].double())
                ref, spread = ref * f, spread * f
            # weights enter the second product as bfloat16 (relative 2^-9 each, independent), so may a rotated query that lies on a tie; the result is
            # stored as bfloat16
            bound = 2.0 ** -8 * ref.abs() + 6 * 2.0 ** -9 * spread + 1e-5
            err = (out[first:first + n, h] - ref).abs()
            assert (err <= bound).all(), (b, h, (err / bound).max())
    assert torch.isfinite(out[[i for b, f, n in items if b != 1 for i in range(f, f + n)]]).all()


@pytest.mark.parametrize("tokens, starts, taken", [((65,), (0,), True), ((64,), (0,), False), ((128, 1), (0, 40), True), ((128, 1), (0, 4000), False),
                                                   ((1,) * 80, (0,) * 80, False), ((512,), (1536,), True), ((512,), (1544,), False)])
def test_where_it_is_taken(tokens, starts, taken):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    dev = torch.device("cuda:0")
    ops, at, items = make_ops("hip", torch.bfloat16, dev), 0, []
    for b, n in enumerate(tokens):
        items.append((b, at, n))
        at += n
    single = torch.zeros((at, 3), dtype=torch.int32, device=dev) if at == len(tokens) else None
    batch = StepBatch(tokens=None, seq=None, pos=torch.zeros(at, dtype=torch.int32, device=dev), slot=None, block_table=None, max_pos=0, n_tokens=at, items=items,
                      starts=list(starts), _single=single)
    plan = lambda **k: ops.latent_prompt_plan(batch, None, *(k.get(n, d) for n, d in (("H", 16), ("dim", 128), ("rot", 64), ("vdim", 128), ("rank", 512), ("scale", 0.1))))   # noqa: E731
    assert (plan() is not None) == taken
    assert plan(dim=64) is None and plan(vdim=64) is None and plan(rot=32) is None and plan(rank=100) is None and plan(scale=-0.1) is None
    batch.starts = None
    batch._tiles.clear()
    assert plan() is None


class _Turned:
    dims = 64

    def reserve(self, n):
        a = torch.arange(n)[:, None] * 10.0 ** (-torch.arange(32) / 8.0)
        return torch.stack([torch.cos(a), torch.sin(a)], 1).cuda()


def _layer(H=4, D=256, qr=64, rank=64, rot_dim=64, gated=False, window=None, page=64):
    from qserve_amd.layers.latent_attention import LatentAttention
    g = torch.Generator().manual_seed(H + rank)
    mat = lambda o, i: (torch.randn(o, i, generator=g) / i ** 0.5).bfloat16().cuda()               # noqa: E731
    one = lambda n: torch.ones(n, dtype=torch.bfloat16, device="cuda")                             # noqa: E731
    w = dict(dq=mat(qr, D), dq_norm=one(qr), uq=mat(H * (128 + rot_dim), qr), dkv=mat(rank + rot_dim, D), dkv_norm=one(rank), uk=mat(H * 128, rank),
             uv=mat(H * 128, rank), o=mat(D, H * 128))
    if gated:
        w["g"] = mat(H * 128, D)
    return LatentAttention(make_ops("hip", torch.bfloat16, torch.device("cuda:0")), heads=H, dim=128, vdim=128, kv_rank=rank, q_rank=qr, scale=0.1, eps=1e-5, weights=w,
                           rot_dim=rot_dim, rotary=_Turned() if rot_dim else None, gated=gated, window=window, page=page)


def _step(layer, h, runs, pool, table):
    """The layer over runs (sequence, first position, tokens) of one step."""
    dev, at, items, starts, pos, seq = h.device, 0, [], [], [], []
    for b, start, n in runs:
        items.append((b, at, n))
        starts.append(start)
        pos += range(start, start + n)
        seq += [b] * n
        at += n
    p, s = torch.tensor(pos), torch.tensor(seq)
    slot = table.cpu()[s, p // layer.page].long() * layer.page + p % layer.page
    batch = StepBatch(tokens=None, seq=s.int().to(dev), pos=p.int().to(dev), slot=slot.to(dev), block_table=table, max_pos=max(pos), n_tokens=at, items=items, starts=starts)
    return layer(h, batch, pool)


def test_a_pool_off_16_bytes_is_taken():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    layer, g = _layer(page=40), torch.Generator().manual_seed(5)       # (pages that the kernels reading elements one by one serve)
    h, table = torch.randn(150, 256, generator=g).bfloat16().cuda(), torch.tensor([[2, 0, 3, 1]], dtype=torch.int32, device="cuda")
    outs = []
    for off, rule in ((0, False), (1, True), (4, True)):                # (the rule off: on the rows, aligned)
        pool = torch.zeros(160 * 128 + 8, dtype=torch.bfloat16, device="cuda")[off:][:160 * 128].view(160, 128)
        layer.ops.prompt_heads_kernel = rule
        outs.append(_step(layer, h, [(0, 0, 150)], pool, table))
    # the latents' norms sum their squares in another order where the pool is off four elements, so that a latent may round the other way: 2^-9 of some of them
    a = outs[0].double()
    for o in outs[1:]:
        assert (o.double() - a).norm() <= 2.0 ** -9 * a.norm()


def _wide(layer, h, window):
    """The layer over one sequence in float64, all of its tokens at once."""
    H, n, d = layer.H, h.size(0), lambda t: t.double()
    down = d(h) @ d(layer.w_down).t()
    norm = lambda t, w: t / (t.pow(2).mean(-1, keepdim=True) + layer.eps).sqrt() * d(w)            # noqa: E731
    q = (norm(down[:, :layer.q_rank], layer.dq_norm) @ d(layer.w_uq).t()).view(n, H, 128 + layer.rot_dim)
    kv = down[:, layer.kv_off:layer.kv_off + layer.row_width]
    c, kr = norm(kv[:, :layer.rank], layer.dkv_norm), kv[:, layer.rank:]

    def turned(u):
        if not layer.rot_dim:
            return u
        cos, sin = (layer.rotary.reserve(n)[:, i].double().view(n, *[1] * (u.dim() - 2), -1) for i in (0, 1))
        a, b = u[..., 0::2], u[..., 1::2]
        return torch.stack([a * cos - b * sin, b * cos + a * sin], -1).flatten(-2)
    qr, kr = turned(q[..., 128:]), turned(kr)
    i = torch.arange(n, device=h.device)
    seen = (i[None] <= i[:, None]) & (i[None] > i[:, None] - (window or n))
    outs = []
    for j in range(H):
        s = q[:, j, :128] @ (c @ d(layer.w_uk[j]).t()).t() + qr[:, j] @ kr.t()
        outs.append(torch.softmax((s * layer.scale).masked_fill(~seen, -math.inf), 1) @ (c @ d(layer.w_uv[128 * j:128 * j + 128]).t()))
    o = torch.cat(outs, 1)
    return (o * torch.sigmoid(down[:, layer.g_off:]) if layer.gated else o) @ d(layer.w_o).t()


# two sequences in portions (sequence, first position, tokens), step after step: up to 64 tokens and behind more than three times as many keys on the rows, between
# them over written-out heads, both kinds of run in one step, one head too few
@pytest.mark.parametrize("H, rank, rot_dim, gated, window", [(4, 64, 64, False, None), (3, 512, 64, True, None), (5, 128, 0, True, 96), (2, 64, 64, False, None)])
def test_portions_on_both_sides_of_the_line(H, rank, rot_dim, gated, window):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    layer, g = _layer(H=H, rank=rank, rot_dim=rot_dim, gated=gated, window=window), torch.Generator().manual_seed(H)
    steps = [([(0, 0, 200)], True), ([(0, 200, 40)], False), ([(0, 240, 70)], None if window else False), ([(0, 310, 110), (1, 0, 65)], True), ([(0, 420, 1), (1, 65, 1)], False),
             ([(1, 66, 170), (0, 421, 1)], True), ([(0, 422, 129)], None if window else False), ([(0, 551, 300), (1, 236, 3)], True)]
    h = [torch.randn(n, 256, generator=g).bfloat16().cuda() for n in (851, 239)]
    table = torch.randperm(18, generator=g)[:18].int().view(1, -1).cuda()
    table = torch.cat([table[:, :14], torch.cat([table[:, 14:], table[:, :10]], 1)])        # (the second sequence's pages: the last four; the rest is never reached)
    pool = torch.full((18 * 64, rank + rot_dim), float("nan"), dtype=torch.bfloat16, device="cuda")
    plan, taken = layer.ops.latent_prompt_plan, []
    layer.ops.latent_prompt_plan = lambda *a: taken.append(plan(*a)) or taken[-1]
    got = [torch.zeros(t.size(0), 256, dtype=torch.float64, device="cuda") for t in h]
    for runs, heads_form in steps:
        out, at = _step(layer, torch.cat([h[b][s:s + n] for b, s, n in runs]), runs, pool, table), 0
        assert heads_form is None or (taken[-1] is not None) == (heads_form and H > 2)
        for b, s, n in runs:
            got[b][s:s + n] = out[at:at + n].double()
            at += n
    for b in (0, 1):
        ref = _wide(layer, h[b], window)
        # ten roundings to bfloat16 on the way of the values (2^-9 of what they round at most, 0.6 of that in the mean, independent), four on the way of scores of
        # up to 4, which scale their weights: (10 + 4 4^2)^0.5 0.6 2^-9 < 2^-6.5 of a portion's size
        for s, n in [(s, n) for runs, _ in steps for q, s, n in runs if q == b]:
            err = (got[b][s:s + n] - ref[s:s + n]).norm() / ref[s:s + n].norm()
            assert err <= 2.0 ** -6.5, (b, s, n, err)
