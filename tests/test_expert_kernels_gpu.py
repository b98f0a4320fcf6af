"""The expert-major products and the one-expert-per-lane router at the edges of their tiles, against float64."""
import pytest
import torch

from qserve_amd.layers.ops import ExpertRows, linear, make_ops

pytestmark = pytest.mark.gpu


def _silu(x):
    return x * torch.sigmoid(x)


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return make_ops("hip", torch.bfloat16, torch.device("cuda:0"))


def check(o, T, top, E, ident, D, ff, act, weigh, crowd, shift=0, graph=False, none=False):
    """crowd: about that share of the tokens has expert 0 first; shift: the weights start that many elements into their storage; graph: the
    result of a captured call, replayed; none: some slots name no expert."""
    g = torch.Generator().manual_seed(T * 131 + D)
    dev, gated = "cuda:0", act != "relu_sq"
    h = torch.randn(T + 1, D, generator=g).bfloat16()
    up = (torch.randn(E, 2 * ff if gated else ff, D, generator=g) / D ** 0.5).bfloat16()
    down = (torch.randn(E, D, ff, generator=g) / ff ** 0.5).bfloat16()
    idx = torch.rand(T, E + ident, generator=g).argsort(dim=1)[:, :top].int()
    if T > 4:
        idx[: int(T * crowd), 0] = 0
        idx[:, 1:][idx[:, 1:] == 0] = E + ident - 1
    if none:
        idx[torch.rand(T, top, generator=g) < 0.3] = -1
    wt = torch.rand(T, top, generator=g)
    limit = 1.0 if act == "clamped_glu" else 0.0
    hd = h.to(dev)[1:] if T % 2 else h[1:].to(dev)                      # (also a view that starts inside a row of 16 bytes for narrow widths)
    upd, downd = (torch.cat([w.new_zeros(shift), w.flatten()]).to(dev)[shift:].view(w.shape) for w in (up, down))
    args = (hd, upd, downd, idx.to(dev), wt.to(dev))
    call = lambda: o.moe_experts(*args, act=act, limit=limit, weigh=weigh)                                # noqa: E731
    if graph:
        call()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            y = call()
        for _ in range(3):
            y.zero_()
            g.replay()
    else:
        y = call()
    y = y.double().cpu()
    x, ref, size = h[1:].double(), torch.zeros(T, D, dtype=torch.float64), torch.zeros(T, D, dtype=torch.float64)
    for e in range(E + ident):
        t, k = (idx == e).nonzero(as_tuple=True)
        if not len(t):
            continue
        w = wt[t, k].double()[:, None]
        if e >= E:
            v = x[t] * (w if weigh == "output" else 1.0)
        else:
            a = (x[t] @ up[e].double().T) * (w if weigh == "input" else 1.0)
            if act == "relu_sq":
                a = torch.relu(a) ** 2
            elif act == "swiglu":
                a = _silu(a[:, 0::2]) * a[:, 1::2]
            else:
                p, q = a[:, 0::2].clamp(max=limit), a[:, 1::2].clamp(-limit, limit)
                a = p * torch.sigmoid(1.702 * p) * (q + 1.0)
            v = (a @ down[e].double().T) * (w if weigh == "output" else 1.0)
            # the activations are stored in bfloat16 (relative 2^-9 each, independent), in the grouped form the experts' rows too
            size.index_add_(0, t, (a.pow(2) @ down[e].double().pow(2).T) * (w * w if weigh == "output" else 1.0) + v.pow(2))
        ref.index_add_(0, t, v)
    bound = 2.0 ** -8 * ref.abs() + 6 * 2.0 ** -9 * size.sqrt() + 1e-5
    assert ((y - ref).abs() <= bound).all(), ((y - ref).abs() / bound).max()


ACTS = pytest.mark.parametrize("act, weigh", [("relu_sq", "output"), ("swiglu", "input"), ("clamped_glu", "output")])


# tokens, top, experts, identity outputs, width, ff: tiles of 32 weight rows, stages of 64 elements in four waves, chunks of 16 and 32
# slots, windows of 1024 slots
@pytest.mark.parametrize("T, top, E, ident, D, ff", [
    (1, 1, 1, 0, 8, 8), (1, 4, 16, 0, 2048, 1408), (2, 2, 3, 2, 72, 40), (3, 4, 5, 0, 64, 32), (16, 1, 1, 0, 200, 24), (17, 1, 1, 0, 264, 33 * 8),
    (32, 1, 1, 0, 4096, 16), (33, 1, 2, 0, 16, 4096), (70, 2, 4, 1, 520, 136), (64, 4, 16, 0, 2048, 96), (300, 4, 6, 1, 56, 64)])
@ACTS
def test_expert_major_form(ops, T, top, E, ident, D, ff, act, weigh):
    o = make_ops("hip", torch.bfloat16, torch.device("cuda:0"))
    o.moe_expert_major_slots = 10 ** 9
    check(o, T, top, E, ident, D, ff, act, weigh, 0.5)


# tiles of 256 rows x 256, 128 or 64 slots, K steps of 64 in two halves of the buffer; more tiles than workgroups; more experts than lanes
@pytest.mark.parametrize("T, top, E, ident, D, ff, crowd", [
    (1, 1, 1, 0, 64, 64, 0.0), (64, 1, 1, 0, 128, 64, 1.0), (65, 1, 1, 0, 64, 192, 1.0), (128, 1, 1, 0, 320, 128, 1.0), (129, 2, 3, 0, 256, 64, 1.0),
    (256, 1, 2, 0, 64, 320, 1.0), (257, 1, 1, 0, 1088, 64, 1.0), (700, 4, 6, 2, 512, 448, 0.5), (1500, 4, 100, 5, 64, 64, 0.2), (40, 3, 70, 0, 4096, 64, 0.0),
    (2100, 2, 2, 0, 4096, 128, 0.3),
    # whole rounds of workgroups, and tiles left over in halves and quarters
    (3000, 2, 8, 0, 64, 2816, 0.0), (2600, 1, 3, 0, 64, 7168, 0.4), (1024, 1, 1, 0, 128, 18432, 1.0)])
@ACTS
def test_grouped_form(ops, T, top, E, ident, D, ff, crowd, act, weigh):
    o = make_ops("hip", torch.bfloat16, torch.device("cuda:0"))
    o.moe_expert_major_slots, o.moe_sorted_above = 0, 0
    check(o, T, top, E, ident, D, ff, act, weigh, crowd)


# a tile a workgroup at most: one step and runs of steps around the two that are requested ahead; rows in and out of 16; empty, full and nearly empty tiles; the
# gather through slot / div and rows as they lie
@pytest.mark.parametrize("K", [64, 128, 192, 320, 384, 448])
@pytest.mark.parametrize("N, E, div", [(4, 14, 1), (132, 14, 3), (260, 14, 0), (528, 14, 2), (128, 7679, 1), (272, 7680, 1)])
def test_grouped_products_of_sorted_runs(ops, K, N, E, div):
    g, dev = torch.Generator().manual_seed(K + N), "cuda:0"
    counts = torch.tensor([0, 1, 63, 64, 65, 0, 127, 128, 129, 255, 256, 257, 600, 0])
    counts = torch.cat([counts[:7], counts.new_zeros(E - 14), counts[7:]])
    n = int(counts.sum())
    off = torch.cat([counts.new_zeros(1), counts.cumsum(0)]).int()
    order = torch.randperm(n, generator=g).int() if div else torch.arange(n, dtype=torch.int32)
    x, w14 = torch.randn(-(-n // max(div, 1)), K, generator=g).bfloat16(), (torch.randn(14, N, K, generator=g) / K ** 0.5).bfloat16()
    w = torch.empty(E, N, K, dtype=torch.bfloat16, device=dev)          # (empty experts' weights are never read)
    w[:7], w[-7:] = w14[:7].to(dev), w14[7:].to(dev)
    xd, od, offd = x.to(dev), order.to(dev), off.to(dev)
    out = torch.full((n + 1, N), 3.0, dtype=torch.bfloat16, device=dev)
    for _ in range(2):                                                  # (a second launch finds what the first one left in LDS)
        ops.check(ops.L.qsv_grouped_gemm_sorted(out.data_ptr(), xd.data_ptr(), od.data_ptr() if div else None, max(div, 1), w.data_ptr(), offd.data_ptr(),
                                                E, N, K, 0, 0.0, None, torch.cuda.current_stream().cuda_stream), "grouped")
    y, rows = out.cpu(), x.double()[order.long() // max(div, 1)]
    at = 0
    for e in range(E):
        c = int(counts[e])
        if c:
            ref = rows[at:at + c] @ w14[e if e < 7 else e - (E - 14)].double().T
            # half a unit in the last of bfloat16's 8 digits; float sums of K products of order K^-1/2
            assert ((y[at:at + c].double() - ref).abs() <= 2.0 ** -8 * ref.abs() + K * 2.0 ** -22).all(), (e, c)
        at += c
    assert (y[n] == 3.0).all()


# ... and workgroups that take a second and a third tile: an odd and an even number of steps (the half of the buffer that a tile starts in), input rows of the
# next tile through LDS (from six steps on, up to 7679 experts) and not, stores of 16 and of 8 bytes, rows folded in pairs; the callers' own tiles, whose gather is of 64-bit numbers
@pytest.mark.parametrize("K", [64, 192, 320, 384, 448, 1088])
@pytest.mark.parametrize("N, E, div, act, times, listed", [(8192, 14, 3, 0, 1, False), (12300, 14, 1, 0, 1, False), (8192, 14, 2, 2, 1, False), (5120, 14, 0, 1, 1, False),
                                                           (272, 7679, 2, 0, 20, False), (272, 7680, 2, 0, 20, False), (8192, 14, 3, 0, 1, True), (5120, 14, 0, 2, 1, True)])
def test_grouped_products_of_many_tiles(ops, K, N, E, div, act, times, listed):
    gen, dev = torch.Generator(device="cuda:0").manual_seed(K + N), "cuda:0"
    counts = [times * c for c in (0, 1, 63, 64, 65, 0, 127, 128, 129, 255, 256, 257, 600, 0)]
    n, names = sum(counts), list(range(7)) + list(range(E - 7, E))
    first = [sum(counts[:i]) for i in range(14)]
    order = torch.randperm(n, generator=gen, device=dev) if div else torch.arange(n, device=dev)
    x = torch.randn(-(-n // max(div, 1)), K, generator=gen, device=dev).bfloat16()
    w = torch.empty(E, N, K, dtype=torch.bfloat16, device=dev)          # (empty experts' weights are never read)
    for e, c in zip(names, counts):
        if c:
            w[e] = torch.randn(N, K, generator=gen, device=dev) / K ** 0.5
    wide, s = N // 2 if act == 2 else N, torch.cuda.current_stream().cuda_stream
    out = torch.full((n + 1, wide), 3.0, dtype=torch.bfloat16, device=dev)
    if listed:
        size = ops.L.qsv_grouped_gemm_tile_slots()
        tiles = [(e, f + o, min(size, c - o)) for e, f, c in zip(names, first, counts) for o in range(0, max(c, 1), size)]
        td = torch.tensor(tiles, dtype=torch.int32, device=dev)
        many = len(tiles) * -(-N // 256)
        call = lambda: ops.L.qsv_grouped_gemm(out.data_ptr(), x.data_ptr(), order.data_ptr() if div else None, max(div, 1), w.data_ptr(), td.data_ptr(), len(tiles),      # noqa: E731
                                              N, K, act, 0.0, None, s)
    else:
        at = torch.zeros(E + 1, dtype=torch.int32)
        for e, c in zip(names, counts):
            at[e + 1] = c
        at, od = at.cumsum(0).int().to(dev), order.int()
        many = sum(-(-c // 256) for c in counts) * -(-N // 256)
        call = lambda: ops.L.qsv_grouped_gemm_sorted(out.data_ptr(), x.data_ptr(), od.data_ptr() if div else None, max(div, 1), w.data_ptr(), at.data_ptr(),             # noqa: E731
                                                     E, N, K, act, 0.0, None, s)
    assert many > 256                                                   # (a workgroup for each of 256 CUs)
    for _ in range(2):
        ops.check(call(), "grouped")
    for e, f, c in zip(names, first, counts):
        if not c:
            continue
        # float sums of K products of order K^-1/2; half a unit in the last of bfloat16's 8 digits (or a rounding that falls the other way)
        a, d = x[order[f:f + c] // max(div, 1)].double() @ w[e].double().t(), K * 2.0 ** -22
        if act == 2:
            g, u = a[:, 0::2], a[:, 1::2]
            a, d = _silu(g) * u, d * (1.1 * u.abs() + g.abs()) + 2.0 ** -20 * (_silu(g) * u).abs()
        elif act == 1:
            a, d = torch.relu(a) ** 2, 2.0 * d * a.abs() + d * d
        assert ((out[f:f + c].double() - a).abs() <= 2.0 ** -8 * a.abs() + d).all(), (e, c)
    assert (out[n] == 3.0).all()


@pytest.mark.parametrize("E", [1025, 1600, 8064])
def test_grouped_form_of_many_experts(ops, E):
    check(ops, 600, 2, E, 3, 64, 64, "relu_sq", "input", 0.1)


# The sum over a mixture's rows inside the kernel that uses it: float rows (a step) and rows in the storage type found through their places (a prompt), slots
# without an expert, weights on the inputs, chunks of 1024 columns; and widths that only the sum as a tensor serves.
@pytest.mark.parametrize("T, top, D, ff", [(1, 1, 8, 8), (3, 4, 72, 40), (5, 5, 1032, 64), (64, 4, 2048, 64), (17, 7, 4096, 64), (3, 2, 4104, 64), (600, 2, 64, 64), (400, 4, 1088, 64)])
@pytest.mark.parametrize("weigh", ["output", "input"])
def test_sums_over_experts_inside_their_users(ops, T, top, D, ff, weigh):
    g = torch.Generator().manual_seed(T + D)
    dev, E = "cuda:0", 8
    h, up, down = torch.randn(T, D, generator=g).bfloat16(), (torch.randn(E, ff, D, generator=g) / D ** 0.5).bfloat16(), (torch.randn(E, D, ff, generator=g) / ff ** 0.5).bfloat16()
    idx, wt = torch.rand(T, E, generator=g).argsort(1)[:, :top].int(), torch.rand(T, top, generator=g)
    idx[torch.rand(T, top, generator=g) < 0.2] = -1
    rows = ops.moe_experts(h.to(dev), up.to(dev), down.to(dev), idx.to(dev), wt.to(dev), weigh=weigh, rows=True)
    assert isinstance(rows, ExpertRows)
    k = torch.arange(T * top).view(T, top) if rows.place is None else rows.place.cpu().long().view(T, top).clamp(0)
    w = (wt if weigh == "output" else torch.ones_like(wt)) * (idx >= 0)
    y = (w.double()[..., None] * rows.ys.double().cpu()[torch.where(idx >= 0, k, torch.zeros_like(k))].where((idx >= 0)[..., None], torch.zeros(()).double())).sum(1)
    x, a, c = torch.randn(T, D, generator=g), torch.randn(T, D, generator=g).bfloat16(), torch.randn(T, D, generator=g).bfloat16()
    v, s = torch.randn(D, generator=g).bfloat16(), [torch.randn(D, generator=g).bfloat16() for _ in range(3)]
    gains = [torch.randn(D, generator=g) for _ in range(2)]
    near = lambda got, ref, size: ((got.double().cpu() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -18 + 2.0 ** -7 * size).all()    # noqa: E731
    y = y.bfloat16().double()                                           # (as a tensor holds it; a sum near half a unit may fall the other way)
    xd = x.to(dev)
    hd = ops.add_layer_norm(xd, rows, v.to(dev), 1e-5)
    d = y - y.mean(-1, keepdim=True)
    scale = 1.0 / (d.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt()
    ref = x.double() + d * scale * v.double()
    size = (y.abs().amax(-1, keepdim=True) * scale * v.double().abs() * 4)
    assert near(xd, ref, size) and near(hd, ref, size)
    for parts, more in (([(a, s[0]), (rows, s[1]), (c, s[2])], True), ([(a, None), (rows, None)], False)):
        xd = x.to(dev)
        _, hs = ops.scaled_sum_rms_norms(xd, [(p if p is rows else p.to(dev), None if f is None else f.to(dev)) for p, f in parts], [t.to(dev) for t in gains], 1e-5)
        one = torch.ones(D, dtype=torch.float64)
        ref = x.double() + a.double() * (s[0].double() if more else one) + y * (s[1].double() if more else one) + (c.double() * s[2].double() if more else 0.0)
        inv = 1.0 / (ref.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt()
        size = y.abs() * (s[1].double().abs() if more else 1.0) + ref.abs()
        assert near(xd, ref, size)
        assert all(near(t, ref * inv * gn.double(), size * inv * gn.double().abs()) for t, gn in zip(hs, gains))
    S = 3
    x3, mix, out = torch.randn(T, S, D, generator=g), torch.randn(S, S, generator=g), torch.randn(S, generator=g)
    xd = x3.to(dev)
    ops.hc_write(xd, rows, mix.to(dev), out.to(dev))
    ref = torch.einsum("tsd,sr->trd", x3.double(), mix.double()) + out.double()[None, :, None] * y[:, None]
    assert near(xd, ref, y.abs()[:, None] * out.abs()[None, :, None] + 4)


# ... to the bit what the sum as a tensor gives: slots without an expert, sums in one and two rounds of requests, streams that take the tensor
# (more than four placed slots, 2^22 elements and more) and the last that do not
@pytest.mark.parametrize("placed", [False, True])
@pytest.mark.parametrize("weighed", [False, True])
@pytest.mark.parametrize("T, top, D", [(1, 1, 4), (5, 4, 256), (3, 5, 516), (17, 8, 1028), (2, 9, 3076), (33, 6, 4096), (1024, 5, 4096), (1023, 5, 4096), (1024, 4, 4096)])
def test_sums_inside_their_users_have_the_tensors_bits(ops, T, top, D, placed, weighed):
    g, dev, E = torch.Generator().manual_seed(T + D + top), "cuda:0", 6
    bf = lambda *s: torch.randn(*s, generator=g).bfloat16().to(dev)                                        # noqa: E731
    fl = lambda *s: torch.randn(*s, generator=g).to(dev)                                                   # noqa: E731
    idx = torch.randint(-1, E, (T, top), generator=g, dtype=torch.int32).to(dev)
    place = torch.randperm(T * top, generator=g).int().to(dev) if placed else None
    wt, ys, h = fl(T, top) if weighed else None, bf(T * top, D) if placed else fl(T * top, D), bf(T, D)
    rows = ExpertRows(ops, ys, place, wt, idx, h, E)
    y = rows.dense()
    at = torch.arange(T * top, device=dev) if place is None else place.long()
    terms = ys[at].view(T, top, D).double() * (idx >= 0)[..., None] * (1.0 if wt is None else wt.double()[..., None])
    ref, size = terms.sum(1), terms.abs().sum(1)
    # half a unit in the last of bfloat16's 8 digits (or a rounding that falls the other way), a float sum of `top` products
    assert ((y.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + (top + 1) * 2.0 ** -24 * size).all()
    del terms, ref
    x, a, c, w, f = fl(T, D), bf(T, D), bf(T, D), bf(D), [bf(D) for _ in range(3)]
    x1, x2 = x.clone(), x.clone()
    assert torch.equal(ops.add_layer_norm(x1, rows, w, 1e-5), ops.add_layer_norm(x2, y, w, 1e-5)) and torch.equal(x1, x2)
    for parts in ([(a, f[0]), (y, f[1]), (c, f[2])], [(a, None), (y, None)]):
        x1, x2, gains = x.clone(), x.clone(), [fl(D), fl(D)]
        _, h1 = ops.scaled_sum_rms_norms(x1, [(rows if p is y else p, v) for p, v in parts], gains, 1e-5)
        _, h2 = ops.scaled_sum_rms_norms(x2, parts, gains, 1e-5)
        assert torch.equal(x1, x2) and all(map(torch.equal, h1, h2))
        ref, size = x.double(), x.double().abs()
        for p, v in parts:
            t = p.double() * (1.0 if v is None else v.double())
            ref, size = ref + t, size + t.abs()
        assert ((x1.double() - ref).abs() <= 2.0 ** -22 * size).all()
    for S in (2, 5):
        s1, mix, out = fl(T, S, D), fl(S, S), fl(S)
        s2, s0 = s1.clone(), s1.double()
        ops.hc_write(s1, rows, mix, out)
        ops.hc_write(s2, y, mix, out)
        assert torch.equal(s1, s2)
        ref = s0.transpose(1, 2) @ mix.double() + y.double()[..., None] * out.double()
        size = s0.abs().transpose(1, 2) @ mix.abs().double() + y.abs().double()[..., None] * out.abs().double()
        assert ((s1.double() - ref.transpose(1, 2)).abs() <= (S + 2) * 2.0 ** -24 * size.transpose(1, 2)).all()


@pytest.mark.parametrize("T, top, D, ff", [(3, 2, 64, 64), (40, 4, 72, 40), (1200, 2, 64, 128)])
@pytest.mark.parametrize("knobs", [{}, dict(moe_token_slots=10 ** 9, moe_sorted_above=10 ** 9)], ids=["rule", "per token"])
def test_slots_without_an_expert_add_nothing(T, top, D, ff, knobs):
    o = make_ops("hip", torch.bfloat16, torch.device("cuda:0"))
    for k, v in knobs.items():
        setattr(o, k, v)
    check(o, T, top, 6, 1, D, ff, "swiglu", "output", 0.2, none=True)


# rows longer than 4096, up to a layer of 5120 x 5632
@pytest.mark.parametrize("T, top, E, D, ff", [(1, 4, 6, 5120, 5632), (16, 4, 6, 4104, 16), (17, 2, 3, 64, 8200), (3, 4, 4, 20000, 24), (20, 3, 4, 24, 12288)])
@ACTS
def test_expert_major_form_of_wide_layers(ops, T, top, E, D, ff, act, weigh):
    check(ops, T, top, E, 0, D, ff, act, weigh, 0.5)


@pytest.mark.parametrize("T, D, ff", [(2, 64, 4104), (3, 16400, 24)])
def test_float_storage_beyond_a_workgroups_lds(T, D, ff):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    dev, E, top = torch.device("cuda:0"), 5, 4
    g = torch.Generator().manual_seed(ff)
    h, up, down = torch.randn(T, D, generator=g), torch.randn(E, ff, D, generator=g) / D ** 0.5, torch.randn(E, D, ff, generator=g) / ff ** 0.5
    idx, wt = torch.rand(T, E, generator=g).argsort(1)[:, :top].int(), torch.rand(T, top, generator=g)
    y = make_ops("hip", torch.float32, dev).moe_experts(*(t.to(dev) for t in (h, up, down, idx, wt))).double().cpu()
    ref = torch.stack([sum(w.double() * (down[e].double() @ torch.relu(up[e].double() @ h[t].double()) ** 2) for e, w in zip(idx[t], wt[t])) for t in range(T)])
    # float sums of D and of ff products of order one on average, squared in between
    assert ((y - ref).abs() <= 2.0 ** -23 * (2 * D + ff) * 4).all()


# sizes the grouped kernel does not take, weights inside 16 bytes: what was computed (any weighting) and captured stays so
@pytest.mark.parametrize("T, top, E, D, ff, shift, graph", [(500, 2, 4, 72, 40, 0, False), (256, 4, 6, 200, 64, 0, True), (450, 2, 4, 64, 128, 3, False),
                                                            (20, 3, 5, 64, 64, 1, False), (600, 2, 4, 64, 128, 5, False)])
@pytest.mark.parametrize("act, weigh", [("relu_sq", "input"), ("relu_sq", "output"), ("swiglu", "input")])
def test_sizes_and_addresses_between_the_forms(ops, T, top, E, D, ff, shift, graph, act, weigh):
    check(ops, T, top, E, 0, D, ff, act, weigh, 0.3, shift, graph)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [1, 5, 1023, 1025, 2050])
@pytest.mark.parametrize("E, G, keep, top, D, score, group_top, renorm", [
    (1, 1, 1, 1, 8, "softmax", 1, False), (16, 4, 2, 4, 2048, "softmax", 1, False), (16, 1, 1, 4, 2040, "softmax", 1, True),
    (17, 17, 5, 3, 64, "sigmoid", 1, False), (64, 8, 3, 24, 4096, "sigmoid", 2, True), (33, 1, 1, 33, 136, "sigmoid", 1, False),
    (64, 64, 64, 6, 8, "softmax", 1, False), (8, 2, 1, 3, 1032, "softmax", 1, True), (9, 1, 1, 2, 1024, "sigmoid", 1, False)])
def test_router(dtype, n, E, G, keep, top, D, score, group_top, renorm):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    dev = torch.device("cuda:0")
    o = make_ops("hip", dtype, dev)
    g = torch.Generator().manual_seed(n + E)
    h, r = torch.randn(n, D, generator=g).to(dtype), (torch.randn(E, D, generator=g) / D ** 0.5 * 2).to(dtype)
    corr = torch.randn(E, generator=g) * 0.1
    idx, wt = o.moe_route(h.to(dev), r.to(dev), top, G, keep, score=score, correction=corr.to(dev), group_top=group_top, renorm=renorm, scale=1.5)
    idx, wt = idx.cpu().long(), wt.cpu().double()
    z = h.double() @ r.double().T
    s = torch.softmax(z, -1) if score == "softmax" else torch.sigmoid(z)
    c = s + corr.double()
    best = c.view(n, G, E // G).sort(-1, descending=True).values[..., :group_top].sum(-1)
    kept = torch.zeros(n, G, dtype=torch.bool).scatter_(1, best.topk(keep, -1).indices, True)
    c = c.masked_fill(~kept.repeat_interleave(E // G, 1), -9.0)
    tol = 4e-6                                                          # float sums of D products of order one
    # every chosen expert is eligible and the k-th of them is as good as the k-th best, up to float rounding of the scores
    got = c.gather(1, idx)
    assert (idx.sort(1).values.diff(dim=1) > 0).all() and ((got - c.topk(top, -1).values).abs() <= tol).all()
    w = s.gather(1, idx)
    w = (w / w.sum(-1, keepdim=True) if renorm else w) * 1.5
    assert ((wt - w).abs() <= 4 * tol).all()


def test_router_takes_what_is_not_a_number_last_and_ties_by_index():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    dev = torch.device("cuda:0")
    o = make_ops("hip", torch.float32, dev)
    h = torch.zeros(1, 8)
    h[0, 0] = 1.0
    r = torch.zeros(6, 8)
    r[:, 0] = torch.tensor([0.0, -0.0, 2.0, float("nan"), 2.0, float("-inf")])
    idx, _ = o.moe_route(h.to(dev), r.to(dev), 6, 1, 1, score="sigmoid")
    assert idx.cpu()[0].tolist() == [2, 4, 0, 1, 5, 3]
    idx, _ = o.moe_route(torch.full_like(h, float("nan")).to(dev), r.to(dev), 3, 3, 2)
    assert sorted(set(idx.cpu()[0].tolist())) == sorted(idx.cpu()[0].tolist()) and idx.min() >= 0 and idx.max() < 6


# a shared expert in the same two launches: edges of 16 / 32 tokens, narrower and wider than the others, remainders of rows and of the reduction
@pytest.mark.parametrize("T", [1, 2, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("D, ff, sff, weigh", [(256, 128, 128, "input"), (264, 72, 200, "output"), (2048, 64, 24, "output"), (72, 136, 1408, "input")])
def test_shared_expert_in_the_launch(ops, T, D, ff, sff, weigh):
    E, top, g = 5, 2, torch.Generator().manual_seed(T + D)
    mat = lambda *s: (torch.randn(*s, generator=g) / s[-1] ** 0.5).bfloat16()                              # noqa: E731
    h, up, down, sup, sdown = torch.randn(T, D, generator=g).bfloat16(), mat(E, 2 * ff, D), mat(E, D, ff), mat(2 * sff, D), mat(D, sff)
    idx, wt = torch.rand(T, E, generator=g).argsort(dim=1)[:, :top].int(), torch.rand(T, top, generator=g)
    args = [t.cuda() for t in (h, up, down, idx, wt)]
    both = ops.moe_experts_shared(*args, sup.cuda(), sdown.cuda(), weigh=weigh)
    assert both is not None and torch.equal(both[0], ops.moe_experts(*args, act="swiglu", weigh=weigh))
    apart = linear(ops.glu(linear(args[0], sup.cuda())), sdown.cuda())
    assert torch.equal(both[1], apart)                                  # (these sizes go through the same stream of products: the same bits)


def test_shared_expert_where_it_is_left_alone(ops):
    t = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device="cuda:0")                                  # noqa: E731
    route = lambda T: (torch.zeros(T, 2, dtype=torch.int32, device="cuda:0"), torch.zeros(T, 2, device="cuda:0"))       # noqa: E731
    up, down = t(5, 256, 128), t(5, 128, 128)
    for T, sup, sdown in ((65, t(256, 128), t(128, 128)), (4, t(200, 128), t(128, 100)), (4, t(256, 128).float(), t(128, 128).float()),
                          (4, t(32769)[1:].view(256, 128), t(128, 128))):
        assert ops.moe_experts_shared(t(T, 128), up, down, *route(T), sup, sdown) is None


# Row kernels that route the row they leave: the bits of the two launches one by one; one to four chunks of 1024 columns, parts of one, more experts than are
# summed side by side, every option of the router.
ROUTERS = [(16, dict(top_k=4, groups=4, keep=2)), (5, dict(top_k=2, groups=1, keep=1, bias=True, renorm=True)), (64, dict(top_k=6, groups=8, keep=3, score="sigmoid", correction=True,
           group_top=2, scale=1.5)), (17, dict(top_k=17, groups=1, keep=1, score="sigmoid", group_top=2)), (1, dict(top_k=1, groups=1, keep=1))]


@pytest.mark.parametrize("T, D", [(1, 8), (3, 264), (2, 1024), (64, 2048), (5, 2056), (33, 4096)])
@pytest.mark.parametrize("E, kind", ROUTERS, ids=[str(e) for e, _ in ROUTERS])
def test_routing_on_the_way_out(ops, T, D, E, kind):
    g, dev = torch.Generator().manual_seed(T + D + E), "cuda:0"
    bf = lambda *s: torch.randn(*s, generator=g).bfloat16().to(dev)                                        # noqa: E731
    fl = lambda *s: torch.randn(*s, generator=g).to(dev)                                                   # noqa: E731
    route = dict(kind, router=bf(E, D) * (3.0 / D ** 0.5))
    if kind.get("bias"):
        route["bias"] = bf(E)
    if kind.get("correction"):
        route["correction"] = fl(E)

    def same(fused, apart, x1, x2):
        h, (idx, wt) = fused
        i2, w2 = ops.moe_route(apart, **route)
        assert torch.equal(h, apart) and torch.equal(x1, x2) and torch.equal(idx, i2) and torch.equal(wt, w2)

    x, y, w, b = fl(T, D), bf(T, D), bf(D), bf(D)
    x1, x2 = x.clone(), x.clone()
    same(ops.add_layer_norm(x1, y, w, 1e-5, route=route), ops.add_layer_norm(x2, y, w, 1e-5), x1, x2)
    for S in (1, 2, 4):
        s1 = fl(T, S, D)
        s2, mix, out, then = s1.clone(), fl(S, S), fl(S), (fl(S), (w, b, 0.7))
        same(ops.hc_write(s1, y, mix, out, then_read=then, route=route), ops.hc_write(s2, y, mix, out, then_read=then), s1, s2)
    gains, table, tokens = [fl(D), fl(D)], bf(11, D), torch.randint(0, 11, (T,), generator=g, dtype=torch.int32).to(dev)
    x1, hs, routed = ops.scaled_sum_rms_norms(None, [], gains, 1e-5, tokens=tokens, table=table, route=route)
    x2, apart = ops.scaled_sum_rms_norms(None, [], gains, 1e-5, tokens=tokens, table=table)
    assert torch.equal(hs[0], apart[0])
    same((hs[1], routed), apart[1], x1, x2)
    top = min(2, E)
    idx = torch.randint(-1, E, (T, top), generator=g, dtype=torch.int32).to(dev)
    for wt, parts in ((fl(T, top), 2), (None, 3)):
        rows = ExpertRows(ops, fl(T * top, D), None, wt, idx, y, E)
        ps = [(bf(T, D), bf(D)), (rows, bf(D)), (bf(T, D), bf(D))][:parts]
        x1, x2 = x.clone(), x.clone()
        _, hs, routed = ops.scaled_sum_rms_norms(x1, ps, gains, 1e-5, route=route)
        _, apart = ops.scaled_sum_rms_norms(x2, ps, gains, 1e-5)
        assert torch.equal(hs[0], apart[0])
        same((hs[1], routed), apart[1], x1, x2)


def test_routing_apart_where_the_rows_do_not_take_it(ops):
    t = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device="cuda:0")                                  # noqa: E731
    for T, D, E, kw in ((513, 64, 8, {}), (2, 4104, 8, {}), (2, 60, 4, {}), (2, 64, 65, {}), (2, 64, 8, dict(groups=3)), (2, 64, 8, dict(top_k=9))):
        route = dict(dict(top_k=2, groups=1, keep=1), router=t(E, D)) | kw
        assert ops.add_layer_norm(torch.zeros(T, D, device="cuda:0"), t(T, D), t(D), 1e-5, route=route)[1] is None
    route = dict(top_k=2, groups=1, keep=1, router=t(8, 64))
    then = (torch.zeros(5, device="cuda:0"), (t(64), t(64), 1.0))
    assert ops.hc_write(torch.zeros(2, 5, 64, device="cuda:0"), t(2, 64), torch.zeros(5, 5, device="cuda:0"), torch.zeros(5, device="cuda:0"), then_read=then, route=route)[1] is None


# weights left in the caches: the same products from the same launches, only how the weights are asked for differs
@pytest.mark.parametrize("T", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("D, ff, sff", [(256, 128, 64), (2048, 384, 1408), (72, 136, 200)])
def test_weights_kept_in_the_caches(ops, T, D, ff, sff):
    from qserve_amd.layers.ops import float_linear
    kept, g, E, top = make_ops("hip", torch.bfloat16, torch.device("cuda:0")), torch.Generator().manual_seed(T + D), 5, 3
    mat = lambda *s: (torch.randn(*s, generator=g) / s[-1] ** 0.5).bfloat16().cuda()                       # noqa: E731
    h, up, down, sup, sdown = mat(T, D), mat(E, 2 * ff, D), mat(E, D, ff), mat(2 * sff, D), mat(D, sff)
    idx, wt = torch.rand(T, E, generator=g).argsort(1)[:, :top].int().cuda(), torch.rand(T, top, generator=g).cuda()
    idx[0, 0] = -1
    assert kept.kept_above is None and not kept._kept(64)
    kept.kept_above = 0
    assert torch.equal(kept.linear(h, sup), linear(h, sup)) and torch.equal(kept.float_linear(h, sup), float_linear(h, sup))
    for act, u in (("swiglu", up), ("relu_sq", up[:, :ff].contiguous())):
        for weigh in ("input", "output"):
            assert torch.equal(kept.moe_experts(h, u, down, idx, wt, act=act, weigh=weigh), ops.moe_experts(h, u, down, idx, wt, act=act, weigh=weigh))
    a, b = (o.moe_experts_shared(h, up, down, idx, wt, sup, sdown) for o in (kept, ops))
    assert (a is None) == (b is None) and (a is None or all(torch.equal(x, y) for x, y in zip(a, b)))
