"""Kernels of a step that make what two launches made: the same bits."""
import types

import pytest
import torch

from qserve_amd.layers.ops import ExpertRows, NormedPair, make_ops

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16


@pytest.fixture
def ops():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return make_ops("hip", BF, DEV)


def _rand(g, *shape, dtype=BF, scale=1.0):
    return (torch.randn(*shape, generator=g) * scale).to(dtype).to(DEV)


def _runs(T, fresh):
    """T runs of one token on slots in another order; those in `fresh` start their sequence."""
    rows = [[T - 1 - i, i, 1, 0 if i in fresh else 5 + i] for i in range(T)]
    return types.SimpleNamespace(items=[(r[0], r[1], 1) for r in rows], runs=lambda r=torch.tensor(rows, dtype=torch.int32, device=DEV): r)


# one to four groups of 64 rows, heads that share keys, columns of less than a workgroup, each kind of decay and gate
@pytest.mark.parametrize("T, H, QH, dim, vdim", [(1, 2, 2, 8, 4), (16, 16, 4, 64, 128), (3, 6, 3, 72, 64), (5, 4, 4, 256, 32), (64, 3, 1, 128, 16)])
@pytest.mark.parametrize("delta, floats, decays", [(True, True, "channel"), (False, False, "channel"), (True, False, "head"), (False, True, "constant")])
@pytest.mark.parametrize("kind", ["silu", "sigmoid"])
def test_recurrence_with_its_norm_and_gate(ops, T, H, QH, dim, vdim, delta, floats, decays, kind):
    g = torch.Generator().manual_seed(T + dim)
    q, k = (_rand(g, T, QH * dim + 4, dtype=torch.float32 if floats else BF, scale=dim ** -0.5)[:, 4:] for _ in range(2))
    v, beta = _rand(g, T, H * vdim, dtype=q.dtype), _rand(g, T, H + 1)[:, 1:] if delta else None
    decay = torch.rand(*{"channel": (T, H * dim), "head": (T, H), "constant": (H,)}[decays], generator=g).to(DEV)
    state, w, gate = _rand(g, T, H, dim, vdim, dtype=torch.float32), _rand(g, vdim), _rand(g, T, H * vdim + 4)[:, 4:]
    batch, other = _runs(T, {0, T - 1}), state.clone()
    ref = ops.head_rms_gate(ops.recurrent_scan(q, k, v, decay, beta, state, batch, H, QH, dim, vdim, 0.3), w, gate, kind, 1e-5)
    ops.recurrent_scan = None                                                                    # (one launch, or an error)
    out = ops.recurrent_gated(q, k, v, decay, beta, other, batch, H, QH, dim, vdim, 0.3, w, gate, kind, 1e-5)
    assert torch.equal(out, ref) and torch.equal(state, other)


# widths of one and several workgroups a token and their remainders, one to four streams, sequences that start, tokens without experts
@pytest.mark.parametrize("T, S, D", [(1, 1, 4), (5, 2, 2048), (16, 3, 1028), (64, 4, 4096), (600, 2, 1040)])
@pytest.mark.parametrize("weighted", [True, False])
def test_streams_written_and_read_shifted(ops, T, S, D, weighted):
    g = torch.Generator().manual_seed(T + D)
    f32 = dict(dtype=torch.float32)
    x, ys, mix = _rand(g, T, S, D, **f32), _rand(g, T * 3, D, **f32), _rand(g, S, S, **f32)
    idx = torch.randint(-1, 9, (T, 3), generator=g, dtype=torch.int32).to(DEV)
    y = ExpertRows(ops, ys, None, torch.rand(T, 3, generator=g).to(DEV) if weighted else None, idx, torch.empty(T, D, dtype=BF, device=DEV), 8)
    w_out, w_in, norm, shift = _rand(g, S, **f32), _rand(g, S, **f32), (_rand(g, D), _rand(g, D), 0.7), _rand(g, D)
    prev, i32 = _rand(g, 2 * T, D, **f32), lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)             # noqa: E731
    batch = types.SimpleNamespace(items=[(i, i, 1) for i in range(T)], run_off=i32([0] * T), state_rd=i32([-1 if i % 5 == 0 else 2 * i for i in range(T)]),
                                  state_wr=i32([2 * i + 1 for i in range(T)]))
    a, b, pa, pb = x.clone(), x, prev.clone(), prev
    ops.hc_write(a, y, mix, w_out)
    ref = ops.hc_read(a, w_in, norm, shift, batch, pa)
    ops.hc_read = None
    h = ops.hc_write_read(b, y, mix, w_out, w_in, norm, shift, batch, pb)
    assert torch.equal(h, ref) and torch.equal(a, b) and torch.equal(pa, pb)


@pytest.mark.parametrize("T, S, D", [(1, 2, 8), (16, 2, 2048), (3, 4, 1032), (64, 3, 4096)])
def test_mean_of_normed_rows_on_the_way_to_the_router(ops, T, S, D):
    g = torch.Generator().manual_seed(D)
    x, mix, w_out, w_in = (_rand(g, *s, dtype=torch.float32) for s in ((T, S, D), (S, S), (S,), (S,)))
    pair = NormedPair(ops, _rand(g, T, D), _rand(g, D), _rand(g, T, D), _rand(g, D), 1e-5)
    route = dict(router=_rand(g, 16, D, scale=D ** -0.5), top_k=4, groups=1, keep=1, bias=_rand(g, 16), renorm=True)
    then, other = (w_in, (_rand(g, D), _rand(g, D), 0.7)), x.clone()
    ref, (idx, wt) = ops.hc_write(x, pair.dense(), mix, w_out, then_read=then, route=route)
    ops.rms_pair_mean = None
    h, routed = ops.hc_write(other, pair, mix, w_out, then_read=then, route=route)
    assert torch.equal(h, ref) and torch.equal(x, other) and torch.equal(routed[0], idx) and torch.equal(routed[1], wt)


# the smallest and largest latent, one to four stages a wave and waves without one, one to four rows a wave, part groups of weight rows
@pytest.mark.parametrize("T", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("q_rank, kv_rank, rot_dim, rot_n, N", [(64, 8, 0, 0, 1024), (768, 512, 64, 64, 3072), (768, 512, 0, 0, 2048), (320, 256, 64, 22, 1532), (1024, 2000, 64, 64, 1028),
                                                                (512, 512, 64, 32, 3076)])
def test_latents_normed_by_their_product(ops, T, q_rank, kv_rank, rot_dim, rot_n, N):
    g = torch.Generator().manual_seed(T + q_rank)
    R = kv_rank + rot_dim
    down, qw, kw, w = _rand(g, T, q_rank + R + 16), _rand(g, q_rank), _rand(g, kv_rank), _rand(g, N, q_rank, scale=q_rank ** -0.5)
    rope = torch.randn(T + 1, 2, rot_n // 2, generator=g).to(DEV) if rot_n else None
    pos, slot = torch.arange(T, 0, -1, dtype=torch.int32, device=DEV), torch.randperm(2 * T, generator=g)[:T].to(DEV)
    pools = [torch.zeros(2 * T, R, dtype=BF, device=DEV) for _ in range(2)]
    args = [(down, 8, q_rank, qw, q_rank + 12, kv_rank, kw, rot_dim, rot_n, rope, p, slot, pos, 1e-5) for p in pools]
    out = ops.latent_up(*args[0], w)
    assert out is not None and torch.equal(out, ops.linear(ops.latent_prep(*args[1]), w)) and torch.equal(*pools)
    kept = make_ops("hip", BF, DEV)
    kept.kept_above = 0
    assert torch.equal(out, kept.latent_up(*args[0], w))


def test_latents_that_take_two_launches(ops):
    g = torch.Generator().manual_seed(1)
    pos, slot = torch.arange(64, dtype=torch.int32, device=DEV), torch.arange(65, device=DEV)
    for T, q_rank, kv_rank, N, off in ((17, 768, 512, 2048, 0), (9, 1024, 512, 6144, 0), (4, 768, 512, 6160, 0), (4, 1088, 512, 2048, 0), (4, 96, 512, 2048, 0), (4, 768, 510, 2048, 0),
                                       (4, 768, 512, 2048, 4)):
        down, pool = _rand(g, T, q_rank + kv_rank + off)[:, off:].contiguous(), torch.zeros(65, kv_rank, dtype=BF, device=DEV)
        qw = _rand(g, q_rank + 1)[1:] if off else _rand(g, q_rank)
        assert ops.latent_up(down, 0, q_rank, qw, q_rank, kv_rank, _rand(g, kv_rank), 0, 0, None, pool, slot[:T], pos[:T], 1e-5, _rand(g, N, q_rank)) is None


# one and two rows, one and several stages a wave (and waves without one), rows shorter than their threads, part groups of weight rows; each form of the sum, more experts than a trip takes
@pytest.mark.parametrize("T", [1, 2])
@pytest.mark.parametrize("D, N, E", [(64, 1024, 8), (576, 1028, 16), (1024, 4096, 5), (1088, 2560, 16), (2048, 5120, 16), (2048, 4096, 40), (1024, 6148, 16)])
def test_norms_with_the_product_of_the_first(ops, T, D, N, E):
    g = torch.Generator().manual_seed(T + D)
    f32 = dict(dtype=torch.float32)
    gains, w, table = [_rand(g, D, **f32) for _ in range(2)], _rand(g, N, D, scale=D ** -0.5), _rand(g, 11, D)
    route = dict(router=_rand(g, E, D, scale=3.0 * D ** -0.5), top_k=2, groups=1, keep=1, score="sigmoid", scale=1.5)
    tokens, x = torch.randint(0, 11, (T,), generator=g, dtype=torch.int32).to(DEV), _rand(g, T, D, **f32)
    forms = [(None, [], dict(tokens=tokens, table=table))]
    for top, weighted, parts in ((2, True, 2), (4, False, 3), (6, True, 3)):
        idx = torch.randint(-1, E, (T, top), generator=g, dtype=torch.int32).to(DEV)
        y = ExpertRows(ops, _rand(g, T * top, D, **f32), None, torch.rand(T, top, generator=g).to(DEV) if weighted else None, idx, _rand(g, T, D), E)
        forms.append((x, [(_rand(g, T, D), _rand(g, D)), (y, _rand(g, D) if weighted else None), (_rand(g, T, D), _rand(g, D))][:parts], {}))
    if N > (6144 if T == 1 else 4096):                                      # (two launches)
        assert ops.scaled_sum_rms_norms_product(None, [], gains, 1e-5, route, w, tokens=tokens, table=table) is None
        return
    for at, parts, kw in forms:
        x1, h1, r1, out = ops.scaled_sum_rms_norms_product(at, parts, gains, 1e-5, route, w, **kw)
        x2, h2, r2 = ops.scaled_sum_rms_norms(None if at is None else at.clone(), parts, gains, 1e-5, route=route, **kw)
        assert torch.equal(x1, x2) and all(torch.equal(a, b) for a, b in zip((*h1, *r1), (*h2, *r2))) and torch.equal(out, ops.linear(h2[0], w))
        assert at is None or at is x and x1 is not x
    assert ops.scaled_sum_rms_norms_product(None, [], gains, 1e-5, route, w, tokens=torch.zeros(3, dtype=torch.int32, device=DEV), table=table) is None
    assert ops.scaled_sum_rms_norms_product(None, [], gains[:1], 1e-5, route, w, tokens=tokens, table=table) is None


# three stages a wave and a row that ends inside one, rows that end inside a workgroup, all slots of a search, experts with none, up to 16, up to 32 and more slots; beside
# experts that nobody chooses (so many that the slots are looked for first)
@pytest.mark.parametrize("T, top, D, ff", [(16, 4, 768, 776), (64, 2, 776, 768), (64, 4, 2048, 1032), (256, 4, 1024, 840), (250, 4, 1304, 2048)])
@pytest.mark.parametrize("act, weigh", [("relu_sq", "output"), ("swiglu", "input")])
@pytest.mark.parametrize("kept", [None, 0])
def test_expert_weights_requested_before_their_slots(ops, T, top, D, ff, act, weigh, kept):
    g = torch.Generator().manual_seed(T + D)
    E, more = 8, T * top // 4 + 1
    rows = ff * (2 if act == "swiglu" else 1)
    up, down, h = _rand(g, E, rows, D, scale=D ** -0.5), _rand(g, E, D, ff, scale=ff ** -0.5), _rand(g, T, D)
    share = torch.tensor([0.0, 0.02, 0.05, 0.08, 0.1, 0.15, 0.2, 0.4])
    idx = torch.multinomial(share, T * top, replacement=True, generator=g).int().view(T, top)
    idx[0, 0] = -1
    idx, wt = idx.to(DEV), torch.rand(T, top, generator=g).to(DEV)
    ops.moe_expert_major_slots, ops.kept_above = 10 ** 9, kept
    out = ops.moe_experts(h, up, down, idx, wt, act=act, weigh=weigh)
    wide = [torch.cat([w, w.new_zeros(more - E, *w.shape[1:])]) for w in (up, down)]
    assert torch.equal(out, ops.moe_experts(h, *wide, idx, wt, act=act, weigh=weigh))
