"""Row kernels that take four columns a thread against their forms for any width and address: the same operands a few elements off the alignment."""
import numpy as np
import pytest
import torch

from qserve_amd.layers.ops import make_ops
from qserve_amd.serving.engine import StepBatch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TYPES = pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])


def make(dtype):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return make_ops("hip", dtype, torch.device(DEV))


def off(t):
    """The same values, the storage starting one element late."""
    return torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)


def ints(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


@TYPES
@pytest.mark.parametrize("T, q_rank, kv_rank, rot_dim, rot_n", [(1, 4, 4, 0, 0), (3, 768, 512, 64, 64), (5, 768, 512, 64, 22), (2, 8, 1024, 4, 2), (65, 1536, 2000, 64, 64), (2, 2056, 2040, 0, 0)])
def test_latent_prep(dtype, T, q_rank, kv_rank, rot_dim, rot_n):
    ops, g = make(dtype), torch.Generator().manual_seed(T + q_rank)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)                                        # noqa: E731
    R = kv_rank + rot_dim
    down, qw, kw = rnd(T, q_rank + R + 8), rnd(q_rank), rnd(kv_rank)
    rope = torch.randn(T + 1, 2, rot_n // 2, generator=g).to(DEV) if rot_n else None
    pos, slot = ints(list(range(T, 0, -1))), torch.randperm(2 * T, generator=g)[:T].to(DEV)
    out = []
    for q in (qw, off(qw)):                                              # (off the alignment: a column at a time)
        pool = torch.zeros(2 * T, R, dtype=dtype, device=DEV)
        out.append((ops.latent_prep(down, 0, q_rank, q, q_rank + 4, kv_rank, kw, rot_dim, rot_n, rope, pool, slot, pos, 1e-5), pool))
    for a, b in zip(*out):
        # sums of squares in another order, and a turn's second product rounded or not before the sum (terms below 10: 2^-24 of each): the last bit
        a, b = a.double(), b.double()
        assert ((a - b).abs() <= (2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -20) * b.abs() + 2e-6).all()
        assert (a != b).float().mean() < 0.02 or dtype == torch.float32


@TYPES
@pytest.mark.parametrize("T, H, dim", [(1, 1, 4), (3, 5, 12), (16, 16, 64), (65, 3, 1028)])
@pytest.mark.parametrize("log", [False, True])
def test_decay_and_rotation(dtype, T, H, dim, log):
    ops, g = make(dtype), torch.Generator().manual_seed(T + dim)
    z, b = (torch.randn(T, H * dim + 8, generator=g).to(dtype).to(DEV), torch.randn(H * dim, generator=g).to(dtype).to(DEV))
    a = torch.randn(H, generator=g).to(DEV) if log else None
    z = z[:, 4:4 + H * dim]
    assert torch.equal(ops.decay(z, b, a, 16.0, H, dim), ops.decay(z, off(b), a, 16.0, H, dim))
    n = dim // 4 * 8
    o, pos, rope = torch.randn(T, H, n, generator=g).to(dtype).to(DEV), ints(list(range(T))), torch.randn(T, 2, n // 2, generator=g).to(DEV)
    assert torch.equal(ops.rotate_heads(o.clone(), rope, pos, -1.0), ops.rotate_heads(off(o), rope, pos, -1.0))


@TYPES
@pytest.mark.parametrize("T, S, D", [(1, 1, 4), (3, 2, 1028), (16, 3, 2048), (5, 4, 4096), (2, 5, 72)])
def test_streams_norm_and_branches(dtype, T, S, D):
    ops, g = make(dtype), torch.Generator().manual_seed(T + D)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)                                        # noqa: E731
    x, w, b, rows = torch.randn(T, S, D, generator=g).to(DEV), rnd(D), rnd(D), ints(list(range(T))[::-1])
    assert torch.equal(ops.dyt_sum_rows(x, rows, (w, b, 0.6)), ops.dyt_sum_rows(x, rows, (off(w), b, 0.6)))
    u, v = rnd(T, D), rnd(T, D)
    ref = 0.5 * sum(t.double() / (t.double().pow(2).mean(-1, keepdim=True) + 1e-5).sqrt() * f.double() for t, f in ((u, w), (v, b)))
    got = ops.rms_pair_mean(u, w, v, b, 1e-5).double()
    assert ((got - ref).abs() <= (2.0 ** -8 if dtype == torch.bfloat16 else 0.0) * ref.abs() + 2e-5).all()


# runs: (first position, tokens); a run behind its first token reads the history
@TYPES
@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("runs", [((0, 1), (7, 1), (1, 1)), ((0, 5), (3, 2)), ((2, 3), (0, 2), (9, 4))])
def test_convolved_heads(dtype, taps, runs):
    ops, g = make(dtype), torch.Generator().manual_seed(taps + len(runs))
    T, qc, G, kd, vd = sum(n for _, n in runs), 40, 2, 8, 12
    C, past = qc + G * (kd + vd), taps - 1
    proj, w = torch.randn(T, C + 4, generator=g).to(dtype).to(DEV), torch.randn(taps, C, generator=g).to(DEV)
    hist = torch.randn(2 * len(runs), past, C, generator=g).to(DEV)
    off_, rd, wr, pos, items, at = [], [], [], [], [], 0
    for r, (start, n) in enumerate(runs):
        off_ += range(n)
        rd += [2 * r if start else -1] * n
        wr += [-1] * (n - 1) + [2 * r + 1]
        pos += range(start, start + n)
        items.append((r, at, n))
        at += n
    batch = StepBatch(tokens=None, seq=None, pos=ints(pos), slot=torch.arange(T, device=DEV), block_table=None, max_pos=max(pos), n_tokens=T, items=items,
                      run_off=ints(off_), state_rd=ints(rd), state_wr=ints(wr))
    out = []
    for f in (w, off(w)):
        h, pool = hist.clone(), torch.zeros(G, T, vd + kd, dtype=dtype, device=DEV)
        out.append((ops.conv_heads_cache(proj, f, h, batch, qc, G, kd, vd, pool, 0.3, (0.1, 4.0)), pool, h))
    assert all(torch.equal(a, b) for a, b in zip(*out))
    # ... and the convolution in front of a recurrence
    h1, h2, taps_of = hist.clone(), hist.clone(), w.t().contiguous()
    a, b = ops.conv_silu_unit(proj, 0, taps_of, h1, batch, 4, 8), ops.conv_silu_unit(proj, 0, off(taps_of), h2, batch, 4, 8)
    # eight squares added in another order, four products: some units of 2^-24 of values below 16
    assert ((a - b).abs() <= 1e-5).all() and torch.equal(h1, h2)


# a recurrence's second stages in one launch: the bits of the launches one by one; edges of 16 and 32 rows, widths off the alignment, both kinds of decay
@pytest.mark.parametrize("T", [1, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("H, dim, r, gate, rg, log", [(16, 64, 64, 0, 0, False), (3, 5, 24, 0, 0, True), (16, 128, 16, 2048, 136, True), (1, 17, 8, 40, 72, False)])
def test_decay_products(T, H, dim, r, gate, rg, log):
    from qserve_amd.layers.ops import float_linear, linear
    ops, g = make(torch.bfloat16), torch.Generator().manual_seed(T + dim)
    rnd = lambda *s: torch.randn(*s, generator=g).bfloat16().to(DEV)                                       # noqa: E731
    proj, w, b, wg = rnd(T, r + rg + 16), rnd(H * dim, r) * 0.3, rnd(H * dim), rnd(gate, rg) if gate else None
    a = torch.randn(H, generator=g).to(DEV) if log else None
    z, x = proj[:, 8:8 + r], proj[:, 8 + r:8 + r + rg] if gate else None
    d, y = ops.decay_products(z, w, b, a, 16.0, H, dim, x, wg)
    assert torch.equal(d, ops.decay(linear(z, w), b, a, 16.0, H, dim)) and (y is None if not gate else torch.equal(y, linear(x, wg)))
    assert torch.equal(float_linear(z, w), linear(z, w).float())
    # ... and behind what the one launch takes
    z = rnd(T, r)[:, 1:r - 7 + 1] if r > 16 else rnd(65, r)
    w = w[:, :z.size(1)].contiguous()
    assert torch.equal(ops.decay_products(z, w, b, a, 16.0, H, dim)[0], ops.decay(linear(z, w), b, a, 16.0, H, dim))


@TYPES
@pytest.mark.parametrize("T, D", [(1, 4), (3, 1028), (70, 2048)])
def test_embeddings(dtype, T, D):
    ops, g = make(dtype), torch.Generator().manual_seed(T + D)
    table, tokens = torch.randn(9, D, generator=g).to(dtype).to(DEV), torch.randint(0, 9, (T,), generator=g, dtype=torch.int32).to(DEV)
    assert all(torch.equal(a, b) for a, b in zip(ops.embed(tokens, table), ops.embed(tokens, off(table))))
    assert torch.equal(ops.embed_streams(tokens, table, 1.7, 3), ops.embed_streams(tokens, off(table), 1.7, 3))


@pytest.mark.parametrize("n", [0, 1, 255, 960, 961, 3839, 3840, 3841, 9000])
def test_words_of_a_step(n):
    ops, g = make(torch.bfloat16), np.random.default_rng(n)
    out, words = torch.full((n + 1,), -7, dtype=torch.int32, device=DEV), g.integers(-2 ** 31, 2 ** 31, n, dtype=np.int64).astype(np.int32)
    keep = words.copy()
    ops.put_words(out[:n], words)
    words[:] = 0                                                         # (the caller's array is its own again)
    assert out[:n].tolist() == keep.tolist() and int(out[n]) == -7
    t = torch.randn(3, n, device=DEV)
    for v in (t, t.bfloat16(), t.t(), off(t)):
        c = ops.copied(v)
        assert torch.equal(c, v) and (n == 0 or c.data_ptr() != v.data_ptr())


def test_block_table_on_the_device_is_the_hosts():
    make(torch.bfloat16)
    from qserve_amd.serving.cache import PagedCache
    cache = PagedCache([4], num_pages=1400, max_seqs=5, dtype=torch.bfloat16, device=DEV, page=8)
    slots = [cache.admit() for _ in range(5)]
    for step in ([1] * 5, [7, 8, 9, 200, 1], [3840, 8, 0, 3000, 5], [1] * 5, [8] * 5, [8] * 5):       # (one page to more than travel with a launch)
        for s, n in zip(slots, step):
            if n:
                cache.extend(s, n)
        assert torch.equal(cache.block_table().cpu(), cache.table_host)
        for _ in range(3):                                               # (the same places again and again, before they are uploaded)
            cache.release(slots[1])
            cache.extend(slots[0], 9)
            slots[1] = cache.admit()
            cache.extend(slots[1], 17)
        assert torch.equal(cache.block_table().cpu(), cache.table_host)


def close(got, ref, size, dtype):
    """Within half a unit of the storage type's last place (or a rounding that falls the other way) and float sums whose terms are of `size`."""
    return ((got.double() - ref).abs() <= (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -22) * ref.abs() + 2.0 ** -19 * size).all()


# one wave and two, groups of 1024 columns, rows in one trip and in two; parts with and without a scale, the rows of a table, no norm, one and two
@TYPES
@pytest.mark.parametrize("D", [4, 256, 260, 512, 516, 1024, 2052, 3072, 3076, 4100, 5120, 6144, 6148, 8192, 8196])
@pytest.mark.parametrize("parts, norms, table", [(0, 2, True), (1, 1, False), (2, 2, False), (3, 2, False), (3, 0, True)])
def test_scaled_sums(dtype, D, parts, norms, table):
    ops, g, T = make(dtype), torch.Generator().manual_seed(D + parts), 5
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)                                        # noqa: E731
    x, rows, tokens = torch.randn(T, D, generator=g).to(DEV), rnd(9, D), ints([3, 0, 8, 8, 1])
    ps = [(rnd(T, D), None if j == 1 else rnd(D)) for j in range(parts)]
    gains = [torch.randn(D, generator=g).to(DEV) for _ in range(norms)]
    start = rows[tokens.long()].double() if table else x.double()
    terms = [y.double() * (1.0 if f is None else f.double()) for y, f in ps]
    ref = start + sum(terms)
    size = start.abs() + sum(t.abs() for t in terms)
    got, hs = ops.scaled_sum_rms_norms(x, ps, gains, 1e-5, **(dict(tokens=tokens, table=rows) if table else {}))
    assert len(hs) == norms and close(got, ref, size, torch.float32)
    inv = 1.0 / (ref.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt()
    assert all(close(h, ref * inv * w.double(), size * inv * w.double().abs(), dtype) for h, w in zip(hs, gains))


# heads in one round of the workgroup, two, four and more; a head's lanes a power of two and not
@TYPES
@pytest.mark.parametrize("dim", [8, 40, 64, 128, 256])
@pytest.mark.parametrize("extra", [0, 1])
@pytest.mark.parametrize("rounds", [1, 2, 4])
def test_head_norms_by_rounds(dtype, dim, extra, rounds):
    ops, g, T = make(dtype), torch.Generator().manual_seed(dim + rounds), 3
    lanes = 1
    while lanes * 4 < dim:
        lanes *= 2
    G = 2
    H = rounds * (256 // lanes) + extra - G
    if (H + G) * dim * 4 > 64 * 1024:
        pytest.skip("more heads than the launch takes")
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)                                        # noqa: E731
    q, k, v, qw, kw = rnd(T, H * dim), rnd(T, G * dim), rnd(T, G * dim), rnd(dim), rnd(dim)
    rot = dim // 8 * 8 - (4 if dim == 40 else 0)
    rope, pos = torch.randn(T + 2, 2, rot // 2, generator=g).to(DEV), [4, 0, 2]
    batch = StepBatch(tokens=None, seq=None, pos=ints(pos), slot=torch.tensor([2, 0, 1], device=DEV), block_table=None, max_pos=4, n_tokens=T, items=[(i, i, 1) for i in range(T)])
    pool = torch.zeros(G, T, 2 * dim, dtype=dtype, device=DEV)
    qf = ops.qk_norm_rope_prep(q, k, v, H, G, dim, dim, qw, kw, True, 1e-5, rope, rot, 0.5, pool, batch, q_pad=0)

    def ref(u, w):
        u = u.double().view(T, -1, dim)
        n = u / (u.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt() * w.double()
        c, s = (rope[pos, i].double()[:, None] for i in (0, 1))
        a, b = n[..., 0:rot:2].clone(), n[..., 1:rot:2].clone()
        n[..., 0:rot:2], n[..., 1:rot:2] = a * c - b * s, b * c + a * s
        return n
    assert close(qf, ref(q, qw) * 0.5, 16.0, torch.float32)
    rows = pool[:, [2, 0, 1]].transpose(0, 1)
    assert torch.equal(rows[..., :dim], v.view(T, G, dim)) and close(rows[..., dim:], ref(k, kw), 16.0, dtype)


@TYPES
@pytest.mark.parametrize("T", [128, 129, 1023, 1024])
@pytest.mark.parametrize("S, D", [(1, 4), (2, 1028), (3, 64), (4, 1024)])
def test_streams_read_by_number_of_rows(dtype, T, S, D):
    ops, g = make(dtype), torch.Generator().manual_seed(T + D)
    x, w_in = torch.randn(T, S, D, generator=g).to(DEV), torch.randn(S, generator=g).to(DEV)
    w, b = (torch.randn(D, generator=g).to(dtype).to(DEV) for _ in range(2))
    ref = torch.tanh(0.6 * torch.einsum("s,tsd->td", w_in.double(), x.double())) * w.double() + b.double()
    assert close(ops.hc_read(x, w_in, (w, b, 0.6)), ref, 16.0, dtype)


# below 1024 channels one a thread, from there four
@TYPES
@pytest.mark.parametrize("H, dim", [(1, 4), (2, 128), (255, 4), (256, 4), (257, 4), (3, 341)])
@pytest.mark.parametrize("log", [False, True])
def test_decay_by_width(dtype, H, dim, log):
    ops, g, T = make(dtype), torch.Generator().manual_seed(H * dim), 17
    z, b = torch.randn(T, H * dim + 4, generator=g).to(dtype).to(DEV)[:, 4:], torch.randn(H * dim, generator=g).to(dtype).to(DEV)
    a = torch.randn(H, generator=g).to(DEV) if log else None
    u = z.double() + b.double()
    if log:
        power = -a.double().exp().repeat_interleave(dim) * torch.nn.functional.softplus(u)
    else:
        power = -torch.nn.functional.softplus(-u) / 16.0
    # a power of e that carries some units of 2^-24 of itself, exponentials of a few more
    assert ((ops.decay(z, b, a, 16.0, H, dim).double() - power.exp()).abs() <= 2.0 ** -20 * (1.0 + power.abs()) * power.exp() + 1e-30).all()


# The forms of four columns a thread against their statements in 64 bits: rotated pairs, norms of a latent row, sums of streams, embeddings
@TYPES
@pytest.mark.parametrize("T, n", [(1, 4), (3, 64), (65, 260), (2, 2052)])
def test_rows_against_64_bits(dtype, T, n):
    ops, g = make(dtype), torch.Generator().manual_seed(T + n)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)                                        # noqa: E731
    rms = lambda t, w: t.double() / (t.double().pow(2).mean(-1, keepdim=True) + 1e-5).sqrt() * w.double()  # noqa: E731
    pos, slot = torch.randperm(T, generator=g), torch.randperm(2 * T, generator=g)[:T].to(DEV)
    # a latent row: query latent, key-value latent and rotated key with neighbours as pairs
    rot_n = min(n, 64) // 4 * 2
    down, qw, kw, rope = rnd(T, 3 * n + 4), rnd(n), rnd(n), torch.randn(T + 1, 2, rot_n // 2, generator=g).to(DEV)
    pool = torch.zeros(2 * T, 2 * n, dtype=dtype, device=DEV)
    cq = ops.latent_prep(down, 0, n, qw, n + 4, n, kw, n, rot_n, rope, pool, slot, pos.int().to(DEV), 1e-5)
    c, s = (rope[pos, i].double() for i in (0, 1))
    kr = down[:, 2 * n + 4:].double()
    a, b = kr[:, 0:rot_n:2].clone(), kr[:, 1:rot_n:2].clone()
    kr[:, 0:rot_n:2], kr[:, 1:rot_n:2] = a * c - b * s, b * c + a * s
    assert close(cq, rms(down[:, :n], qw), 16.0, dtype)
    assert close(pool[slot][:, :n], rms(down[:, n + 4:2 * n + 4], kw), 16.0, dtype) and close(pool[slot][:, n:], kr, 16.0, dtype)
    # pairs half a head apart, turned back
    o, rope = rnd(T, 3, 2 * n), torch.randn(T, 2, n, generator=g).to(DEV)
    c, s = (rope[pos, i].double()[:, None] for i in (0, 1))
    a, b = o.double()[..., :n], o.double()[..., n:]
    assert close(ops.rotate_heads(o.clone(), rope, pos.int().to(DEV), -1.0), torch.cat([a * c + b * s, b * c - a * s], -1), 16.0, dtype)
    x, w, b, rows = torch.randn(T, 3, n, generator=g).to(DEV), rnd(n), rnd(n), ints(pos.tolist())
    assert close(ops.dyt_sum_rows(x, rows, (w, b, 0.6)), torch.tanh(0.6 * x[rows.long()].double().sum(1)) * w.double() + b.double(), 16.0, dtype)
    table, tokens = rnd(9, n), torch.randint(0, 9, (T,), generator=g).to(DEV)
    h, t = ops.embed(tokens.int(), table)
    assert torch.equal(h, table[tokens].float()) and torch.equal(t, table[tokens])
    streams = ops.embed_streams(tokens.int(), table, 1.7, 3)
    assert close(streams, (1.7 * table[tokens].double())[:, None].expand(T, 3, n), 0.0, torch.float32)


# ... convolutions over time: runs with and without a history, the histories that they leave
@TYPES
@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("runs", [((0, 1), (7, 1), (1, 1)), ((2, 3), (0, 2), (9, 4))])
def test_convolutions_against_64_bits(dtype, taps, runs):
    ops, g = make(dtype), torch.Generator().manual_seed(taps + len(runs))
    T, qc, G, kd, vd = sum(n for _, n in runs), 40, 2, 8, 12
    C, past = qc + G * (kd + vd), taps - 1
    proj, w = torch.randn(T, C + 4, generator=g).to(dtype).to(DEV), torch.randn(taps, C, generator=g).to(DEV)
    hist = torch.randn(2 * len(runs), past, C, generator=g).to(DEV)
    off_, rd, wr, pos, items, at, y, left = [], [], [], [], [], 0, [], hist.double()
    for r, (start, n) in enumerate(runs):
        off_ += range(n)
        rd += [2 * r if start else -1] * n
        wr += [-1] * (n - 1) + [2 * r + 1]
        pos += range(start, start + n)
        items.append((r, at, n))
        seq = torch.cat([hist[2 * r].double() if start else torch.zeros(past, C, device=DEV), proj[at:at + n, :C].double()])
        y.append(sum(seq[j:j + n] * w[j].double() for j in range(taps)))
        left[2 * r + 1] = seq[n:]
        at += n
    y = torch.cat(y)
    batch = StepBatch(tokens=None, seq=None, pos=ints(pos), slot=torch.arange(T, device=DEV), block_table=None, max_pos=max(pos), n_tokens=T, items=items,
                      run_off=ints(off_), state_rd=ints(rd), state_wr=ints(wr))
    h, pool = hist.clone(), torch.zeros(G, T, vd + kd, dtype=dtype, device=DEV)
    q = ops.conv_heads_cache(proj, w, h, batch, qc, G, kd, vd, pool, 0.3, (0.1, 4.0))
    warm = 1.0 + 0.1 * torch.log(((torch.tensor(pos, device=DEV).double() + 1.0) / 4.0).floor() + 1.0)
    assert close(q, 0.3 * y[:, :qc] * warm[:, None], 16.0, dtype) and torch.equal(h.double(), left)
    k, v = y[:, qc:qc + G * kd].view(T, G, kd).transpose(0, 1), y[:, qc + G * kd:].view(T, G, vd).transpose(0, 1)
    assert close(pool[..., :vd], v, 16.0, dtype) and close(pool[..., vd:], k, 16.0, dtype)
    h = hist.clone()
    got, ref = ops.conv_silu_unit(proj, 0, w.t().contiguous(), h, batch, 4, 8), y * torch.sigmoid(y)
    u = ref[:, :32].reshape(-1, 8)
    ref = torch.cat([(u / (u.pow(2).sum(-1, keepdim=True) + 1e-6).sqrt()).view(T, 32), ref[:, 32:]], 1)
    # unit vectors: float products of up to 16 over a length that may be small
    size = torch.cat([(1.0 + 1.0 / (u.pow(2).sum(-1, keepdim=True) + 1e-6).sqrt()).expand_as(u).reshape(T, 32), torch.ones_like(ref[:, 32:])], 1) * 16.0
    assert ((got.double() - ref).abs() <= 2.0 ** -20 * (ref.abs() + size)).all() and torch.equal(h.double(), left)
