"""The recurrent mixers' row kernels at the edges of their sizes, against the plain PyTorch statements in float32."""
from types import SimpleNamespace

import pytest
import torch

from qserve_amd.layers.ops import HipOps, TorchOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _gen(seed):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.Generator(device=DEV).manual_seed(seed)


def _batch(counts, starts):
    """Runs of counts[i] tokens of sequence i from position starts[i]; states in rows 0 .. n - 1 (old) and n .. 2 n - 1 (new)."""
    n, i32 = len(counts), lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)             # noqa: E731
    items, first = [], 0
    for i, c in enumerate(counts):
        items.append((i, first, c))
        first += c
    pos = [s + k for c, s in zip(counts, starts) for k in range(c)]
    off = [k for c in counts for k in range(c)]
    rd = [i if starts[i] else -1 for i, c in enumerate(counts) for _ in range(c)]
    wr = [n + i if k == c - 1 else -1 for i, c in enumerate(counts) for k in range(c)]
    runs = i32([[s, f, c, starts[s]] for s, f, c in items])
    return SimpleNamespace(items=items, pos=i32(pos), run_off=i32(off), state_rd=i32(rd), state_wr=i32(wr), runs=lambda: runs, max_pos=max(pos),
                           slot=torch.arange(first, dtype=torch.int64, device=DEV).flip(0).contiguous())


def _rounded(dtype, v):
    return (2.0 ** -8 if dtype == torch.bfloat16 else 0.0) * v.abs()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("C, taps, n_unit, dim", [(2560, 4, 8, 64), (1028, 4, 1, 4), (36, 3, 2, 16), (1536, 2, 6, 256), (520, 4, 0, 64), (24, 4, 3, 6), (30, 3, 1, 8),
                                                  (40, 5, 2, 8), (16, 1, 2, 8)])
def test_convolution_and_unit_vectors(C, taps, n_unit, dim, dtype):
    g = _gen(C)
    b = _batch([1, 2, 7, 1, 3], [9, 0, 4, 0, 1])
    T, n = b.pos.numel(), 5
    proj = torch.randn(T, C + 8, device=DEV, generator=g).to(dtype)
    w, hist = torch.randn(C, taps, device=DEV, generator=g), torch.randn(2 * n, max(taps - 1, 1), C, device=DEV, generator=g).to(dtype).float()
    for act in ("silu", "none"):
        h1, h2 = hist.clone(), hist.clone()
        y = HipOps(dtype).conv_silu_unit(proj, 4, w, h1, b, n_unit, dim, act)
        ref = TorchOps(dtype).conv_silu_unit(proj, 4, w, h2, b, n_unit, dim, act)
        # values below 2^5, some ten float roundings on either side; a unit vector divides by a length above 2^-2
        assert ((y - ref).abs() <= 2.0 ** -24 * 2.0 ** 5 * 20 * 4).all() and torch.equal(h1, h2)


@pytest.mark.parametrize("kind", ["silu", "sigmoid"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T, H, dv, extra, per_head", [(1, 16, 128, 0, False), (17, 5, 4, 0, True), (3, 3, 256, 4, True), (5, 7, 64, 0, True), (2, 2, 96, 0, False),
                                                       (4, 3, 16, 1, False), (3, 2, 512, 0, True),
                                                       # heads of several tokens in a workgroup, the last one part empty
                                                       (37, 1, 64, 0, True), (300, 1, 4, 4, False), (9, 3, 256, 0, True)])
def test_read_out_norm_and_gate(T, H, dv, extra, per_head, dtype, kind):
    g = _gen(T + dv)
    o, gate = torch.randn(T, H, dv + extra, device=DEV, generator=g), torch.randn(T, H * dv + 8, device=DEV, generator=g).to(dtype)[:, 4:4 + H * dv]
    w = torch.randn(H * dv if per_head else dv, device=DEV, generator=g).to(dtype)
    den = torch.randn(T, H, device=DEV, generator=g) if extra else None
    y = HipOps(dtype).head_rms_gate(o, w, gate, kind, 1e-5, vdim=dv, den_m=den).float()
    ref = TorchOps(torch.float32).head_rms_gate(o, w, gate, kind, 1e-5, vdim=dv, den_m=den)
    # sums of dv squares and some ten float roundings on either side (the divisor's: relative to a denominator above 2^-10), one rounding to the type
    assert ((y - ref).abs() <= 2.0 ** -22 * (dv + 32) * ref.abs() + _rounded(dtype, ref) + 1e-30).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H, G, dim, vdim, rot", [(16, 4, 128, 128, 64), (3, 1, 8, 8, 8), (2, 2, 36, 24, 16), (4, 2, 20, 16, 0), (4, 2, 20, 12, 12), (2, 1, 6, 10, 4)])
def test_attention_rows(H, G, dim, vdim, rot, dtype):
    g = _gen(dim)
    b = _batch([1, 4, 6], [3, 0, 2])
    T, off = b.pos.numel(), 4
    proj = torch.randn(T, off + (H + G) * dim + G * vdim + (-(off + (H + G) * dim + G * vdim)) % 4, device=DEV, generator=g).to(dtype)

    def table(n):
        a = torch.rand(16, max(n // 2, 1), device=DEV, generator=g) * 6.28
        return torch.stack([a.cos(), a.sin()], 1)[..., :n // 2].contiguous()

    rk, rv = table(rot), table(vdim)
    p1 = torch.zeros(G, T + 2, vdim + dim, device=DEV, dtype=dtype)
    p2 = p1.clone()
    args = (proj, off, off + H * dim, off + (H + G) * dim, H, G, dim, vdim, rot, rk, rv, 0.25)
    qf, ref = HipOps(dtype).attention_prep(*args, p1, b), TorchOps(torch.float32).attention_prep(*args, p2.float(), b)
    p3 = p2.float()
    TorchOps(torch.float32).attention_prep(*args, p3, b)
    # two float products of values below 2^3 and their sum, on either side; the rows rounded to the type
    assert ((qf.reshape(ref.shape) - ref).abs() <= 2.0 ** -19).all()
    assert ((p1.float() - p3).abs() <= 2.0 ** -19 + _rounded(dtype, p3)).all()


@pytest.mark.parametrize("delta", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H, G, dim, vdim, v_cols", [(16, 4, 64, 128, 128), (2, 1, 8, 4, 4), (3, 3, 72, 132, 129), (2, 2, 128, 260, 260), (2, 1, 136, 64, 63),
                                                     (1, 1, 256, 128, 128), (2, 1, 264, 8, 8), (2, 1, 20, 6, 6)])
def test_one_token_of_the_recurrence(H, G, dim, vdim, v_cols, dtype, delta):
    g = _gen(dim + vdim)
    b = _batch([1, 1, 1], [5, 0, 2])
    T = 3
    unit = lambda *s: torch.nn.functional.normalize(torch.randn(*s, device=DEV, generator=g), dim=-1)       # noqa: E731
    q, k = unit(T, G, dim).view(T, -1).to(dtype), unit(T, G, dim).view(T, -1).to(dtype)
    v = torch.randn(T, H * v_cols, device=DEV, generator=g).to(dtype)
    beta = torch.randn(T, H, device=DEV, generator=g).to(dtype) if delta else None
    state = torch.randn(4, H, dim, vdim, device=DEV, generator=g).clamp(-4, 4)
    for decay in (torch.rand(T, H * dim, device=DEV, generator=g), torch.rand(T, H, device=DEV, generator=g), torch.rand(H, device=DEV, generator=g)):
        for ks in (None, torch.rand(T, H, device=DEV, generator=g)):
            s1, s2 = state.clone(), state.clone()
            o = HipOps(dtype).recurrent_scan(q, k, v, decay, beta, s1, b, H, G, dim, vdim, 0.5, ks, v_cols)
            ref = TorchOps(dtype).recurrent_scan(q, k, v, decay, beta, s2, b, H, G, dim, vdim, 0.5, ks, v_cols)
            # sums of dim products of |S| <= 8 with a unit vector (at most 8 sqrt(dim) in absolute values), twice in a row, on either side
            bound = 4 * 2.0 ** -24 * (dim + 8) * 8 * (dim ** 0.5 + 4)
            assert ((o - ref).abs() <= bound).all() and ((s1 - s2).abs() <= bound).all()


@pytest.mark.parametrize("delta", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("counts, H, G, dim, vdim, v_cols", [((1, 15, 16, 17, 33), 2, 1, 64, 128, 128), ((31, 32), 130, 65, 64, 132, 128), ((5, 48), 3, 3, 36, 4, 4),
                                                             ((16, 49), 2, 1, 68, 36, 32), ((2, 40), 128, 64, 128, 64, 64), ((20, 3), 2, 2, 128, 68, 68),
                                                             ((18, 2), 2, 2, 32, 64, 64), ((17, 2), 2, 2, 132, 12, 12), ((17, 2), 2, 2, 34, 10, 9),
                                                             # many workgroups: no more columns than one per lane, narrow states in short and in longer runs
                                                             ((17, 2), 160, 80, 64, 24, 24), ((3, 2), 512, 256, 64, 16, 16), ((9, 2), 512, 256, 40, 16, 16),
                                                             ((8, 1), 512, 512, 68, 8, 8), ((2, 3), 512, 512, 72, 12, 12)])
def test_runs_of_the_recurrence(counts, H, G, dim, vdim, v_cols, dtype, delta):
    """Full chunks of 16 tokens and what is left of them, one and two columns per lane, rows and columns that do not fill a workgroup."""
    g = _gen(dim + vdim)
    b = _batch(list(counts), [5, 0, 2, 0, 1][:len(counts)])
    T = sum(counts)
    unit = lambda *s: torch.nn.functional.normalize(torch.randn(*s, device=DEV, generator=g), dim=-1)       # noqa: E731
    q, k = unit(T, G, dim).view(T, -1).to(dtype), unit(T, G, dim).view(T, -1).to(dtype)
    v = torch.randn(T, H * v_cols, device=DEV, generator=g).to(dtype)
    beta = torch.randn(T, H, device=DEV, generator=g).to(dtype) if delta else None
    state = torch.randn(6, H, dim, vdim, device=DEV, generator=g).clamp(-4, 4)
    for i, shape in enumerate(((T, H * dim), (T, H), (H,))):
        decay, ks = torch.rand(*shape, device=DEV, generator=g) * 0.9, torch.rand(T, H, device=DEV, generator=g) if i == 1 else None
        s1, s2 = state.clone(), state.clone()
        o = HipOps(dtype).recurrent_scan(q, k, v, decay, beta, s1, b, H, G, dim, vdim, 0.5, ks, v_cols)
        ref = TorchOps(dtype).recurrent_scan(q, k, v, decay, beta, s2, b, H, G, dim, vdim, 0.5, ks, v_cols)
        # a token's own error as above (|S| <= 64: inputs below 8, decays below 0.9), carried on by decays of 0.9 at most: ten times it
        bound = 10 * 4 * 2.0 ** -24 * (dim + 8) * 64 * (dim ** 0.5 + 4)
        assert ((o - ref).abs() <= bound).all() and ((s1 - s2).abs() <= bound).all()
        # and element by element against what rounding of that kind does on average (its square root): a wrong row or column stands out by far
        assert ((o - ref).norm() / ref.norm()).item() < 2.0 ** -24 * dim * 16 and ((s1 - s2).norm() / s2.norm()).item() < 2.0 ** -24 * dim * 16


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("S, D", [(2, 4), (2, 1020), (3, 1028), (2, 2048), (4, 2052), (2, 6)])
def test_streams_read_and_written(S, D, dtype):
    g = _gen(S + D)
    b = _batch([1, 3, 1], [4, 0, 0])
    T, n = 5, 3
    x, y = torch.randn(T, S, D, device=DEV, generator=g), torch.randn(T, D, device=DEV, generator=g).to(dtype)
    norm = (torch.randn(D, device=DEV, generator=g).to(dtype), torch.randn(D, device=DEV, generator=g).to(dtype), 0.7)
    w_in, mix, w_out = (torch.rand(*s, device=DEV, generator=g) for s in ((S,), (S, S), (S,)))
    shift, prev = torch.rand(D, device=DEV, generator=g).to(dtype), torch.randn(2 * n, D, device=DEV, generator=g)
    hip, ref = HipOps(dtype), TorchOps(torch.float32)
    p1, p2 = prev.clone(), prev.clone()
    tol = 2.0 ** -24 * 64 * 16                                                # (values below 2^6, some ten float roundings on either side)
    for got, want in ((hip.hc_read(x, w_in, norm), ref.hc_read(x, w_in, norm)), (hip.hc_read(x, w_in, norm, shift, b, p1), ref.hc_read(x, w_in, norm, shift, b, p2))):
        assert ((got.float() - want).abs() <= tol + _rounded(dtype, want)).all()
    assert ((p1 - p2).abs() <= tol).all()
    x1, x2 = x.clone(), x.clone()
    got, want = hip.hc_write(x1, y, mix, w_out, (w_in, norm)), ref.hc_write(x2, y, mix, w_out, (w_in, norm))
    assert ((x1 - x2).abs() <= tol).all() and ((got.float() - want).abs() <= tol + _rounded(dtype, want)).all()


@pytest.mark.parametrize("T", [512, 513, 1023, 1024])
def test_streams_at_the_lines_of_the_split(T):
    """A token's row over several workgroups and in one, at both kernels' lines."""
    g = _gen(T)
    S, D = 2, 2052
    x, y, w_in, mix, w_out = (torch.randn(*s, device=DEV, generator=g) for s in ((T, S, D), (T, D), (S,), (S, S), (S,)))
    norm = (torch.randn(D, device=DEV, generator=g), torch.randn(D, device=DEV, generator=g), 0.7)
    hip, ref = HipOps(torch.float32), TorchOps(torch.float32)
    tol = 2.0 ** -24 * 64 * 16                                                # (values below 2^6, some ten float roundings on either side)
    assert ((hip.hc_read(x, w_in, norm) - ref.hc_read(x, w_in, norm)).abs() <= tol).all()
    x1, x2 = x.clone(), x.clone()
    got, want = hip.hc_write(x1, y, mix, w_out, (w_in, norm)), ref.hc_write(x2, y, mix, w_out, (w_in, norm))
    assert ((x1 - x2).abs() <= tol).all() and ((got - want).abs() <= tol).all()


@pytest.mark.parametrize("C", [96, 252, 256])
@pytest.mark.parametrize("T", [1023, 1024])
def test_convolution_of_few_channels(T, C):
    g = _gen(T + C)
    b = _batch([5, T - 5], [9, 0])
    proj, w, hist = torch.randn(T, C, device=DEV, generator=g), torch.randn(C, 4, device=DEV, generator=g), torch.randn(4, 3, C, device=DEV, generator=g)
    h1, h2 = hist.clone(), hist.clone()
    y, ref = HipOps(torch.float32).conv_silu_unit(proj, 0, w, h1, b, 3, 4), TorchOps(torch.float32).conv_silu_unit(proj, 0, w, h2, b, 3, 4)
    # values below 2^5, some ten float roundings on either side; a unit vector divides by a length above 2^-2
    assert ((y - ref).abs() <= 2.0 ** -24 * 2.0 ** 5 * 20 * 4).all() and torch.equal(h1, h2)
