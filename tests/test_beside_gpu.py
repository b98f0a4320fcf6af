"""Expert products that ride along in another launch of a decoding step (PendingExperts): the same bits as launches of their own."""
import pytest
import torch

from qserve_amd.layers.ops import make_ops
from qserve_amd.serving.cache import PagedCache
from qserve_amd.serving.engine import StepBatch

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16


def _cache(g, lengths, G, R):
    """Sequences of these lengths over one pool of rows, pages out of order; -> their last tokens as one batch."""
    pages = sum((n + 63) // 64 for n in lengths)
    cache = PagedCache([(G, R)], pages + 2, len(lengths), BF, DEV)
    cache.free_pages = torch.randperm(pages + 2, generator=g).tolist()
    cache.pools[0].normal_()
    slots = [cache.admit() for _ in lengths]
    for s, n in zip(slots, lengths):
        cache.extend(s, n)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)                               # noqa: E731
    n = len(lengths)
    return cache.pools[0], StepBatch(tokens=i32([0] * n), seq=i32(slots), pos=i32([v - 1 for v in lengths]), slot=None, block_table=cache.block_table(),
                                     max_pos=max(lengths) - 1, n_tokens=n, items=[(s, i, 1) for i, s in enumerate(slots)],
                                     _single=i32([[s, i, 1] for i, s in enumerate(slots)]).view(n, 3))


def _experts(g, ops, T, E, top, D, ff, shared, weigh="input"):
    mat = lambda *s: (torch.randn(*s, generator=g) / s[-1] ** 0.5).to(BF).to(DEV)                # noqa: E731
    h, up, down = mat(T, D) * D ** 0.5, mat(E, 2 * ff, D), mat(E, D, ff)
    idx = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(T)]).to(torch.int32).to(DEV)
    sh = (mat(2 * ff, D), mat(D, ff)) if shared else (None, None)
    wt = torch.rand(T, top, generator=g).to(DEV)
    return lambda: ops.moe_experts_pending(h, up, down, idx, wt, *sh, weigh=weigh)


def _dense(results):
    return [results[0].ys] + list(results[1:])


# both kinds of maps, one to 16 heads per pool, tokens up to a step's shared limit, cut keys, lengths at the borders of key blocks and pages
@pytest.mark.parametrize("maps, dim, vdim, H, G", [(2, 64, 128, 16, 4), (1, 128, 128, 16, 4), (2, 32, 64, 3, 3), (2, 96, 96, 8, 1), (2, 16, 32, 32, 2), (1, 64, 64, 6, 2)])
@pytest.mark.parametrize("lengths, splits", [((1,), 1), ((333,), 1), ((700,), 3), ((32, 33, 64, 65, 1), 1), (tuple(range(20, 84)), 1), ((300, 17, 511), 2)])
def test_attention_and_output_product_take_experts_along(maps, dim, vdim, H, G, lengths, splits):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    g = torch.Generator().manual_seed(H + len(lengths))
    ops, T, D = make_ops("hip", BF, DEV), len(lengths), 256
    assert ops.L.qsv_maps_beside_ok(dim, vdim, maps, H // G)
    pool, batch = _cache(g, lengths, G, vdim + maps * dim)
    q = (torch.randn(T, H * maps * dim, generator=g) / dim ** 0.5).to(BF).to(DEV)
    gate = torch.randn(T, H * vdim + 8, generator=g).to(BF).to(DEV)[:, 8:]
    w = (torch.randn(D, H * vdim, generator=g) / 16).to(BF).to(DEV)
    fresh = _experts(g, ops, T, 8, 2, D, 72, shared=len(lengths) % 2 == 1)

    def run(beside):
        kw = dict(key_splits=splits, beside=beside)
        o = (ops.diff_attention(q, pool, batch, H, dim, vdim, 0.4, 0.8, 1e-5, gate, 64, **kw) if maps == 2
             else ops.single_map_attention(q, pool, batch, H, dim, vdim, 64, **kw))
        return [o, ops.linear(o, w, beside)]

    apart, alone = run(None), fresh()
    ref = apart + _dense(alone.results())
    riding = fresh()
    out = run(riding)
    assert riding.made == 2                                                                      # both launches were taken
    assert all(torch.equal(a, b) for a, b in zip(ref, out + _dense(riding.results())))


def test_what_is_not_taken_is_made_in_order():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    g = torch.Generator().manual_seed(3)
    ops = make_ops("hip", BF, DEV)
    fresh = _experts(g, ops, 5, 8, 2, 128, 64, shared=True, weigh="output")
    x, w = torch.randn(5, 128, generator=g).to(BF).to(DEV), torch.randn(256, 128, generator=g).to(BF).to(DEV)
    ref, y = _dense(fresh().results()), ops.linear(x, w)
    p = fresh()
    assert torch.equal(ops.linear(x, w, p), y) and p.made == 2                                   # the second product took the first one's launch with it
    assert all(torch.equal(a, b) for a, b in zip(ref, _dense(p.results())))
    p = fresh()
    with torch.cuda.stream(torch.cuda.Stream()):
        assert p.take(0) is None and p.made == 0                                                 # (another stream's)
    assert all(torch.equal(a, b) for a, b in zip(ref, _dense(p.results()))) and p.take(1) is None
