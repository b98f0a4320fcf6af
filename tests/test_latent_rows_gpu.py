"""Attention over plain cache rows of exact sizes: tile edges, windows, key splits and rows nobody wrote, against float64."""
import math

import pytest
import torch

from qserve_amd.layers.ops import make_ops
from qserve_amd.serving.engine import StepBatch

pytestmark = pytest.mark.gpu


# row, rank, heads, pools, first query element; runs: (context, new tokens)
@pytest.mark.parametrize("R, rank, H, G, q_first", [(576, 512, 16, 1, 0), (512, 512, 20, 1, 0), (576, 512, 3, 1, 0), (256, 128, 12, 3, 128), (256, 128, 34, 2, 0)])
@pytest.mark.parametrize("runs, window, splits", [(((1, 1), (33, 33)), None, None), (((64, 7), (65, 1), (200, 130)), None, 1), (((300, 1), (31, 1), (96, 1)), None, 5),
                                                  (((150, 150), (129, 40)), 37, None), (((700, 9),), 64, 3),
                                                  # one token each: rounds of 64 keys, halves of 32
                                                  (tuple((c, 1) for c in (1, 31, 32, 33, 64, 65, 96, 97, 128, 129, 200)), None, 1),
                                                  (tuple((c, 1) for c in (2, 64, 100, 193)), None, 2), (((700, 1), (65, 1), (3, 1)), 64, 3),
                                                  (((300, 1), (40, 1)), 37, 1), (((321, 1), (450, 1), (5, 1)), None, 1), (((1000, 1),), None, 16), (((1200, 1), (63, 1)), None, None)])
def test_plain_rows(R, rank, H, G, q_first, runs, window, splits):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    dev = torch.device("cuda:0")
    ops = make_ops("hip", torch.bfloat16, dev)
    assert ops.L.qsv_latent_rows_ok(rank, R, 64, ops.code)
    g = torch.Generator().manual_seed(R + H + len(runs))
    pages = sum((c + 63) // 64 for c, _ in runs)
    order = torch.randperm(pages + 1, generator=g).tolist()
    table = torch.full((len(runs), pages), order.pop(), dtype=torch.int32)           # (unused entries: a page of nothing)
    pool = torch.full((G, (pages + 1) * 64, R), float("nan"))                        # rows that nobody wrote must not reach a result
    keys, q, seq, pos, items, at = [], [], [], [], [], 0
    for b, (ctx, n) in enumerate(runs):
        rows = torch.randn(ctx, G, R, generator=g).bfloat16()
        for i in range((ctx + 63) // 64):
            table[b, i] = order.pop()
            part = rows[64 * i:64 * i + 64]
            pool[:, table[b, i] * 64:table[b, i] * 64 + part.size(0)] = part.transpose(0, 1).float()
        keys.append(rows.double())
        q.append(torch.randn(n, H, R, generator=g) * (1.5 / math.sqrt(R - q_first)))
        seq += [b] * n
        pos += range(ctx - n, ctx)
        items.append((b, at, n))
        at += n
    q = torch.cat(q)
    q[..., :q_first] = 0
    pool = (pool if G > 1 else pool[0]).bfloat16()
    batch = StepBatch(tokens=None, seq=torch.tensor(seq, dtype=torch.int32, device=dev), pos=torch.tensor(pos, dtype=torch.int32, device=dev), slot=None,
                      block_table=table.to(dev), max_pos=max(pos), n_tokens=at, items=items)
    out = ops.latent_attention(q.to(dev), pool.to(dev), batch, window, rank, 64, key_splits=splits, q_first=q_first).double().cpu()
    qr, per = q.bfloat16().double(), H // G                                          # (queries enter the products as bfloat16)
    for b, first, n in items:
        for i in range(n):
            p = pos[first + i]
            lo = max(0, p - window + 1) if window else 0
            for h in range(H):
                k = keys[b][lo:p + 1, h // per]
                w = torch.softmax(k @ qr[first + i, h], 0)
                ref = w @ k[:, :rank]
                # weights enter the second product as bfloat16 (relative 2^-9 each, independent), the result is stored as bfloat16
                bound = 2.0 ** -8 * ref.abs() + 6 * 2.0 ** -9 * ((w * w) @ (k[:, :rank] ** 2)).sqrt() + 1e-5
                err = (out[first + i, h] - ref).abs()
                assert (err <= bound).all(), (b, i, h, (err / bound).max())
