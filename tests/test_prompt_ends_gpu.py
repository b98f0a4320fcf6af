"""The first and the last launches of a prompt phase: the bits of the operations they replace."""
import pytest
import torch

from qserve_amd import decode as D
from qserve_amd import fused

pytestmark = pytest.mark.gpu


def _half(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g).half()


def _gen(seed):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.Generator(device="cuda").manual_seed(seed)


@pytest.mark.parametrize("batch, tokens", [(1, 1), (3, 1), (1, 255), (2, 128), (7, 37), (300, 1), (5, 20000)])
def test_layout(batch, tokens):
    _gen(0)
    from qserve_backend import fused_attention
    seq, cu, pad = fused.prompt_layout(batch, tokens, torch.device("cuda"))
    assert seq.tolist() == [tokens] * batch and cu.tolist() == [b * tokens for b in range(batch + 1)]
    assert torch.equal(pad, fused_attention.compute_padding_offsets(cu, tokens, batch * tokens))


@pytest.mark.parametrize("with_sum", [True, False])
@pytest.mark.parametrize("T, hid", [(1, 4096), (37, 4096), (5, 2048), (3, 8192), (4, 5120), (2, 264), (3, 8)])
def test_embedding_and_first_norm(T, hid, with_sum):
    from qserve_backend import layernorm_ops
    g = _gen(T + hid)
    table, w, tokens = _half(g, 50, hid), _half(g, hid).abs(), torch.randint(0, 50, (T,), device="cuda", generator=g)
    tokens[0], tokens[-1] = 0, 49
    ref = torch.index_select(table, 0, tokens)
    outs = [(torch.empty((T, hid), dtype=torch.int8, device="cuda"), *(torch.zeros(T, dtype=torch.float16, device="cuda") for _ in range(2))) for _ in range(2)]
    (q, sc, total), (q1, sc1, total1) = outs
    if with_sum:
        layernorm_ops.rms_norm_general_fuse_sum(q, ref, w, total, sc, 1e-5, True)
    else:
        layernorm_ops.rms_norm_general(q, ref, w, sc, 1e-5, True)
    h = torch.empty_like(ref)
    fused.embed_rms_norm_general(q1, h, table, tokens, w, sc1, 1e-5, total1 if with_sum else None)
    assert torch.equal(h, ref) and torch.equal(q, q1) and torch.equal(sc, sc1) and torch.equal(total, total1)


def test_a_token_outside_the_table():
    g = _gen(3)
    table, w, tokens = _half(g, 50, 256), _half(g, 256), torch.tensor([50, 3, -1], device="cuda")
    h, q, sc = torch.empty((3, 256), dtype=torch.float16, device="cuda"), torch.empty((3, 256), dtype=torch.int8, device="cuda"), torch.empty(3, dtype=torch.float16, device="cuda")
    fused.embed_rms_norm_general(q, h, table, tokens, w, sc, 1e-5)
    assert torch.equal(h[1], table[3]) and h[::2].isnan().all() and sc[::2].isnan().all()


@pytest.mark.parametrize("batch, tokens, hid", [(1, 1, 4096), (8, 33, 4096), (3, 5, 2048), (2, 3, 8192), (2, 2, 5120), (4, 3, 264), (1, 2, 8)])
def test_last_rows_and_norm(batch, tokens, hid):
    from qserve_backend import layernorm_ops
    g = _gen(batch + hid)
    h, delta, w = _half(g, batch * tokens, hid), _half(g, batch * tokens, hid), _half(g, hid).abs()
    out, moved, ref = (torch.empty((batch, hid), dtype=torch.float16, device="cuda") for _ in range(3))
    lengths = torch.zeros(batch, dtype=torch.int32, device="cuda")
    fused.last_rows_rms_norm(out, h, moved, delta, w, 1e-5, tokens, lengths)
    rows = (h + delta)[tokens - 1::tokens].contiguous()
    layernorm_ops.rms_norm(ref, rows, w, 1e-5)
    assert torch.equal(moved, rows) and lengths.tolist() == [tokens + 1] * batch
    assert torch.equal(out, ref)


@pytest.mark.parametrize("group, int4_kv", [(-1, True), (128, False)])
def test_prompt_phase(group, int4_kv):
    g = _gen(5)
    cfg = dict(D.LLAMA3_8B, layers=2, vocab=512)
    kw = dict(group_size=group, int4_kv=int4_kv, seed=5)
    eng, ref = D.DecodeEngine(cfg, 3, 70, 4, **kw), D.DecodeEngine(cfg, 3, 70, 4, **kw)
    tokens = torch.randint(0, 512, (3 * 70,), device="cuda", generator=g)
    eng.prefill(70, tokens)
    ref.prefill(70, tokens.to(torch.int32))             # (torch's lookup: the general path)
    assert torch.equal(eng.hidden, ref.hidden) and torch.equal(eng.lengths, ref.lengths)
    assert torch.equal(eng.final, ref.final)


def test_an_engine_without_layers():
    """Embedding, norm and head alone: no layer's norm reads the table on the way."""
    from qserve_backend import layernorm_ops
    g = _gen(7)
    cfg = dict(D.LLAMA3_8B, layers=0, vocab=512)
    eng = D.DecodeEngine(cfg, 3, 70, 4, seed=5)
    tokens = torch.randint(0, 512, (3 * 70,), device="cuda", generator=g)
    eng.prefill(70, tokens)
    rows = eng.embed[tokens.view(3, 70)[:, -1]]
    ref = torch.empty_like(rows)
    layernorm_ops.rms_norm(ref, rows, eng.norm_w, cfg["eps"])
    assert torch.equal(eng.hidden, rows) and torch.equal(eng.final, ref) and eng.lengths.tolist() == [71] * 3
    logits = torch.matmul(ref, eng.lm_head.t())
    assert torch.equal(logits.gather(1, eng.tokens[:, None])[:, 0], logits.amax(1))
