"""A step of few sequences through the products that read their weights into registers: the bits of the step without them, also replayed and step after step."""
import pytest
import torch

from qserve_amd import decode as D

pytestmark = pytest.mark.gpu
CFG = dict(D.LLAMA3_8B, layers=3, vocab=512)


@pytest.mark.parametrize("group, inter, heads, kv_heads", [(-1, 14336, 32, 8), (128, 14336, 32, 8), (-1, 11008, 32, 32), (128, 11008, 32, 32), (-1, 4096, 32, 8)])
@pytest.mark.parametrize("batch", [1, 2, 3])
def test_few_sequences(batch, group, inter, heads, kv_heads):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    cfg = dict(CFG, inter=inter, heads=heads, kv_heads=kv_heads)
    kw = dict(group_size=group, int4_kv=True, seed=5)
    eng, ref = D.DecodeEngine(cfg, batch, 70, 8, **kw), D.DecodeEngine(cfg, batch, 70, 8, planes=("o", "down"), **kw)
    assert ("o" in eng.rows) and not ref.rows and ("qkv" in eng.rows) == (batch == 1 or (batch == 2 and kv_heads == 8))
    assert ("gate_up" in eng.rows) == (batch == 1) and ("down" in eng.rows) == (batch == 1 and inter > 8192 and (group == -1 or inter % 512 == 0))
    assert ("attention" in eng.rows) == (batch <= 2)
    for e in (eng, ref):
        e.prefill_cache(70)
        e.tokens.copy_(torch.arange(batch, device="cuda") + 3)
        e.capture()
        e.lengths.fill_(71)
    for step in range(4):
        for e in (eng, ref):
            e.tokens.copy_(torch.arange(batch, device="cuda") * 7 + step)
            e.run()
        torch.cuda.synchronize()
        assert torch.equal(eng.hidden, ref.hidden)
        assert torch.equal(eng.final, ref.final)
