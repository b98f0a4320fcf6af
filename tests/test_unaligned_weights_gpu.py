"""Weights that are views into a larger buffer - a table with gaps between its rows, gains that start on 2 bytes, scales that start on 4 - give what their copies give."""
import pytest
import torch

from qserve_amd import decode as D

pytestmark = pytest.mark.gpu
LINEARS = ("qkv", "o", "gate_up", "down")


def _tensors(lin):
    return {n: getattr(lin, n) for n in ("qweight", "s1_scales", "s1_szeros", "s2_scales", "s2_zeros") if hasattr(lin, n)}


def _shifted(t, by=1):
    flat = torch.empty(t.numel() + by, dtype=t.dtype, device=t.device)
    view = flat[by:].view(t.shape)
    view.copy_(t)
    return view


def _gapped(t):
    wide = torch.zeros((t.size(0), t.size(1) + 8), dtype=t.dtype, device=t.device)
    wide[:, :t.size(1)] = t
    return wide[:, :t.size(1)]


FORMS = {
    "table with gaps": lambda w: w.update(embed=_gapped(w["embed"])),
    "table": lambda w: w.update(embed=_shifted(w["embed"])),
    "last gain": lambda w: w.update(norm=_shifted(w["norm"])),
    "first gain": lambda w: w["layers"][0].update(ln1=_shifted(w["layers"][0]["ln1"])),
    "other gains": lambda w: w["layers"][1].update(ln1=_shifted(w["layers"][1]["ln1"]), ln2=_shifted(w["layers"][1]["ln2"])),
    "last scales": lambda w: w["layers"][-1]["down"].update({n: _shifted(t, 2) for n, t in w["layers"][-1]["down"].items() if n.startswith("s1_")}),
}


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("batch, group", [(1, -1), (1, 128), (2, -1), (5, -1), (24, 128)])
def test_views(batch, group, form):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    cfg = dict(D.LLAMA3_8B, layers=2, vocab=512, inter=11008)
    kw = dict(group_size=group, int4_kv=True, seed=5)
    ref = D.DecodeEngine(cfg, batch, 40, 4, **kw)
    weights = dict(layers=[dict(ln1=L["ln1"], ln2=L["ln2"], **{n: _tensors(L[n]) for n in LINEARS}) for L in ref.layers], norm=ref.norm_w, embed=ref.embed, lm_head=ref.lm_head)
    FORMS[form](weights)
    eng = D.DecodeEngine(cfg, batch, 40, 4, weights=weights, **kw)
    tokens = torch.randint(0, 512, (batch * 40,), device="cuda", generator=torch.Generator(device="cuda").manual_seed(batch))
    for e in (eng, ref):
        e.prefill(40, tokens)
    assert torch.equal(eng.hidden, ref.hidden) and torch.equal(eng.final, ref.final) and torch.equal(eng.lengths, ref.lengths)
    for _ in range(2):
        for e in (eng, ref):
            e.step()
            e.lengths += 1
        assert torch.equal(eng.hidden, ref.hidden) and torch.equal(eng.final, ref.final) and torch.equal(eng.tokens, ref.tokens)
