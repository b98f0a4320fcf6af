"""Which prompts attend over written-out keys and values: the rule alone, on the host."""
import pytest
import torch

from qserve_amd.layers.ops import HipOps
from qserve_amd.serving.engine import StepBatch


def _batch(runs):
    """runs: (first position, tokens)."""
    at, items = 0, []
    for b, (_, n) in enumerate(runs):
        items.append((b, at, n))
        at += n
    return StepBatch(tokens=None, seq=None, pos=torch.zeros(at, dtype=torch.int32), slot=None, block_table=None, max_pos=max(s + n for s, n in runs) - 1, n_tokens=at,
                     items=items, starts=[s for s, _ in runs])


def _plan(runs, H=16, rot=64, rank=512, window=None, **more):
    return HipOps(torch.bfloat16).latent_prompt_plan(_batch(runs), window, H, 128, rot, 128, rank, 0.1, **more)


def test_a_pool_off_the_alignment_keeps_its_rows():
    rows = torch.zeros(64 * 576 + 8, dtype=torch.bfloat16)
    start = -rows.data_ptr() // 2 % 8                                   # (the first element on 16 bytes)
    for off in range(8):
        pool = rows[(start + off) % 8:][:64 * 576].view(64, 576)
        assert pool.data_ptr() % 16 == 2 * off
        assert (_plan([(0, 100)], pool=pool) is not None) == (off == 0)
    assert _plan([(0, 100)]) is not None


def test_products_that_torch_would_change_keep_the_rows():
    w = lambda **k: torch.zeros(8, 8, **dict(dict(dtype=torch.bfloat16), **k))                     # noqa: E731
    assert _plan([(0, 100)], weights=(w(), w())) is not None
    assert _plan([(0, 100)], weights=(w(), w(dtype=torch.float16))) is None
    assert _plan([(0, 100)], weights=(w(requires_grad=True), w())) is None
    with torch.no_grad():
        assert _plan([(0, 100)], weights=(w(requires_grad=True), w())) is not None
    torch.set_autocast_enabled("cuda", True)
    try:
        assert _plan([(0, 100)], weights=(w(), w())) is None
    finally:
        torch.set_autocast_enabled("cuda", False)


# 512 bytes a key and head written out against 6 rank + 4 rot_dim bytes a token and head on the rows, beyond 256 MB
@pytest.mark.parametrize("runs, H, rot, rank, taken", [([(0, 8192)], 128, 64, 512, True), ([(24576, 8192)], 128, 64, 512, True), ([(8192, 8192)], 64, 64, 64, False),
                                                       ([(0, 8192)], 64, 0, 64, True), ([(0, 8200)], 64, 0, 64, False), ([(0, 4000)], 64, 0, 64, True),
                                                       ([(4000, 4000)], 128, 0, 128, False), ([(4000, 4000)], 128, 0, 176, True)])
def test_what_is_written_out_is_bounded(runs, H, rot, rank, taken):
    plan = _plan(runs, H=H, rot=rot, rank=rank)
    assert (plan is not None) == taken
    assert plan is None or plan[2] * H * 512 <= max(1 << 28, sum(n for _, n in runs) * H * (6 * rank + 4 * rot))


# workgroups (128 tokens and a head each) against the keys that a run's tokens see on average
@pytest.mark.parametrize("runs, H, window, taken", [([(0, 4000)], 1, None, False), ([(0, 300)], 2, None, False), ([(0, 65)], 3, None, True), ([(0, 2000)], 3, None, True),
                                                    ([(512, 512)], 3, None, True), ([(775, 500)], 3, None, False), ([(774, 500)], 3, None, True), ([(3000, 1000)], 3, None, False),
                                                    ([(3000, 1000)], 6, None, True), ([(1500, 500)] * 2, 4, None, False), ([(1500, 500)] * 3, 4, None, True),
                                                    ([(3000, 1000)], 3, 1024, True), ([(3000, 1000)], 3, 1025, False)])
def test_long_walks_need_workgroups(runs, H, window, taken):
    assert (_plan(runs, H=H, window=window) is not None) == taken
