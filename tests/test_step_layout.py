"""The host side of a step: the tokens that `Engine.execute` takes and the arrays that a step's batch is laid out in."""
import numpy as np
import pytest
import torch

from qserve_amd.serving.cache import CacheFull, PagedCache, StateSpec
from qserve_amd.serving.engine import Engine


class _Model:
    vocab = 100


def _engine():
    e = object.__new__(Engine)
    e.model = _Model()
    return e


class _OnAnotherDevice:
    """A token as a 0-dim tensor on the GPU gives it: int() works, numpy's conversion raises."""

    def __init__(self, v):
        self.v = v

    def __int__(self):
        return self.v

    def __array__(self, *args, **kwargs):
        raise TypeError("can't convert cuda:0 device type tensor to numpy")


@pytest.mark.parametrize("tokens", [[3, 99, 0], (3, 99, 0), [_OnAnotherDevice(v) for v in (3, 99, 0)], [3, _OnAnotherDevice(99), 0],
                                    [torch.tensor(3), torch.tensor(99), torch.tensor(0)], [torch.tensor([3]), 99, 0], torch.tensor([3, 99, 0]),
                                    np.array([3, 99, 0], dtype=np.int32), [np.int64(3), np.uint8(99), False], [3.0, 99.7, 0]])
def test_tokens_are_whatever_int_takes(tokens):
    ids = _engine()._token_ids(tokens)
    assert ids.dtype == np.int64 and ids.tolist() == [3, 99, 0]


@pytest.mark.parametrize("tokens", [[3, 100], [-1], [2 ** 70], [3, 2 ** 63], [_OnAnotherDevice(100)], torch.tensor([100]), [100.5]])
def test_tokens_outside_the_vocabulary_are_refused(tokens):
    with pytest.raises(ValueError, match="vocabulary"):
        _engine()._token_ids(tokens)


def _pair(seqs=5, pages=40, page=8):
    """An engine over a cache with a two-copy state, and a cache of the same sizes for the plain statement."""
    e = _engine()
    e.device = "cpu"
    make = lambda: PagedCache([4], num_pages=pages, max_seqs=seqs, dtype=torch.float32, device="cpu", page=page, states=[StateSpec((3,), copies=2)])      # noqa: E731
    e.cache, plain = make(), make()
    return e, plain, [(e.open_sequence(), plain.admit()) for _ in range(seqs)]


def _plain_layout(cache, items):
    """A step's arrays, token by token."""
    tokens, seq, pos, off, rd, wr, rows, runs = [], [], [], [], [], [], [], []
    for slot, t in items:
        start = cache.length[slot]
        if not len(t):
            continue
        runs.append((slot, len(tokens), len(t)))
        new = cache.extend(slot, len(t))
        r, w = cache.step_rows(slot)
        for i, v in enumerate(t):
            tokens.append(int(v))
            seq.append(slot)
            pos.append(start + i)
            off.append(i)
            rd.append(r if start else -1)
            wr.append(w if i == len(t) - 1 else -1)
            rows.append(new[i])
    return tokens, seq, pos, off, rd, wr, rows, runs


def _tiles(runs, n):
    return [[s, f + o, min(n, c - o)] for s, f, c in runs for o in range(0, c, n)]


# lengths of the five sequences' portions, step after step (pages of 8): prompts of odd sizes, steps of one token each, both mixed, idle sequences
@pytest.mark.parametrize("steps", [[(1, 1, 1, 1, 1)] * 11, [(17, 8, 9, 1, 23), (1, 1, 1, 1, 1), (1, 1, 1, 1, 1), (0, 5, 1, 0, 1), (1, 0, 0, 1, 0)],
                                   [(0, 0, 3, 0, 0), (0, 0, 1, 0, 0), (8, 0, 16, 1, 0), (1, 1, 1, 1, 1), (7, 1, 1, 1, 24)]])
def test_a_steps_arrays_are_the_plain_ones(steps):
    g = torch.Generator().manual_seed(len(steps))
    e, plain, slots = _pair()
    for n, counts in enumerate(steps):
        if n == 3:                                                             # a sequence ends and its pages are used again
            a, b = slots[1]
            e.close_sequence(a)
            plain.release(b)
            slots[1] = (e.open_sequence(), plain.admit())
        tokens = [torch.randint(0, 100, (c,), generator=g).tolist() for c in counts]
        order = torch.randperm(len(slots), generator=g).tolist()
        batch = e.layout([(slots[i][0], tokens[i]) for i in order])
        ids, seq, pos, off, rd, wr, rows, runs = _plain_layout(plain, [(slots[i][1], tokens[i]) for i in order])
        for got, want in ((batch.tokens, ids), (batch.seq, seq), (batch.pos, pos), (batch.run_off, off), (batch.state_rd, rd), (batch.state_wr, wr)):
            assert got.dtype == torch.int32 and got.tolist() == want
        assert batch.slot.dtype == torch.int64 and batch.slot.tolist() == rows
        assert (batch.items, batch.n_tokens, batch.max_pos) == (runs, len(ids), max(pos))
        assert batch.runs().tolist() == [[s, f, c, pos[f]] for s, f, c in runs]
        assert torch.equal(batch.block_table, plain.block_table())
        for n_tile in (1, 4, 64):
            assert batch.tiles(n_tile).tolist() == _tiles(runs, n_tile) and batch.tiles(n_tile).is_contiguous()
        for n_tile in (1, 2, 8):
            long, short = batch.split_tiles(n_tile)
            assert short.tolist() == [list(r) for r in runs if r[2] <= n_tile]
            assert long.tolist() == _tiles([r for r in runs if r[2] > n_tile], 4 * n_tile)
    assert e.layout([(slots[0][0], [])]) is None


def test_rows_of_many_tokens_are_the_rows_one_by_one():
    _, plain, _ = _pair()
    e, other, slots = _pair()
    for n in (1, 7, 8, 1, 24, 15, 16):
        a, b = slots[n % 2]
        assert e.cache.extend_array(a, n).tolist() == other.extend(b, n)
    with pytest.raises(CacheFull):
        e.cache.extend_array(slots[0][0], 10 ** 4)
    with pytest.raises(ValueError, match="twice"):
        e.layout([(slots[0][0], [1]), (slots[0][0], [2])])


@pytest.mark.parametrize("want", [[2, 0], (2, 0), [_OnAnotherDevice(2), _OnAnotherDevice(0)], [torch.tensor(2), 0], [np.int64(2), False]])
def test_wanted_rows_are_whatever_int_takes(want):
    e, _, slots = _pair()
    e.decode_graphs, e._forward, seen = False, lambda batch: None, []
    e.model = type("M", (), {"vocab": 100, "logits": lambda self, x, rows: seen.append(rows)})()
    e.execute([(slots[0][0], [1, 2, 3])], want)
    assert seen[0].dtype == torch.int32 and seen[0].tolist() == [2, 0]
    assert e.execute([(slots[0][0], [4])], []) is None and len(seen) == 1


@pytest.mark.parametrize("kinds", [(list, list), (list, tuple, np.array), (list, torch.tensor), (list, lambda t: [float(v) for v in t]), (list, lambda t: [_OnAnotherDevice(v) for v in t]),
                                   (list, lambda t: [np.uint64(v) for v in t]), (list, lambda t: [str(v) for v in t])])
@pytest.mark.parametrize("n", [1, 3])
def test_runs_of_different_kinds_of_tokens(kinds, n):
    e, plain, slots = _pair()
    for step in range(3):
        runs = [[(7 * i + 3 * step + j) % 100 for j in range(n)] for i in range(len(kinds))]
        flat, *rest = e._layout_host([(slots[i][0], k(t)) for i, (k, t) in enumerate(zip(kinds, runs))])
        T = n * len(kinds)
        assert flat[2 * T:3 * T].tolist() == [v for t in runs for v in t]
        assert flat[:2 * T].view(np.int64).tolist() == [r for i in range(len(kinds)) for r in plain.extend(slots[i][1], n)]
        assert rest[2] == [n * step] * len(kinds)
    before = [e.cache.length[s] for s, _ in slots]
    with pytest.raises(ValueError, match="vocabulary"):
        e._layout_host([(slots[0][0], [1] * n), (slots[1][0], [2] * (n - 1) + [100])])
    assert [e.cache.length[s] for s, _ in slots] == before          # (nothing of a refused step stays)
    with pytest.raises(KeyError):
        e._layout_host([(slots[0][0], [1]), (77, [])])


@pytest.mark.parametrize("filled, step", [((8, 8, 8), (1, 1, 1)), ((8, 7, 8), (1, 1, 1)), ((1, 1, 1), (8, 8, 16)), ((3, 9, 0), (5, 8, 1)), ((8, 8, 0), (1, 0, 9))])
def test_a_step_without_room_leaves_every_sequence_as_it_was(filled, step):
    for pages, room in ((0, False), (1, False), (2, None), (3, None), (40, True)):       # (free pages; None: as the counts say)
        e, _, slots = _pair(pages=sum(-(-n // 8) for n in filled) + pages)
        c = e.cache
        for (s, _), n in zip(slots, filled):
            if n:
                e.layout([(s, [1] * n)])
        need = sum(-(-(a + b) // 8) - -(-a // 8) for a, b in zip(filled, step))
        state = lambda: (dict(c.length), {k: list(v) for k, v in c.pages.items()}, list(c.free_pages), list(c.parity), c.table_host.clone().tolist())     # noqa: E731
        before, items = state(), [(s, [2] * n) for (s, _), n in zip(slots, step)]
        assert len(c.free_pages) == pages and (room is None or room == (need <= pages))
        if need <= pages:
            assert e.layout(items).n_tokens == sum(step)
            continue
        with pytest.raises(CacheFull):
            e.layout(items)
        assert state() == before
        e.close_sequence(slots[4][0])                                    # ... and goes on
        assert e.layout([(slots[0][0], [3] * (-filled[0] % 8))]) is not None or filled[0] % 8 == 0


@pytest.mark.parametrize("entries, size, index, taken", [(480, 2 ** 31, 0, True), (481, 100, 0, False), (1, 2 ** 31 + 64, 0, False), (1, 100, 1, False)])
def test_when_new_places_of_the_table_travel_with_a_launch(monkeypatch, entries, size, index, taken):
    e, _, _ = _pair()
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    e.cache._entered = dict.fromkeys(range(entries), 1)
    e.cache.table = type("T", (), {"is_cuda": True, "numel": lambda self: size, "device": torch.device("cuda", index)})()
    assert e.cache._new_by_kernel() == taken


@pytest.mark.parametrize("sizes, dtype, kept", [(dict(a=10 ** 8), torch.bfloat16, 24), (dict(a=10 ** 8, b=1), torch.bfloat16, None), (dict(a=5 * 10 ** 7), torch.float32, 24),
                                                (dict(a=5 * 10 ** 7 + 1), torch.float32, None), (dict(embed=10 ** 8, head=10 ** 8), torch.bfloat16, 24),
                                                (dict(embed=10 ** 8, a=1), torch.bfloat16, None), ({}, torch.bfloat16, 24)])
def test_weights_that_the_caches_hold(sizes, dtype, kept):
    from qserve_amd.serving.engine import kept_above
    assert kept_above({n: torch.empty(s, device="meta") for n, s in sizes.items()} | {"scale": 0.5}, dtype) == kept
