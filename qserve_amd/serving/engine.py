"""The serving engine: a registered model + the paged cache + the scheduler + the sampler.

`Engine.step()` is the generation path: schedule -> `execute` -> sample -> book-keeping.  `execute` is the step function -
it lays the scheduled tokens out as one flat batch (token, sequence slot, position, cache row per token), runs the model
over it and returns float logits at the rows asked for.  Callers that bring their own tokens (a recorded trace, a test)
use `open_sequence` / `execute` / `close_sequence` directly and so drive the very same cache and kernels.
"""
import itertools
from dataclasses import dataclass, field

import numpy as np
import torch

from ..layers.ops import make_ops
from . import registry
from .cache import PagedCache, upload
from .sampler import SamplingParams, sample
from .scheduler import Request, Scheduler

# Weights that the last cache (256 MB) holds from step to step beside the rest; kernels then leave them there in steps of more than 24 rows (streams_once
# in csrc/serve/serve_stream.h has both sides' times)
KEPT_WEIGHTS = 200_000_000
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}


def kept_above(weights, dtype):
    """HipOps.kept_above for a model of these checkpoint tensors (a step reads a few rows of an embedding that is not the head too)."""
    read = sum(w.numel() for n, w in weights.items() if isinstance(w, torch.Tensor) and not (n == "embed" and "head" in weights))
    return 24 if read * dtype.itemsize <= KEPT_WEIGHTS else None


@dataclass
class StepBatch:
    """One step's tokens as the kernels read them (device tensors unless noted)."""
    tokens: torch.Tensor        # int32 [T]
    seq: torch.Tensor           # int32 [T]  sequence slot (row of the block table)
    pos: torch.Tensor           # int32 [T]  position in its sequence
    slot: torch.Tensor          # int64 [T]  flat cache row the token's state is written to
    block_table: torch.Tensor   # int32 [slots, pages]
    max_pos: int                # host: largest position in the batch
    n_tokens: int
    items: list = None          # host: [(sequence slot, first flat token index, tokens)] - runs of consecutive positions
    run_off: torch.Tensor = None    # int32 [T]  index of the token within its run
    state_rd: torch.Tensor = None   # int32 [T]  two-copy state row the token's run reads (-1: the run starts its sequence)
    state_wr: torch.Tensor = None   # int32 [T]  two-copy state row to write, on the LAST token of a run (-1 elsewhere)
    starts: list = None         # host: position of each run's first token (None: not known on the host)
    _tiles: dict = field(default_factory=dict)
    _runs: torch.Tensor = None
    _single: torch.Tensor = None    # int32 [T, 3] = (slot, token, 1) where every run is one token: the tiles of any size

    def runs(self):
        """int32 [n_runs, 4] = (sequence slot, first flat token index, tokens, position of the first token), on the device.
        The engine's layout brings it along with the other metadata; a batch made by hand gets it here (one synchronisation)."""
        if self._runs is None:
            pos = self.pos.tolist()
            rows = [(slot, first, n, pos[first]) for slot, first, n in self.items]
            self._runs = torch.tensor(rows, dtype=torch.int32).reshape(-1, 4).to(self.pos.device)
        return self._runs

    def tiles(self, tokens_per_tile):
        """Work tiles for kernels that serve a few consecutive tokens of one sequence per workgroup: int32 [n, 3] =
        (sequence slot, first flat token index, tokens <= tokens_per_tile), on the device; cached per size."""
        if self._single is not None:
            return self._single
        t = self._tiles.get(tokens_per_tile)
        if t is None:
            rows = [(slot, first + o, min(tokens_per_tile, n - o)) for slot, first, n in self.items
                    for o in range(0, n, tokens_per_tile)]
            t = upload(np.array(rows, dtype=np.int32).reshape(-1, 3), self.tokens.device if self.tokens is not None else self.pos.device)
            self._tiles[tokens_per_tile] = t
        return t

    def split_tiles(self, tokens_per_step_tile):
        """Work tiles for kernels with a form of their own for short runs: -> (prompt tiles, step tiles), int32 [n, 3] as `tiles`.  Runs of at
        most `tokens_per_step_tile` tokens become one step tile each, longer ones prompt tiles of up to four times as many tokens."""
        if self._single is not None:
            return self._single[:0], self._single
        n = int(tokens_per_step_tile)
        key = ("split", n)
        if key not in self._tiles:
            short = [run for run in self.items if run[2] <= n]
            long = [(slot, first + o, min(4 * n, cnt - o)) for slot, first, cnt in self.items if cnt > n for o in range(0, cnt, 4 * n)]
            both = upload(np.array(short + long, dtype=np.int32).reshape(-1, 3), self.pos.device)
            self._tiles[key] = both
        both, k = self._tiles[key], sum(1 for run in self.items if run[2] <= n)
        return both[k:], both[:k]

    def key_runs(self, window, tokens_per_tile):
        """For kernels that lay the keys of whole runs out one behind another: -> (runs int32 [n, 4] = (sequence slot, position of the first key that a
        token of the run sees, keys, first row), tiles int32 [m, 8] = (first flat token index, tokens <= tokens_per_tile, position of the first, then
        the run's last three, 0, 0), the longest first, rows (every run's keys padded to a multiple of 8), most keys of a run).  None where the host does not
        know the positions or every run is one token."""
        if self.starts is None or self._single is not None:
            return None
        key = ("keys", int(window or 0), int(tokens_per_tile))
        if key not in self._tiles:
            runs, tiles, rows = [], [], 0
            for (slot, first, n), start in zip(self.items, self.starts):
                lo = max(0, start - int(window) + 1) if window else 0
                keys = start + n - lo
                runs.append((slot, lo, keys, rows))
                tiles += [(first + o, min(tokens_per_tile, n - o), start + o, lo, rows, keys, 0, 0) for o in range(0, n, tokens_per_tile)]
                rows += (keys + 7) // 8 * 8
            tiles.sort(key=lambda t: -(t[2] + t[1] - max(t[3], t[2] - int(window) + 1 if window else 0)))
            both = upload(np.array([v for r in runs for v in r] + [v for t in tiles for v in t], dtype=np.int32), self.pos.device)
            self._tiles[key] = (both[:4 * len(runs)].view(-1, 4), both[4 * len(runs):].view(-1, 8), rows, max(r[2] for r in runs))
        return self._tiles[key]


class Engine:
    def __init__(self, model_cls, config, weights, dtype="bfloat16", device="cuda:0", max_tokens=4096, max_seqs=4,
                 backend="hip", max_batch_tokens=2048, prefill_chunk=512, page=64, decode_graphs=False):
        """decode_graphs: replay steps in which every sequence brings exactly one token from a hipGraph (captured per batch
        size and context bucket; the launch sequence of such a step has no host synchronisation).  Off unless asked for."""
        self.dtype = DTYPES[dtype] if isinstance(dtype, str) else dtype
        self.device = torch.device(device)
        if self.dtype == torch.float32 and self.device.type == "cuda":
            torch.backends.cuda.matmul.allow_tf32 = False          # float32 means float32 products
            torch.backends.cudnn.allow_tf32 = False
        self.ops = make_ops(backend, self.dtype, self.device)
        self.ops.kept_above = kept_above(weights, self.dtype)
        self.model = model_cls.from_config(config, weights, self.ops, self.device, self.dtype, page=page)
        self.cache = PagedCache(self.model.cache_rows, (int(max_tokens) + page - 1) // page, max_seqs, self.dtype, self.device,
                                page=page, states=getattr(self.model, "state_specs", ()))
        self.scheduler = Scheduler(self.cache, max_batch_tokens, prefill_chunk)
        self.requests = {}
        self._ids = itertools.count()
        self.decode_graphs = bool(decode_graphs) and backend == "hip"
        self._graphs = {}                      # key -> _DecodeGraph, or False where capture failed (that shape runs eagerly)

    @classmethod
    def from_pretrained(cls, model_dir, **kw):
        """model_dir: config.json + *.safetensors; the model class is chosen by the config's architecture."""
        from ..loader import iterate_checkpoint
        config = registry.read_config(model_dir)
        model_cls, kind = registry.resolve_model(config)
        if kind != "paged":
            raise ValueError(f"architecture {registry.architecture_of(config)!r} is served by the {kind} engine, not this one")
        return cls(model_cls, config, dict(iterate_checkpoint(model_dir)), **kw)

    # ---- the step function -------------------------------------------------------------------------------------------------
    def open_sequence(self):
        return self.cache.admit()

    def close_sequence(self, slot):
        self.cache.release(slot)

    def _token_ids(self, t):
        """The tokens of one run as an int64 array, checked against the vocabulary.  Anything whose elements int() takes: whole numbers go
        through numpy at once, the rest (tensors on a GPU, other arrays) one by one."""
        a = None
        if isinstance(t, (list, tuple)) and t and type(t[0]) is int:
            try:
                a = np.array(t)
            except Exception:                                          # (an element further on that numpy cannot convert)
                pass
        if a is None or a.dtype != np.int64 or a.ndim != 1:
            ids = [int(v) for v in t]
            if any(not 0 <= v < self.model.vocab for v in ids):
                raise ValueError(f"token id outside the vocabulary of {self.model.vocab}")
            return np.array(ids, dtype=np.int64)
        if a.size and (a.min() < 0 or a.max() >= self.model.vocab):
            raise ValueError(f"token id outside the vocabulary of {self.model.vocab}")
        return a

    def _all_ids(self, runs):
        """The tokens of several runs, one behind another.  Runs of whole numbers go through numpy together: 64 runs of 75 tokens took 0.5 ms one by one."""
        if all(isinstance(t, (list, tuple)) and type(t[0]) is int for t in runs):
            try:
                a = np.array(list(itertools.chain.from_iterable(runs)))
            except Exception:                                          # (an element that numpy cannot convert)
                a = None
            if a is not None and a.dtype == np.int64 and a.ndim == 1 and a.min() >= 0 and a.max() < self.model.vocab:
                return a
        return np.concatenate([self._token_ids(t) for t in runs])     # (one by one: also where one is outside the vocabulary)

    def _layout_host(self, items):
        """Host side of a step's batch: extends the sequences' pages, swaps their two-copy states.  -> (everything the device needs as one
        int32 array, see `_batch_of`; runs [(slot, first flat token, tokens)]; largest position; every run's first position) or None."""
        cache, counts = self.cache, [len(t) for _, t in items]
        slots = [slot for (slot, _), n in zip(items, counts) if n]
        if len(set(slots)) != len(slots):
            raise ValueError("a sequence appears twice in one step")
        for slot, _ in items:
            cache.length[slot]                                         # (a slot that is not live raises, also with no tokens)
        if not slots:
            return None
        ids = self._all_ids([t for (_, t), n in zip(items, counts) if n])
        counts = [n for n in counts if n]
        cache.room_for(slots, counts)                                  # (a step that is refused leaves every sequence as it was)
        R, T = len(slots), len(ids)
        single = T == R
        flat = np.empty(8 * T + (7 if single else 4) * R, dtype=np.int32)
        row_of, meta, runs4 = flat[:2 * T].view(np.int64), flat[2 * T:8 * T].reshape(6, T), flat[8 * T:8 * T + 4 * R].reshape(R, 4)
        if single:
            rows, starts, firsts = [], [], range(R)
            for slot in slots:
                r, start = cache.extend_one(slot)
                rows.append(r)
                starts.append(start)
            row_of[:] = rows
        else:
            starts, firsts = [], [0, *itertools.accumulate(counts[:-1])]
            for slot, n in zip(slots, counts):
                starts.append(cache._grow(slot, n)[1])
        states = [cache.step_rows(slot) for slot in slots]
        read, write = [rd if start else -1 for (rd, _), start in zip(states, starts)], [wr for _, wr in states]
        runs4[:, 0], runs4[:, 1], runs4[:, 2], runs4[:, 3] = slots, firsts, counts, starts
        meta[0] = ids
        if single:
            meta[1], meta[2], meta[3], meta[4], meta[5] = slots, starts, 0, read, write
            tiles = flat[8 * T + 4 * R:].reshape(R, 3)
            tiles[:, 0], tiles[:, 1], tiles[:, 2] = slots, firsts, 1
        else:
            lasts = np.cumsum(counts) - 1
            meta[1], meta[4], meta[5] = np.repeat(slots, counts), np.repeat(read, counts), -1
            meta[3] = np.arange(T) - np.repeat(firsts, counts)
            meta[2] = meta[3] + np.repeat(starts, counts)
            meta[5, lasts] = write
            row_of[:] = cache.rows_of(meta[1], meta[2])
        return flat, list(zip(slots, firsts, counts)), max(start + n for start, n in zip(starts, counts)) - 1, starts

    def layout(self, items):
        """items: [(slot, tokens)] -> the StepBatch of these tokens on the device (None if there are none).  Part of `execute`;
        callers that run single layers use it directly."""
        host = self._layout_host(items)
        return None if host is None else self._batch_of(upload(host[0], self.device), *host[1:])

    def _batch_of(self, flat, runs, max_pos, starts=None):
        """The StepBatch over one int32 tensor: cache rows (int64 [T]) | token, slot, position, index in run, state row to read, state row to
        write ([6, T]) | runs ([R, 4]) | the tiles of single tokens ([R, 3], where every run is one)."""
        T, R = sum(n for _, _, n in runs), len(runs)
        meta = flat[2 * T:8 * T].view(6, T)
        return StepBatch(tokens=meta[0], seq=meta[1], pos=meta[2], slot=flat[:2 * T].view(torch.int64), block_table=self.cache.block_table(),
                         max_pos=max_pos, n_tokens=T, items=list(runs), run_off=meta[3], state_rd=meta[4], state_wr=meta[5],
                         starts=starts, _runs=flat[8 * T:8 * T + 4 * R].view(R, 4), _single=flat[8 * T + 4 * R:].view(R, 3) if T == R else None)

    @torch.no_grad()
    def execute(self, items, want):
        """items: [(slot, tokens)] - the next tokens of live sequences, all run as one batch; want: flat indices into the
        concatenated tokens.  -> float logits [len(want), vocab] (None if want is empty)."""
        host = self._layout_host(items)
        if host is None:
            return None
        if self.decode_graphs and all(n == 1 for _, _, n in host[1]):
            out = self._execute_graph(*host[:3])
            if out is not None:
                if not want:
                    return None
                want = [int(v) for v in want]
                return self.ops.copied(out) if want == list(range(out.size(0))) else out[upload(np.array(want, dtype=np.int64), self.device)]
        batch = self._batch_of(upload(host[0], self.device), *host[1:])
        x = self._forward(batch)
        if not want:
            return None
        return self.model.logits(x, upload(np.array([int(v) for v in want], dtype=np.int32), self.device))

    def _forward(self, batch):
        if self.cache.states:
            return self.model.forward(batch, self.cache.pools, states=self.cache.states)
        return self.model.forward(batch, self.cache.pools)

    # ---- decode steps from a hipGraph ------------------------------------------------------------------------------------------
    GRAPH_BUCKET = 128                         # positions per context bucket (a graph freezes what is derived from max_pos)

    def _execute_graph(self, flat, runs, max_pos):
        """One token per sequence: fill the static input of the graph captured for (batch size, context bucket, model
        signature) and replay it.  -> float logits for every row (the graph's own buffer), or None if this shape runs eagerly."""
        B, dev = len(runs), self.device
        bucket = max_pos // self.GRAPH_BUCKET
        sig = self.model.graph_signature() if hasattr(self.model, "graph_signature") else ()
        key = (B, bucket, sig)
        G = self._graphs.get(key)
        if G is False:
            return None
        if G is None:
            if len(self._graphs) >= 16:
                self._graphs.clear()
            G = {"flat": upload(flat, dev), "rows": torch.arange(B, dtype=torch.int32, device=dev)}
            G["batch"] = batch = self._batch_of(G["flat"], runs, (bucket + 1) * self.GRAPH_BUCKET - 1)
            if hasattr(self.model, "reserve_positions"):
                self.model.reserve_positions(batch.max_pos + 1)
                key = (B, bucket, self.model.graph_signature() if hasattr(self.model, "graph_signature") else ())
            try:
                side = torch.cuda.Stream()
                side.wait_stream(torch.cuda.current_stream())
                kept = [s.clone() for s in self.cache.states]      # a recurrent state must not advance twice: the warm-up's
                with torch.cuda.stream(side):                      # warm-up outside capture (allocator, lazy initialisation)
                    self.model.logits(self._forward(batch), G["rows"])
                torch.cuda.current_stream().wait_stream(side)
                for s, k in zip(self.cache.states, kept):          # ... step is taken back before the replay takes it
                    s.copy_(k)
                torch.cuda.synchronize()
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g):
                    G["logits"] = self.model.logits(self._forward(batch), G["rows"])
                G["graph"] = g
            except Exception:                                      # e.g. a launch sequence that synchronises: run eagerly
                torch.cuda.synchronize()
                self._graphs[key] = False
                return None
            self._graphs[key] = G
        else:
            self.ops.put_words(G["flat"], flat)
        self.cache.block_table()
        G["graph"].replay()
        return G["logits"]

    # ---- generation ------------------------------------------------------------------------------------------------------------
    def add_request(self, prompt, params=None, request_id=None):
        params = params or SamplingParams()
        rid = request_id if request_id is not None else f"req{next(self._ids)}"
        r = Request(rid, [int(t) for t in prompt], params)
        if params.seed is not None:
            r.generator = torch.Generator(device=self.device).manual_seed(params.seed)
        self.scheduler.add(r)
        self.requests[rid] = r
        return rid

    def step(self):
        """Run one scheduled batch.  -> [(request id, new token, finished)] for the requests that got a token."""
        work = self.scheduler.schedule()
        if not work:
            return []
        want, at = [], 0
        for w in work:
            at += len(w.tokens)
            if w.sample:
                want.append(at - 1)
        logits = self.execute([(w.request.slot, w.tokens) for w in work], want)
        for w in work:
            w.request.computed += len(w.tokens)
        out = []
        if want:
            sampling = [w.request for w in work if w.sample]
            new = sample(logits, [r.params for r in sampling], [r.generator for r in sampling])
            for r, tok in zip(sampling, new):
                r.output.append(tok)
                done = len(r.output) >= r.params.max_new or (r.params.stop_token is not None and tok == r.params.stop_token)
                if done:
                    self.scheduler.finish(r)
                out.append((r.id, tok, done))
        return out

    def has_work(self):
        return bool(self.scheduler.waiting or self.scheduler.running)

    def generate(self, prompts, params=None, **kw):
        """prompts: lists of token ids -> lists of generated token ids (same order)."""
        if params is None:
            params = SamplingParams(**kw)
        ids = [self.add_request(p, params) for p in prompts]
        while self.has_work():
            if not self.step() and not self.scheduler.running:
                raise RuntimeError("the scheduler cannot place any waiting request")
        return [self.requests.pop(i).output for i in ids]
