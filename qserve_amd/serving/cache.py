"""Paged cache with sequence slots, and the fixed-size state of a sequence.

One page id space serves every layer: page p is rows [p * page, (p + 1) * page) of each layer's pool, and a pool's rows are as
wide as that layer's cached state per token (layers may differ; a width (n, w) makes n pools of one allocation, [n, rows, w]:
the key / value heads of one attention layer; (n, w, r) gives a page r rows instead of `page`: state kept per block of B
positions with r = ceil(page / B), the block that starts in page p at offset o owning row p r + o // B).  A live sequence owns a slot (a row of the block table) and the pages its
tokens fill; both go back to the free lists when it ends and are handed out again, most recently freed first.

State that does not grow with the sequence (a recurrent matrix, the last inputs of a short convolution, the previous token of
a token shift) lives in per-slot tensors, one per `StateSpec`:
* copies = 1: row `slot`.  One workgroup reads it, runs the sequence's tokens of the step, and writes it back.
* copies = 2: rows 2 slot + {0, 1}, read from one and written to the other, swapped every step the sequence takes part in
  (`step_rows`).  For state that the step's FIRST token reads and its LAST token writes from different workgroups.
A sequence's state is never cleared: kernels take a run that starts at position 0 as starting from zeros.
"""
import numpy as np
import torch

from ._lib import check, lib


def upload(a, device):
    """numpy array -> tensor on `device`.  To a GPU through a pinned buffer and without waiting for the copy (torch hands a pinned buffer
    out again only after the copies from it have run); a copy from pageable memory would wait for everything on the stream."""
    t = torch.from_numpy(a)
    if torch.device(device).type != "cuda":
        return t.to(device)
    return torch.empty(t.shape, dtype=t.dtype, pin_memory=True).copy_(t).to(device, non_blocking=True)


class CacheFull(RuntimeError):
    pass


class StateSpec:
    """Per-sequence state of fixed size: `shape` per sequence, float unless `dtype` says otherwise; copies: see the module."""

    def __init__(self, shape, dtype=torch.float32, copies=1):
        if copies not in (1, 2):
            raise ValueError("a state has one copy or two")
        self.shape, self.dtype, self.copies = tuple(int(n) for n in shape), dtype, copies


class PagedCache:
    def __init__(self, row_widths, num_pages, max_seqs, dtype, device, page=64, states=()):
        if num_pages <= 0 or max_seqs <= 0:
            raise ValueError("the cache needs at least one page and one slot")
        self.page, self.num_pages, self.max_seqs = page, int(num_pages), int(max_seqs)
        rows = self.num_pages * page
        self.pools = []
        for w in row_widths:
            if isinstance(w, int):
                shape = (rows, w)
            else:
                if len(w) > 2 and not 0 < int(w[2]) <= page:
                    raise ValueError(f"a page of {page} positions cannot hold {w[2]} block rows")
                shape = (int(w[0]), self.num_pages * int(w[2]) if len(w) > 2 else rows, int(w[1]))
            self.pools.append(torch.zeros(shape, dtype=dtype, device=device))
        self.states = [torch.zeros((self.max_seqs * s.copies,) + s.shape, dtype=s.dtype, device=device) for s in states]
        self.parity = [0] * self.max_seqs
        self.free_pages = list(range(self.num_pages - 1, -1, -1))      # pop() -> lowest id first; freed pages are reused first
        self.free_slots = list(range(self.max_seqs - 1, -1, -1))
        self.pages = {}                                                # slot -> [page ids]
        self.length = {}                                               # slot -> tokens held
        self.table_host = torch.zeros((self.max_seqs, self.num_pages), dtype=torch.int32)
        self.table_rows = self.table_host.numpy()                      # the same memory: [slot, page of the sequence] -> page id
        self.table = self.table_host.to(device)
        self._dirty = False
        self._entered = {}                                             # place in the table -> page id, since the last upload

    def pages_for(self, tokens):
        return (tokens + self.page - 1) // self.page

    def admit(self):
        if not self.free_slots:
            raise CacheFull(f"all {self.max_seqs} sequence slots are in use")
        s = self.free_slots.pop()
        self.pages[s], self.length[s] = [], 0
        return s

    def room_for(self, slots, counts):
        """Raises CacheFull, with nothing changed, if these sequences cannot all grow by their counts."""
        if sum(counts) // self.page + len(slots) <= len(self.free_pages):      # (no sequence needs more than n / page + 1)
            return
        need = sum(self.pages_for(self.length[s] + n) - len(self.pages[s]) for s, n in zip(slots, counts))
        if need > len(self.free_pages):
            raise CacheFull(f"{need} more pages needed, {len(self.free_pages)} free of {self.num_pages}")

    def _grow(self, slot, n):
        """Pages for n more tokens of `slot`.  -> (its pages, tokens it held before)."""
        have, start = self.pages[slot], self.length[slot]
        need = self.pages_for(start + n) - len(have)
        if need > len(self.free_pages):
            raise CacheFull(f"{need} more pages needed, {len(self.free_pages)} free of {self.num_pages}")
        for _ in range(need):
            p = self.free_pages.pop()
            self.table_rows[slot, len(have)] = p                       # (an element of a tensor takes 40 times as long)
            self._entered[slot * self.num_pages + len(have)] = p
            have.append(p)
            self._dirty = True
        self.length[slot] = start + n
        return have, start

    def extend(self, slot, n):
        """Make room for n more tokens of `slot`; returns their flat row indices (position order)."""
        have, start = self._grow(slot, n)
        return [have[j // self.page] * self.page + j % self.page for j in range(start, start + n)]

    def extend_array(self, slot, n):
        """`extend` for many tokens: the row indices as an int64 array."""
        start = self._grow(slot, n)[1]
        return self.rows_of(slot, np.arange(start, start + n, dtype=np.int64))

    def extend_one(self, slot):
        """`extend` for one token: -> (its row index, its position)."""
        start = self.length[slot]
        at = start % self.page
        if not at:
            return self.extend(slot, 1)[0], start
        self.length[slot] = start + 1
        return self.pages[slot][start // self.page] * self.page + at, start

    def rows_of(self, slots, positions):
        """The flat row indices of positions that sequences hold, slots and positions as arrays."""
        return self.table_rows[slots, positions // self.page].astype(np.int64) * self.page + positions % self.page

    def step_rows(self, slot):
        """-> (row to read, row to write) of the two-copy states for this step of `slot`; the next step reads what this one
        writes.  Call once per step and sequence."""
        p = self.parity[slot]
        self.parity[slot] = 1 - p
        return 2 * slot + p, 2 * slot + 1 - p

    def release(self, slot):
        self.free_pages.extend(reversed(self.pages.pop(slot)))
        del self.length[slot]
        self.free_slots.append(slot)

    def _new_by_kernel(self):
        """Whether a launch's arguments carry what is new in the table: few entries, places that 32 bits hold, the device that launches go to."""
        return (self.table.is_cuda and len(self._entered) <= 480 and self.table.numel() <= 2 ** 31 and self.table.device.index == torch.cuda.current_device())

    def block_table(self):
        """The device copy of the block table, uploaded if pages were handed out since the last call."""
        if self._dirty:
            if self._new_by_kernel():                                  # (a step's few: no copy command, and no more than what is new)
                new = np.array(list(self._entered.items()), dtype=np.int32)
                check(lib().qsv_set_words(self.table.data_ptr(), new.ctypes.data, len(new), torch.cuda.current_stream(self.table.device).cuda_stream), "set_words")
            elif self.table.is_cuda:                                   # (a pinned copy: the host's table may change before the device has read it)
                self.table.copy_(torch.empty(self.table_host.shape, dtype=torch.int32, pin_memory=True).copy_(self.table_host), non_blocking=True)
            else:
                self.table.copy_(self.table_host)
            self._dirty, self._entered = False, {}
        return self.table
