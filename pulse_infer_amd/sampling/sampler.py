"""Choosing next tokens for a batch of logits rows on the GPU.

One kernel call serves all rows; each row carries its own options.  The "seen"
sets of the presence penalty live in the per-request slots (one bit per
vocabulary entry), are cleared when a slot is taken and updated as tokens
arrive.
"""
from __future__ import annotations

from typing import List, Optional, Sequence

import torch

from ..ops import kernels
from .params import SamplingParams


def one_a_row(values: Sequence, rows: int, name: str) -> Sequence:
    """``values`` for ``rows`` rows: as they are, or the one there is for all of them."""
    if len(values) == 1 and rows > 1:
        return [values[0]] * rows
    if len(values) < rows:
        raise ValueError(f"sampling: {len(values)} {name} for {rows} rows")
    return values


class Sampler:
    def __init__(self, vocab_size: int, num_slots: int, device: torch.device,
                 banned_tokens: Optional[Sequence[int]] = None):
        self.vocab = int(vocab_size)
        self.device = torch.device(device)
        self.words = (self.vocab + 31) // 32
        self.num_slots = int(num_slots)
        self.seen: Optional[torch.Tensor] = None  # [slots, words], made when a request first needs it
        self.banned: Optional[torch.Tensor] = None
        self._part_val: Optional[torch.Tensor] = None
        self._part_idx: Optional[torch.Tensor] = None
        self._chunked: Optional[dict] = None             # scratch of the sampling in chunks
        # pinned [6, rows] int32 and device twins, two of each used in turn: a step's per-row options go up without
        # the host waiting, and a caller may queue a step's sampling while it still waits for the tokens of the step
        # before (not for older ones: a pair is used again two calls later)
        self._options_host: List[Optional[torch.Tensor]] = [None, None]
        self._options_dev: List[Optional[torch.Tensor]] = [None, None]
        self._options_views: List[Optional[tuple]] = [None, None]     # of the device twins: (rows, a view an option)
        self._turn = 0
        if banned_tokens:
            host = torch.zeros(self.words, dtype=torch.int64)
            for tok in banned_tokens:
                if 0 <= tok < self.vocab:
                    host[tok >> 5] |= 1 << (tok & 31)
            # keep the bit patterns when narrowing to int32
            host = torch.where(host >= 2 ** 31, host - 2 ** 32, host)
            self.banned = host.to(torch.int32).to(self.device)

    # -------------------------------------------------------------- seen sets
    def start_request(self, slot: int, params: SamplingParams, tokens: Sequence[int]) -> None:
        """A request took ``slot``: clear its seen set and mark the tokens it starts with."""
        if params.presence_penalty > 0.0:
            if self.seen is None:
                self.seen = torch.zeros((self.num_slots, self.words), dtype=torch.int32, device=self.device)
            self.seen[slot].zero_()
            self.note_tokens([slot] * len(tokens), list(tokens))

    def note_tokens(self, slots: Sequence[int], tokens: Sequence[int]) -> None:
        if self.seen is None or not slots:
            return
        both = torch.tensor([list(slots), list(tokens)], dtype=torch.int32).to(self.device)   # one upload
        kernels.mark_seen(self.seen, both[0], both[1], self.vocab)

    def note_on_device(self, slots: torch.Tensor, tokens: torch.Tensor) -> None:
        """``note_tokens`` for tokens that are still on the device (``launch``'s result): ``slots`` int32 on the
        device, -1 where a row's request keeps no seen set; rows without a token (-1) mark nothing."""
        if self.seen is not None and slots.numel():
            kernels.mark_seen(self.seen, slots, tokens, self.vocab)

    # ---------------------------------------------------------------- sampling
    def sample(self, logits: torch.Tensor, params: Sequence[SamplingParams], slots: Sequence[int],
               counters: Sequence[int], default_seeds: Sequence[int]) -> List[int]:
        """One token per row.  ``counters[r]`` is how many tokens row r's request has drawn before."""
        if logits.shape[0] == 0:
            return []
        return self.launch(logits, params, slots, counters, default_seeds).tolist()

    def launch(self, logits: torch.Tensor, params: Sequence[SamplingParams], slots: Sequence[int],
               counters: Sequence[int], default_seeds: Sequence[int]) -> torch.Tensor:
        """``sample`` without waiting: the tokens as an int32 vector on the device, the kernels only queued."""
        rows = logits.shape[0]
        out = torch.empty(rows, dtype=torch.int32, device=self.device)
        if rows == 0:
            return out
        if all(p.greedy and p.presence_penalty == 0.0 for p in params) and self.banned is None:
            need = rows * kernels.argmax_chunks(logits.shape[1])
            if self._part_val is None or self._part_val.numel() < need:
                self._part_val = torch.empty(need, dtype=torch.float32, device=self.device)
                self._part_idx = torch.empty(need, dtype=torch.int32, device=self.device)
            kernels.argmax(logits, out, self._part_val, self._part_idx)
            return out
        params = one_a_row(params, rows, "options")
        if len(params) != rows:
            raise ValueError(f"sampling: options of {len(params)} requests for {rows} rows")
        slots, counters, default_seeds = (one_a_row(v, rows, name) for v, name in (
            (slots, "slots"), (counters, "counters"), (default_seeds, "seeds")))
        # every per-row option in one upload: rows of a [6, R] int32 array, the float ones as their bit patterns
        turn = self._turn
        self._turn = 1 - turn
        if self._options_host[turn] is None or self._options_host[turn].shape[1] < rows:
            self._options_host[turn] = torch.empty((6, max(rows, 64)), dtype=torch.int32, pin_memory=True)
            self._options_dev[turn] = torch.empty((6, max(rows, 64)), dtype=torch.int32, device=self.device)
            self._options_views[turn] = None
        # (the copy out of these pinned rows two calls ago has run: its tokens have been waited for)
        dev = self._options_dev[turn]
        by_k, by_p, penalized = kernels.sample_options(self._options_host[turn], dev, [p.packed for p in params], slots, counters,
                                                       default_seeds)
        views = self._options_views[turn]
        if views is None or views[0] != rows:
            floats = tuple(dev[i, :rows].view(torch.float32) for i in (0, 2, 3, 4))
            views = self._options_views[turn] = (rows, dev[1, :rows], dev[5, :rows], *floats)
        _, top_k, seen_row, temperature, top_p, uniform, penalty = views
        if not (penalized and self.seen is not None):
            penalty = seen_row = None
        seen = self.seen if penalty is not None else None
        # in chunks of the vocabulary; which way a row goes there depends on its own options alone, so a seeded
        # request draws the same tokens whatever else is in the batch.  An option that no row uses is left out
        # (a kernel less), which changes no row's choice.
        if self._chunked is None or self._chunked["done"].numel() < rows:
            self._chunked = kernels.sample_chunked_scratch(rows, logits.shape[1], self.device)
        kernels.sample_chunked(logits, out, self._chunked, temperature=temperature,
                               top_k=top_k if by_k else None, top_p=top_p if by_p else None,
                               uniform=uniform, penalty=penalty, seen_row=seen_row, seen_masks=seen,
                               banned=self.banned)
        return out
