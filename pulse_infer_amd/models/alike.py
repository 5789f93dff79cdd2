"""Runs that differ in their tensors alone: their launches from one record.

A step that is not replayed as a graph (a prompt, a portion beside decoded tokens) goes through the same launches in every layer
of a deep model: the same entry points with the same numbers, on the same buffers of the workspace, over the layer's own weights
and pages.  Choosing and checking them takes the host some 15 us a launch, and up to a hundred tokens the GPU waits for it (a
step of 23 tokens of the 8B shape 5.6 ms for 4.0 of kernels).  So two neighbouring runs go through their parts and are listened
to; if the second's calls are the first's with every tensor of the first run replaced by the second's, the runs behind them that
are alike are launched from that record, their own tensors put in.

Alike are runs of a pre-norm block of paged attention and a gated feed-forward whose attributes, their parts' attributes and
their cache views are equal and whose tensors have equal types, shapes, strides and alignment.  That is looked at in every step,
of the objects as they are then, and a record does not outlive its step.  Whatever else happens in the two runs (a product of the
vendor library, an update added with statistics for the next norm, memory asked for, a tensor that both have or that a call names
in any other way than by its first byte) leaves everything to the parts.
"""
from __future__ import annotations

import ctypes
from operator import attrgetter
from typing import Any, List, Optional, Tuple

import torch

from ..cache.specs import PagedCacheView
from ..ops import library, timing
from ..parts import linear
from ..parts.attention import PagedAttention
from ..parts.block import PreNormBlock
from ..parts.mlp import GatedMLP
from ..parts.norm import RMSNorm

MIN_RUNS = 6      # of a stretch: fewer gain nothing
_NESTED = (PagedAttention, GatedMLP, RMSNorm, linear.Linear)


def _attributes(thing: Any, prefix: str = "") -> List[Tuple[str, bool]]:
    """The dotted names of what a block and its parts consist of, and whether each is a tensor."""
    out: List[Tuple[str, bool]] = []
    for name, value in vars(thing).items():
        if type(value) in _NESTED:
            out += _attributes(value, f"{prefix}{name}.")
        else:
            out.append((prefix + name, isinstance(value, torch.Tensor)))
    return out


def _of_its_class(thing: Any) -> bool:
    """Whether nobody has put a function of their own in the place of one of its methods (which is to be called, then)."""
    return not any(callable(getattr(type(thing), name, None)) for name in vars(thing))


def _same_tensors(a: Tuple, b: Tuple) -> bool:
    """Whether tensors differ in their contents alone (and lie at equal places of 16 bytes)."""
    return len(a) == len(b) and all(
        isinstance(y, torch.Tensor) and x.dtype == y.dtype and x.shape == y.shape and x.stride() == y.stride()
        and x.device == y.device and (x.data_ptr() ^ y.data_ptr()) % 16 == 0 for x, y in zip(a, b))


def _reach(tensor: torch.Tensor) -> int:
    """Bytes from a tensor's first value to the end of its last."""
    return (sum((n - 1) * s for n, s in zip(tensor.shape, tensor.stride())) + 1) * tensor.element_size() if tensor.numel() else 0


class AlikeRuns:
    """The runs of one step, from order index 1 on (the first run's input comes from the embedding)."""

    def __init__(self, blocks: List[Any], order: List[Any], views: List[Any]):
        self.blocks, self.order, self.views = blocks, order, views
        self.tries = 2      # stretches that are looked for

    @staticmethod
    def of(model: Any, views: List[Any]) -> Optional["AlikeRuns"]:
        """For this step, or None where the runs go through their parts all the same."""
        order = model.spec.order
        if len(order) < MIN_RUNS + 2 or model.mode != "bfloat16" or timing.active() or library.listening():
            return None
        return AlikeRuns(model.blocks, order, views)

    def _plain(self, index: int) -> bool:
        run = self.order[index]
        block = self.blocks[run.layer]
        return (type(self.views[index]) is PagedCacheView and run.offset is None and run.rejoin is None
                and type(block) is PreNormBlock and type(block.mixer) is PagedAttention and type(block.ffn) is GatedMLP
                and type(block.mixer_norm) is RMSNorm and type(block.ffn_norm) is RMSNorm)

    def _describe(self, index: int) -> Tuple[Tuple, Tuple]:
        """What must be equal for a run to be alike, and its tensors."""
        block, view = self.blocks[self.order[index].layer], self.views[index]
        numbers = tuple(len(vars(part)) for part in (block, *self._parts_of(block)))      # (an attribute that the first has not)
        return ((self._plain_of(block), numbers, view.group, view.page_size, view.writable),
                self._tensors_of(block) + (view.keys, view.values))

    def _alike(self, first: Tuple, index: int) -> bool:
        try:
            other = self._describe(index)
            return bool(other[0] == first[0]) and _same_tensors(first[1], other[1])
        except (AttributeError, TypeError, ValueError, RuntimeError):      # (one that it has not; a comparison without an answer)
            return False

    def _table(self, index: int) -> List[int]:
        """Where the tensors lie that a run's calls may name: its own and its cache's.  (Of the norm that reads its result only an
        update with statistics wants to know; ``_left`` refuses it.)"""
        return [t.data_ptr() for t in self._describe(index)[1]]

    def go(self, index: int, stream: Any, forward) -> int:
        """Run ``index`` (through ``forward(index)``) and as many behind it as are alike; the index behind them.  The last run of the
        order is left to the parts: who reads its result is no block."""
        if self.tries == 0 or index < 1 or len(self.order) - 1 - index < MIN_RUNS or not (self._plain(index) and self._plain(index + 1)):
            forward(index)
            return index + 1
        self.tries -= 1
        before = linear.library_calls

        def heard(run: int) -> Optional[List[Tuple]]:
            """The run's calls, or None where it leaves more than they do."""
            with library.listen() as calls:
                forward(run)
            left.append(self._left(stream))
            return calls if linear.library_calls == before and left[-1] is not None and left[-1] == left[0] else None

        # (the first run by itself: where a model's steps are none to record, that is all they wait for)
        left: List[Tuple] = []
        records = [heard(index)]
        if records[0] is None:
            self.tries = 0
            return index + 1
        names = _attributes(self.blocks[self.order[index].layer])
        self._plain_of = attrgetter(*[n for n, is_tensor in names if not is_tensor])
        self._tensors_of = attrgetter(*[n for n, is_tensor in names if is_tensor])
        self._parts_of = attrgetter("mixer", "mixer.qkv", "mixer.o", "ffn", "ffn.gate_up", "ffn.down", "mixer_norm", "ffn_norm")
        first, block = self._describe(index), self.blocks[self.order[index].layer]
        if not (all(_of_its_class(part) for part in (block, *self._parts_of(block))) and self._alike(first, index + 1)):
            return index + 1
        records.append(heard(index + 1))
        places = None
        if records[1] is not None:
            places = self._places(records, self._table(index), self._table(index + 1), [_reach(t) for t in first[1]])
        if places is None:
            self.tries = 0
            return index + 2
        at = index + 2
        while at + 1 < len(self.order) and self._plain(at) and self._plain(at + 1) and self._alike(first, at):
            table = self._table(at)
            for fn, name, lib, args, own in places:
                for arg, i in own:
                    arg.value = table[i]
                if fn(*args) != 0:
                    library.refused(lib, name)
            at += 1
        return at

    @staticmethod
    def _left(stream: Any) -> Optional[Tuple]:
        """What a run leaves to the next, if that is an update in a buffer and nothing else."""
        update = stream.pending
        if not isinstance(update, torch.Tensor) or stream.stats is not None or stream.copy is not None:
            return None
        return update.data_ptr(), update.dtype, update.shape, update.stride(), stream.pending_scale

    @staticmethod
    def _places(records: List[List[Tuple]], first: List[int], second: List[int], extents: List[int]) -> Optional[List[Tuple]]:
        """The second run's calls with the arguments that name tensors of its own, or None where they are not the first's.  The
        tensors lie from ``first`` and ``second`` on, ``extents`` bytes each.  Arguments that are equal in both calls stay as they are
        for every run, so none of them may lie in a tensor of the two (a tensor that both have: another run may have one of its own)."""
        if len(records[0]) != len(records[1]) or len(set(first)) != len(first) or len(set(second)) != len(second):
            return None
        if any(a == b for a, b in zip(first, second)):
            return None
        at = {pointer: i for i, pointer in enumerate(first)}
        inside = lambda value: any(p <= value < p + n for pointers in (first, second) for p, n in zip(pointers, extents))
        out = []
        for (lib, name, fn, a_args, clean), (lib_b, name_b, fn_b, b_args, clean_b) in zip(*records):
            if lib is not lib_b or name != name_b or len(a_args) != len(b_args) or not (clean and clean_b):
                return None
            own = []
            for a, b in zip(a_args, b_args):
                if type(a) is not type(b):
                    return None
                if a is None:
                    continue
                if isinstance(a, ctypes._SimpleCData):
                    if isinstance(a, ctypes.c_void_p) and a.value in at:
                        if b.value != second[at[a.value]]:
                            return None
                        own.append((b, at[a.value]))
                    elif a.value != b.value or (isinstance(a, ctypes.c_void_p) and inside(a.value or 0)):
                        return None
                    continue
                struct = getattr(a, "_obj", None), getattr(b, "_obj", None)
                if None in struct or bytes(struct[0]) != bytes(struct[1]):     # (a structure by reference)
                    return None
                held = bytes(struct[0])
                if any(inside(int.from_bytes(held[i:i + 8], "little")) for i in range(0, len(held) - 7, 8)):   # (a pointer's place)
                    return None
            out.append((fn_b, name, lib, b_args, own))
        return out
