"""What makes two runs' calls a record that other runs can be launched from."""
import ctypes

import types

import numpy as np
import pytest
import torch

from pulse_infer_amd.cache.specs import PagedCacheView
from pulse_infer_amd.models.alike import AlikeRuns
from pulse_infer_amd.models.spec import RunSpec
from pulse_infer_amd.ops import library
from pulse_infer_amd.parts.attention import PagedAttention
from pulse_infer_amd.parts.block import ParallelBlock, PreNormBlock
from pulse_infer_amd.parts.linear import Linear
from pulse_infer_amd.parts.mlp import GatedMLP
from pulse_infer_amd.parts.norm import RMSNorm

P, I, F = ctypes.c_void_p, ctypes.c_int, ctypes.c_float


class Pair(ctypes.Structure):
    _fields_ = [("a", ctypes.c_int), ("b", ctypes.c_float)]


def calls(weight, number=3, factor=0.5, name="entry", pair=(1, 2.0), clean=True, kind=I):
    lib, entry = "library", "function"
    return [(lib, name, entry, (P(7), P(weight), kind(number), F(factor), None, P(0), ctypes.byref(Pair(*pair))), clean),
            (lib, "second", entry, (P(weight + 64), P(weight)), clean)]


FIRST, SECOND = [100, 164, 300], [200, 264, 400]      # where the runs' tensors lie
EXTENTS = [32, 32, 32]                                # and how far they reach


def test_the_second_runs_arguments_take_the_tensors_of_others():
    second = calls(200)
    places = AlikeRuns._places([calls(100), second], FIRST, SECOND, EXTENTS)
    assert [[i for _, i in own] for *_, own in places] == [[0], [1, 0]]
    for *_, own in places:
        for arg, i in own:
            arg.value = [1000, 1064, 1300][i]
    assert second[0][3][1].value == 1000 and second[1][3][0].value == 1064 and second[0][3][0].value == 7


@pytest.mark.parametrize("other", [dict(weight=201), dict(number=4), dict(factor=0.25), dict(name="another"), dict(pair=(1, 3.0)),
                                   dict(clean=False), dict(weight=100), dict(kind=ctypes.c_int64)])
def test_calls_that_differ_in_more_than_tensors_are_no_record(other):
    assert AlikeRuns._places([calls(100), calls(**{"weight": 200, **other})], FIRST, SECOND, EXTENTS) is None


def test_no_record_where_calls_are_missing_or_places_are_shared():
    assert AlikeRuns._places([calls(100), calls(200)[:1]], FIRST, SECOND, EXTENTS) is None
    assert AlikeRuns._places([calls(100), calls(200)], [100, 164, 100], SECOND, EXTENTS) is None
    assert AlikeRuns._places([calls(100), calls(100)], FIRST, FIRST, EXTENTS) is None     # (the same tensors: another run's may differ)
    assert AlikeRuns._places([calls(100), calls(200)], FIRST, [200, 264, 300], EXTENTS) is None


class Sunk(ctypes.Structure):
    _fields_ = [("sink", ctypes.c_void_p), ("softcap", ctypes.c_float)]


def made(kind, **attributes):
    part = kind.__new__(kind)
    vars(part).update(attributes)
    return part


def block():
    linear = lambda: made(Linear, weight=torch.zeros(4, 4), mode="bfloat16")
    norm = lambda: made(RMSNorm, weight=torch.zeros(4), eps=1e-6)
    return made(PreNormBlock, mixer=made(PagedAttention, qkv=linear(), o=linear(), sink=torch.zeros(4)),
                ffn=made(GatedMLP, gate_up=linear(), down=linear()), mixer_norm=norm(), ffn_norm=norm())


class Launches:
    """A step over ``order``, whose runs make two calls each: one with a structure that holds the sinks' place.  Every call that
    was made, by a run's parts or from a record, is kept as the places it named."""

    def __init__(self, blocks, order):
        self.blocks, self.order, self.through = blocks, order, []
        self.views = [PagedCacheView(0, torch.zeros(2, 4), torch.zeros(2, 4), 16) for _ in order]
        self.seen = []
        self.update = torch.zeros(4)
        self.stream = types.SimpleNamespace(pending=self.update, stats=None, copy=None, pending_scale=1.0)

    def entry(self, *args):
        self.seen.append([getattr(a, "value", None) if not hasattr(a, "_obj") else a._obj.sink for a in args])
        return 0

    def calls_of(self, index):
        block, view = self.blocks[self.order[index].layer], self.views[index]
        mixer = block.mixer
        return [(P(7), P(mixer.qkv.weight.data_ptr()), P(view.keys.data_ptr()), ctypes.byref(Sunk(mixer.sink.data_ptr(), 2.0))),
                (P(mixer.o.weight.data_ptr()), P(block.ffn.down.weight.data_ptr()))]

    def forward(self, index):
        self.through.append(index)
        if type(self.blocks[self.order[index].layer]) is not PreNormBlock:
            return
        for args in self.calls_of(index):
            if library.listening():
                library._heard.calls.append((None, "entry", self.entry, args, True))
            self.entry(*args)

    def step(self):
        alike = AlikeRuns(self.blocks, self.order, self.views)
        index = 0
        while index < len(self.order):
            index = alike.go(index, self.stream, self.forward)
        made, self.seen = self.seen, []
        for index in range(len(self.order)):
            if type(self.blocks[self.order[index].layer]) is PreNormBlock:
                for args in self.calls_of(index):
                    self.entry(*args)
        assert made == self.seen      # what every run's parts would have called
        return self.through


def test_runs_that_share_a_tensor_are_no_record_for_others():
    """What two runs share (their sinks, which a structure names) is not what a run of another layer must be given."""
    blocks = [block() for _ in range(9)]
    assert Launches(blocks, [RunSpec(layer) for layer in (0, 1, 1, 2, 3, 4, 5, 6, 7, 8)]).step() == list(range(10))
    blocks[2].mixer.sink = blocks[1].mixer.sink
    assert Launches(blocks, [RunSpec(layer) for layer in range(9)]).step() == list(range(9))


def test_a_structure_that_names_a_tensor_of_a_run_is_no_record():
    weight, extents = torch.zeros(64), [256]
    at = weight.data_ptr()
    for inside in (at, at + 8, at + 255):
        same = [("library", "entry", "function", (P(at), ctypes.byref(Sunk(inside, 2.0))), True)]
        other = [("library", "entry", "function", (P(at + 4096), ctypes.byref(Sunk(inside, 2.0))), True)]
        assert AlikeRuns._places([same, other], [at], [at + 4096], extents) is None
        same, other = ([("library", "entry", "function", (P(first), P(inside + 4096)), True)] for first in (at, at + 4096))
        assert AlikeRuns._places([same, other], [at], [at + 4096], extents) is None
    beside = [[("library", "entry", "function", (P(first), P(at + 256), ctypes.byref(Sunk(at - 8, 2.0))), True)] for first in (at, at + 4096)]
    assert AlikeRuns._places(beside, [at], [at + 4096], extents) is not None


def test_layers_without_sinks_are_launched_from_the_record():
    blocks = [block() for _ in range(9)]
    for b in blocks:
        b.mixer.sink = blocks[0].mixer.sink.new_zeros(4)
    launches = Launches(blocks, [RunSpec(layer) for layer in range(9)])
    launches.calls_of = lambda index: Launches.calls_of(launches, index)[1:]
    assert launches.step() == [0, 1, 2, 8]      # (the last run is left to its parts)


@pytest.mark.parametrize("kinds", [[2], [3], [5, 8]])
def test_a_block_of_another_kind_behind_alike_runs(kinds):
    """Its norms have other names, and nobody asks it for theirs."""
    blocks = [block() if layer not in kinds else made(ParallelBlock, norm=made(RMSNorm, weight=torch.zeros(4))) for layer in range(10)]
    for b in blocks:
        if type(b) is PreNormBlock:
            del b.mixer.sink
    launches = Launches(blocks, [RunSpec(layer) for layer in range(10)])
    launches.calls_of = lambda index: [(P(7), P(blocks[index].mixer.qkv.weight.data_ptr()))]
    through = launches.step()
    assert through == {2: [0, 1, 2, 3, 4, 9], 3: list(range(10)), 5: [0, 1, 2, *range(4, 10)]}[kinds[0]]


def without_sinks():
    blocks = [block() for _ in range(9)]
    for b in blocks:
        del b.mixer.sink
    launches = Launches(blocks, [RunSpec(layer) for layer in range(9)])
    launches.calls_of = lambda index: [(P(7), P(blocks[index].mixer.qkv.weight.data_ptr()))]
    return blocks, launches


@pytest.mark.parametrize("kind", ["arrays", "tensors", "array and none"])
def test_attributes_that_cannot_be_compared_leave_the_runs_to_their_parts(kind):
    """Whatever somebody keeps at a block: a comparison that has no answer is no error of the step."""
    blocks, launches = without_sinks()
    for layer, b in enumerate(blocks):
        b.mixer.note = {"arrays": lambda: np.arange(3), "tensors": lambda: [torch.arange(3)],
                        "array and none": lambda: np.arange(3) if layer != 4 else None}[kind]()
    assert launches.step() == list(range(9))


@pytest.mark.parametrize("place", ["block", "mixer", "norm"])
def test_a_method_replaced_at_every_block_is_called_for_every_block(place):
    """The same function put in a method's place at all of them: nothing else tells them apart."""
    blocks, launches = without_sinks()
    of = {"block": (lambda b: b, "forward"), "mixer": (lambda b: b.mixer, "attend"), "norm": (lambda b: b.mixer_norm, "apply")}[place]
    watched = lambda *args, **kw: None
    for b in blocks:
        setattr(of[0](b), of[1], watched)
    assert launches.step() == list(range(9))
