"""What makes two runs' calls a record that other runs can be launched from."""
import ctypes

import pytest

from pulse_infer_amd.models.alike import AlikeRuns

P, I, F = ctypes.c_void_p, ctypes.c_int, ctypes.c_float


class Pair(ctypes.Structure):
    _fields_ = [("a", ctypes.c_int), ("b", ctypes.c_float)]


def calls(weight, number=3, factor=0.5, name="entry", pair=(1, 2.0), clean=True, kind=I):
    lib, entry = "library", "function"
    return [(lib, name, entry, (P(7), P(weight), kind(number), F(factor), None, P(0), ctypes.byref(Pair(*pair))), clean),
            (lib, "second", entry, (P(weight + 64), P(weight)), clean)]


FIRST, SECOND = [100, 164, 300], [200, 264, 400]      # where the runs' tensors lie


def test_the_second_runs_arguments_take_the_tensors_of_others():
    second = calls(200)
    places = AlikeRuns._places([calls(100), second], FIRST, SECOND)
    assert [[i for _, i in own] for *_, own in places] == [[0], [1, 0]]
    for *_, own in places:
        for arg, i in own:
            arg.value = [1000, 1064, 1300][i]
    assert second[0][3][1].value == 1000 and second[1][3][0].value == 1064 and second[0][3][0].value == 7


@pytest.mark.parametrize("other", [dict(weight=201), dict(number=4), dict(factor=0.25), dict(name="another"), dict(pair=(1, 3.0)),
                                   dict(clean=False), dict(weight=100), dict(kind=ctypes.c_int64)])
def test_calls_that_differ_in_more_than_tensors_are_no_record(other):
    assert AlikeRuns._places([calls(100), calls(**{"weight": 200, **other})], FIRST, SECOND) is None


def test_no_record_where_calls_are_missing_or_places_are_shared():
    assert AlikeRuns._places([calls(100), calls(200)[:1]], FIRST, SECOND) is None
    assert AlikeRuns._places([calls(100), calls(200)], [100, 164, 100], SECOND) is None
    assert AlikeRuns._places([calls(100), calls(100)], FIRST, FIRST) is not None     # (the same tensors: any run's fit)
