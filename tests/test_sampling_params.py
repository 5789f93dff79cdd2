"""Sampling options and the per-request random numbers (CPU)."""
import pytest

from pulse_infer_amd.sampling.params import SamplingParams, uniform_for


def test_uniform_numbers_depend_only_on_seed_and_counter():
    a = [uniform_for(7, i) for i in range(2000)]
    assert a == [uniform_for(7, i) for i in range(2000)]
    assert all(0.0 <= u < 1.0 for u in a)
    assert abs(sum(a) / len(a) - 0.5) < 0.03 and len(set(a)) > 1990
    assert a[:5] != [uniform_for(8, i) for i in range(5)]
    # neighbouring seeds and counters are not correlated in the obvious way
    assert len({uniform_for(s, 0) for s in range(100)}) == 100


def test_options_are_checked():
    assert SamplingParams().greedy and not SamplingParams(temperature=0.7).greedy
    assert SamplingParams(temperature=-1.0).greedy
    for bad in (dict(top_k=-1), dict(top_p=1.5), dict(top_p=-0.1), dict(presence_penalty=-1.0)):
        with pytest.raises(ValueError):
            SamplingParams(**bad)


def test_a_steps_options_as_the_kernels_read_them():
    """Rows with and without seeds of their own, counters and seeds of any sign and size: the same uniform numbers as one by one."""
    import struct

    import torch

    from pulse_infer_amd.ops import kernels
    from pulse_infer_amd.ops.library import KernelError

    params = [SamplingParams(), SamplingParams(temperature=0.7, seed=-3), SamplingParams(temperature=1.5, top_k=40, top_p=0.9, seed=2 ** 80 + 5),
              SamplingParams(temperature=0.8, top_p=1.0), SamplingParams(temperature=1e39, top_k=1, presence_penalty=1.5, seed=0)]
    slots, counters, seeds = range(3, 8), [0, 7, -2, 2 ** 40, 123456789], [11, 12, 13, -(2 ** 70) - 1, 15]
    host = torch.full((6, 9), -77, dtype=torch.int32)
    packed = [p.packed for p in params]
    assert kernels.sample_options(host, None, packed, slots, counters, seeds) == (True, True, True)
    single = lambda v: struct.unpack("f", struct.pack("f", v))[0]
    floats = host.view(torch.float32)
    assert floats[0, :5].tolist() == [0.0, single(0.7), 1.5, single(0.8), float("inf")]
    assert host[1, :5].tolist() == [0, 0, 40, 0, 1] and floats[2, :5].tolist() == [0.0, 0.0, single(0.9), 1.0, 0.0]
    assert floats[3, :5].tolist() == [uniform_for(p.seed if p.seed is not None else d, c) for p, c, d in zip(params, counters, seeds)]
    assert floats[4, :5].tolist() == [0.0] * 4 + [1.5] and host[5, :5].tolist() == [-1] * 4 + [7]
    assert (host[:, 5:] == -77).all()                       # nothing beside the rows
    some = lambda *i: kernels.sample_options(host, None, [packed[j] for j in i], [0] * len(i), [0] * len(i), [0] * len(i))
    assert some(0, 3) == (False, False, False) and some(1, 4) == (True, False, True)
    assert kernels.sample_options(host, None, [], [], [], []) == (False, False, False)
    for bad in (lambda: kernels.sample_options(host[:, :4].contiguous(), None, packed, slots, counters, seeds),
                lambda: kernels.sample_options(host, None, packed, slots, counters[:4], seeds),
                lambda: kernels.sample_options(host, None, packed, slots, counters, seeds[:2]),
                lambda: kernels.sample_options(host.float(), None, packed, slots, counters, seeds)):
        with pytest.raises(KernelError):
            bad()


def test_options_for_other_than_a_steps_rows_are_refused():
    """What the kernels read of a row is the row's own: fewer or more options than rows are an error, one may stand for all."""
    import torch

    from pulse_infer_amd.sampling.sampler import Sampler, one_a_row

    sampler, drawn = Sampler(100, 4, torch.device("cpu")), SamplingParams(temperature=0.7, presence_penalty=1.0)
    for params, slots, counters, seeds in (([drawn] * 3, range(4), [0] * 4, [0] * 4), ([drawn] * 5, range(5), [0] * 5, [0] * 5),
                                           ([drawn] * 4, range(3), [0] * 4, [0] * 4), ([drawn] * 4, range(4), [0] * 2, [0] * 4),
                                           ([drawn] * 4, range(4), [0] * 4, [])):
        with pytest.raises(ValueError, match="sampling"):
            sampler.launch(torch.zeros(4, 100), params, slots, counters, seeds)
    assert one_a_row([drawn], 3, "options") == [drawn] * 3 and one_a_row([7], 1, "seeds") == [7]
    assert list(one_a_row(range(5), 4, "slots")) == [0, 1, 2, 3, 4]      # (those behind the rows are not read)


def test_options_that_were_stored_field_by_field_can_be_drawn_with():
    """Objects that were pickled before requests packed their options, or copied: the same row."""
    import copy
    import pickle

    made = SamplingParams(temperature=0.7, top_k=5, seed=3)
    stored = SamplingParams.__new__(SamplingParams)
    stored.__dict__.update(temperature=0.7, top_k=5, top_p=0.0, presence_penalty=0.0, seed=3, ignore_eos=False)
    assert stored == made and stored.packed == made.packed == pickle.loads(pickle.dumps(made)).packed == copy.copy(made).packed
    assert hash(stored) == hash(made)
