"""Runs launched from their neighbours' record: the bits of the same steps through their parts, and where the parts are kept to."""
import pytest
import torch

from conftest import TINY_B

pytestmark = pytest.mark.gpu

SIZES = dict(TINY_B, hidden_size=256, intermediate_size=512, num_hidden_layers=11, num_attention_heads=8, num_key_value_heads=2,
             head_dim=32, vocab_size=300)


def built(**changes):
    from pulse_infer_amd.config import Qwen3Config
    from pulse_infer_amd.models.causal_lm import expected_tensors
    from pulse_infer_amd.models.factory import build_model
    from pulse_infer_amd.weights.random_init import RandomSource

    cfg = Qwen3Config.from_dict(dict(SIZES, **changes))
    return build_model(cfg, RandomSource(expected_tensors(cfg.model_spec()), seed=3), mode="bfloat16")


FEW_ROWS = ([("a", 40)], [("a", 1), ("b", 33)], [("a", 1), ("b", 1), ("c", 17)], [("d", 60)], [("a", 5), ("b", 20), ("d", 1)])
MORE_ROWS = ([("a", 97)], [("a", 1), ("b", 128)], [("c", 192)], [("a", 20), ("c", 45)])      # 97, 129, 192 and 65


def steps(model, plan=FEW_ROWS):
    """Logits of a prompt, of portions beside decoded tokens and of another prompt, at 17 to 64 rows; pages dealt out anew."""
    from pulse_infer_amd.engine.runner import ModelRunner, StepEntry

    runner = ModelRunner(model, page_size=16, num_pages=40, max_requests=4)
    token = lambda i, n: [(7 * i + 13 * k) % 300 for k in range(n)]
    out, fed = [], {}
    for entries in plan:
        made = []
        for name, n in entries:
            if name not in fed:
                runner.add_request(name)
                fed[name] = 0
            runner.reserve(name, fed[name] + n)
            made.append(StepEntry(name, token(fed[name], n), [n - 1]))
            fed[name] += n
        out.append(runner.step(made).cpu())
    return out


def counted(monkeypatch, model, on, plan=FEW_ROWS):
    from pulse_infer_amd.models import alike
    from pulse_infer_amd.ops import library

    calls = []
    was = library._invoke
    with monkeypatch.context() as patch:
        patch.setattr(library, "_invoke", lambda lib, name, args: (calls.append(name), was(lib, name, args)))
        if not on:
            patch.setattr(alike, "MIN_RUNS", 10 ** 6)
        return steps(model, plan), len(calls)


def test_alike_runs_give_the_bits_of_their_parts(monkeypatch):
    model = built()
    recorded, few = counted(monkeypatch, model, True)
    through, many = counted(monkeypatch, model, False)
    assert few < 0.6 * many          # runs 3 .. 9 of eleven
    for a, b in zip(recorded, through):
        assert torch.equal(a, b)


@pytest.mark.parametrize("change", ["scale", "eps", "new attribute", "weight's place", "weight's type", "window"])
def test_a_run_that_is_not_alike_goes_through_its_parts(monkeypatch, change):
    """A layer changed after the model was built, in any of the ways a record would not see."""
    model = built()
    mixer, norm = model.blocks[6].mixer, model.blocks[6].ffn_norm
    if change == "scale":
        mixer.scale *= 2.0
    elif change == "eps":
        norm.eps = 0.3
    elif change == "new attribute":
        mixer.score_cap = 0.5
    elif change == "window":
        mixer.window = 9
    elif change == "weight's type":
        norm.weight = norm.weight.float()
    else:
        held = torch.empty(norm.weight.numel() + 1, dtype=norm.weight.dtype, device=norm.weight.device)
        held[1:] = norm.weight
        norm.weight = held[1:]
    recorded, few = counted(monkeypatch, model, True)
    through, many = counted(monkeypatch, model, False)
    assert 0.6 * many < few < many   # runs 3 .. 5
    for a, b in zip(recorded, through):
        assert torch.equal(a, b)


def test_weights_replaced_between_steps_are_the_ones_that_are_used(monkeypatch):
    model = built()
    first = steps(model)
    for block in model.blocks:
        block.ffn.down.weight = (block.ffn.down.weight * 0.5).contiguous()
    recorded, _ = counted(monkeypatch, model, True)
    through, _ = counted(monkeypatch, model, False)
    assert all(torch.equal(a, b) for a, b in zip(recorded, through)) and not torch.equal(first[0], recorded[0])


def test_projections_in_shares_are_launched_from_a_record(monkeypatch):
    """Layers 4,096 wide at 65 to 192 rows: q, k and v leave their product as shares that the rotation adds up.  The bits of the same
    step through its parts, and the results of the whole product within the rounding of bfloat16."""
    from pulse_infer_amd.parts.linear import Linear

    model = built(hidden_size=4096, num_hidden_layers=9, num_attention_heads=16, num_key_value_heads=8)
    recorded, few = counted(monkeypatch, model, True, MORE_ROWS)
    through, many = counted(monkeypatch, model, False, MORE_ROWS)
    assert few < 0.7 * many          # runs 3 .. 7 of nine
    for a, b in zip(recorded, through):
        assert torch.equal(a, b)
    made = []
    real = Linear.forward_parts
    monkeypatch.setattr(Linear, "forward_parts", lambda self, x, ws: made.append(real(self, x, ws)) or made[-1])
    assert all(torch.equal(a, b) for a, b in zip(steps(model, MORE_ROWS), through))
    assert made and all(parts is not None for parts in made)
    monkeypatch.setattr(Linear, "forward_parts", lambda self, x, ws: None)
    for a, b in zip(through, steps(model, MORE_ROWS)):
        assert not torch.equal(a, b) and float((a - b).abs().max()) <= 4e-2 * float(b.abs().max())


def test_a_rows_projection_does_not_depend_on_the_rows_beside_it():
    from pulse_infer_amd.parts.base import Workspace
    from pulse_infer_amd.parts.linear import Linear

    gen = torch.Generator().manual_seed(11)
    x = torch.randn(256, 4096, generator=gen).to(torch.bfloat16).to("cuda:0")
    linear = Linear((torch.randn(6144, 4096, generator=gen) / 64).to(torch.bfloat16).to("cuda:0"), "bfloat16")
    ws = Workspace(torch.device("cuda:0"))
    want = linear.forward_parts(x[:65], ws).clone()
    for rows in (66, 96, 128, 129, 130, 192, 193, 255, 256):
        assert torch.equal(linear.forward_parts(x[:rows], ws)[:, :65], want), rows
