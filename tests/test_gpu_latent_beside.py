"""Decoded tokens over latent rows, alone and beside portions whose keys are expanded: both kernels that take them, and over how many
workgroups their keys are shared out."""
import inspect

import pytest
import torch

from plain import sosuvik_plain as P
from test_gpu_sosuvik import config, latent, new_runner

pytestmark = pytest.mark.gpu
TOL = 4e-2


@pytest.fixture(scope="module", params=[(256, 32), (576, 32)], ids=["288 channels", "608 channels"])
def model(request, tmp_path_factory):
    """Two layers of latent attention alone, rows as wide as given (those of 608 are left to the kernel for wide values)."""
    from pulse_infer_amd.config import SosuvikConfig
    from pulse_infer_amd.weights import write_model_folder

    rank, turned = request.param
    layers = [{"type": kind, "mixer": mixer, "mlp": None} for kind, mixer in
              (latent(heads, 64, turned, 64, rank, 1e4, 0.12) for heads in (8, 3))]
    folder = write_model_folder(SosuvikConfig.from_dict(config(300, 256, 1e-6, 2.0, None, layers)),
                                str(tmp_path_factory.mktemp("latent") / "m"), seed=5)
    return rank, folder, P.PlainSosuvik.from_folder(folder)


def test_decoded_tokens_beside_expanded_portions(model, monkeypatch):
    """Every logit against the plain model; no more shares of a decoded token's keys than it has blocks, however long the
    portion's context is."""
    from pulse_infer_amd.engine.runner import StepEntry
    from pulse_infer_amd.ops import kernels

    rank, folder, oracle = model
    taken = []

    def heard(name):
        real = getattr(kernels, name)
        says = inspect.signature(real)

        def call(*args, **kw):
            taken.append((name, says.bind(*args, **kw).arguments.get("n_splits", 1)))
            return real(*args, **kw)

        monkeypatch.setattr(kernels, name, call)

    heard("attn_latent")
    heard("attn_wide")
    runner = new_runner(folder, "bfloat16", 16, 1536)
    lengths = {"a": 821, "b": 62, "c": 321}
    gen = torch.Generator().manual_seed(3)
    ids = {k: torch.randint(0, 300, (n,), generator=gen).tolist() for k, n in lengths.items()}
    steps = [{"b": 40, "c": 299}, {"b": 1, "a": 700}, {"b": 20, "a": 120, "c": 20}, {"b": 1, "a": 1, "c": 1}, {"c": 1}]
    fed, got, shares = {k: 0 for k in ids}, {k: [] for k in ids}, []
    for k in ids:
        runner.add_request(k)
    for step in steps:
        for k, n in step.items():
            runner.reserve(k, fed[k] + n)
        taken.clear()
        logits = runner.step([StepEntry(k, ids[k][fed[k]:fed[k] + n], list(range(n))) for k, n in step.items()])
        shares.append(sorted(set(taken)))
        row = 0
        for k, n in step.items():
            got[k].append(logits[row:row + n].double().cpu())
            fed[k], row = fed[k] + n, row + n
    assert fed == lengths
    for k in ids:
        want = oracle.logits(ids[k])
        assert float((torch.cat(got[k]) - want).abs().max()) <= TOL * max(1.0, float(want.abs().max())), k
    if rank == 256:
        # 40 tokens; one at 41 keys beside 700; 20 each at up to 61 and 319 beside 120 of 820: shares of one, one, five blocks
        assert shares[0] == shares[1] == [("attn_latent", 1)] and {n for _, n in shares[2]} <= set(range(1, 6))
        assert all(name == "attn_latent" for step in shares for name, _ in step)
    else:
        # (its merge covers every row of a step, so beside an expanded portion its keys stay whole)
        assert shares[:3] == [[("attn_wide", 1)]] * 3
    assert any(n > 1 for _, n in shares[-1]) or not shares[-1]
