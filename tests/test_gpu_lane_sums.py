"""Maxima and sums over a wavefront by lane moves: what the kernels that are made of them choose among equals."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("experts,top", [(5, 2), (64, 8), (200, 6)])
def test_equal_scores_go_to_the_lowest_expert(experts, top):
    """The router's choice over lanes, equal scores in every distance of two lanes; softmax weights sum to one."""
    from pulse_infer_amd.ops import kernels

    rows = 64
    z = torch.zeros(rows, experts)
    for r in range(rows):
        z[r, r % experts] = z[r, (r * 7 + 3) % experts] = 4.0
        z[r, (r * 11 + 1) % experts] = -100.0
    idx = torch.empty(rows, top, dtype=torch.int32, device=DEV)
    weight = torch.empty(rows, top, device=DEV)
    kernels.moe_route(z.to(DEV), None, top, idx, weight)
    assert torch.equal(idx.cpu().long(), torch.sort(z, dim=1, descending=True, stable=True).indices[:, :top])
    assert ((weight.sum(1) - 1.0).abs() <= 2.0 * top * 2.0 ** -24 * 4).all()


@pytest.mark.parametrize("rows", [1, 3, 70])
@pytest.mark.parametrize("vocab", [1, 63, 64, 65, 2049, 5000])
def test_the_largest_of_equal_logits_is_the_first(rows, vocab):
    from pulse_infer_amd.ops import kernels

    logits = torch.randint(0, 3, (rows, vocab), generator=torch.Generator().manual_seed(rows * 10000 + vocab)).float()
    out, chunks = torch.empty(rows, dtype=torch.int32, device=DEV), kernels.argmax_chunks(vocab)
    kernels.argmax(logits.to(DEV), out, torch.empty(rows, chunks, device=DEV), torch.empty(rows, chunks, dtype=torch.int32, device=DEV))
    first = (logits == logits.amax(1, keepdim=True)).int().argmax(1)
    assert torch.equal(out.cpu().long(), first)
