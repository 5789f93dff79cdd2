"""Attention over wide values with its keys shared out over workgroups: what the merge of their sums keeps."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F64 = torch.float64


class Token:
    def __init__(self, first_row):
        self.first_row, self.count = first_row, 1


def attend(q, ks, vs, nq, d, wv, splits, sink=None):
    """Every request's last token over its keys [requests, n, d] and values."""
    from pulse_infer_amd.ops import kernels

    requests, n = ks.shape[:2]
    page, pages = 16, (n + 15) // 16
    kc = torch.zeros(requests * pages, 1, page, d, dtype=torch.bfloat16)
    vc = torch.zeros(requests * pages, 1, d, page, dtype=torch.bfloat16)
    for r in range(requests):
        for j in range(n):
            kc[r * pages + j // page, 0, j % page] = ks[r, j]
            vc[r * pages + j // page, 0, :, j % page] = vs[r, j]
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    flat, hp = kernels.attn_wide_items([Token(i) for i in range(requests)], nq, 1, 1)
    out = torch.full((requests, nq * d), float("nan"), device=DEV)
    part = torch.full((requests * nq * splits, d), float("nan"), device=DEV)
    ml = torch.full((requests * nq * splits, 2), float("nan"), device=DEV)
    kernels.attn_wide(q.to(DEV), out, nq, 1, d, wv, False, kc.to(DEV), vc.to(DEV), ints([n - 1] * requests),
                      ints(list(range(requests))), torch.arange(requests * pages, dtype=torch.int32, device=DEV).view(requests, pages),
                      ints(flat), hp, 0.25, sink=None if sink is None else sink.to(DEV), n_splits=splits, part=part, part_ml=ml)
    return out.cpu().view(requests, nq, d)[..., :wv]


def rnd(*shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16)


@pytest.mark.parametrize("splits", [2, 7, 8, 9, 64])
def test_merge_of_splits_full_and_empty(splits):
    """More splits than steps of keys leave some without any; numbers of splits round the eight that are read together."""
    requests, n, nq, d, wv = 3, 300, 4, 96, 80
    q, ks, vs, sink = rnd(requests, nq * d, seed=1), rnd(requests, n, d, seed=2), rnd(requests, n, d, seed=3), torch.randn(nq)
    got = attend(q, ks, vs, nq, d, wv, splits, sink).to(F64)
    s = torch.matmul(q.to(F64).view(requests, nq, d), ks.to(F64).transpose(1, 2)) * 0.25
    e = torch.exp(s - s.amax(-1, keepdim=True))
    p = e / (e.sum(-1, keepdim=True) + torch.exp(sink.to(F64).view(1, nq, 1) - s.amax(-1, keepdim=True)))
    want, size = torch.matmul(p, vs.to(F64)), torch.matmul(p, vs.to(F64).abs())
    # weights rounded to bfloat16 (2^-8 with the rounding of their sum), sums and exponentials in float32
    assert ((got - want[..., :wv]).abs() <= 2.0 ** -7 * size[..., :wv] + 1e-4).all()


def test_merge_of_splits_hides_no_value_that_is_not_a_number():
    """A NaN value that a token sees makes its row NaN also where its share of the keys weighs nothing beside the others
    (scores hundreds below), and so does a share whose keys are all NaN; the other requests' rows are numbers."""
    requests, n, nq, d, wv, splits = 3, 512, 4, 64, 64, 4
    q = rnd(requests, nq * d, seed=1)
    q.view(requests, nq, d)[:] = q.view(requests, nq, d)[:, :1]
    ks, vs = rnd(requests, n, d, seed=2), rnd(requests, n, d, seed=3)
    ks[1, :128] = 0.0
    ks[1, 128:] = 40.0 * q[1, :d]
    vs[1, 5, 3] = float("nan")
    ks[2, 128:256] = float("nan")
    out = attend(q, ks, vs, nq, d, wv, splits)
    assert not torch.isnan(out[0]).any()
    assert torch.isnan(out[1, :, 3]).all() and not torch.isnan(out[1, :, :3]).any() and not torch.isnan(out[1, :, 4:]).any()
    assert torch.isnan(out[2]).all()
