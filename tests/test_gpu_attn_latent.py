"""Attention over latent rows that all heads share (``pulse_attn_latent``), against the same sums in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F64 = torch.float64


class Entry:
    def __init__(self, first_row, count):
        self.first_row, self.count = first_row, count


def rnd(*shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16)


def attend(q, rows, spans, nq, d, wv, page=16, splits=1, window=0, sink=None, cap=0.0, scale=0.25, skip=()):
    """``rows``: the stored rows [n, d] of every request, ``spans`` its last tokens that ask; page numbers dealt out at random,
    what was never stored is NaN.  Requests in ``skip`` have rows in the step that no item holds."""
    from pulse_infer_amd.ops import kernels

    width = max((len(r) + page - 1) // page for r in rows)
    order = torch.randperm(len(rows) * width, generator=torch.Generator().manual_seed(9)).view(len(rows), width)
    kc = torch.full((len(rows) * width, 1, page, d), float("nan"), dtype=torch.bfloat16)
    vc = torch.full((len(rows) * width, 1, d, page), float("nan"), dtype=torch.bfloat16)
    for i, r in enumerate(rows):
        for j in range(len(r)):
            kc[order[i, j // page], 0, j % page] = r[j]
            vc[order[i, j // page], 0, :, j % page] = r[j]
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    entries, positions, entry = [], [], []
    for i, (r, n) in enumerate(zip(rows, spans)):
        if i not in skip:
            entries.append(Entry(len(positions), n))
        positions += range(len(r) - n, len(r))
        entry += [i] * n
    flat, hp = kernels.attn_latent_items(entries, nq)
    tokens = len(positions)
    out = torch.full((tokens, nq * d), 7.0, device=DEV)
    part = torch.full((len(flat) // 4 * kernels.LATENT_ROWS * splits, wv), float("nan"), device=DEV)
    ml = torch.full((part.shape[0], 2), float("nan"), device=DEV)
    kernels.attn_latent(q.to(DEV), out, nq, d, wv, kc.to(DEV), vc.to(DEV), ints(positions), ints(entry),
                        order.to(torch.int32).to(DEV).contiguous(), ints(flat), hp, scale, window,
                        None if sink is None else sink.to(DEV), cap, splits, part, ml, several=max(flat[1::4]) > 1)
    return out.cpu().view(tokens, nq, d)


def expected(q, rows, spans, nq, d, wv, window=0, sink=None, cap=0.0, scale=0.25):
    want, size, at = [], [], 0
    for r, n in zip(rows, spans):
        for k in range(n):
            p = len(r) - n + k
            low = max(0, p - window + 1) if window else 0
            keys = r[low:p + 1].to(F64)
            s = q[at].to(F64).view(nq, d) @ keys.T * scale
            if cap:
                s = cap * torch.tanh(s / cap)
            m = s.amax(-1, keepdim=True)
            e = torch.exp(s - m)
            total = e.sum(-1, keepdim=True)
            if sink is not None:
                total = total + torch.exp(sink.to(F64).view(nq, 1) - m)
            want.append(e / total @ keys[:, :wv])
            size.append(e / total @ keys[:, :wv].abs())
            at += 1
    return torch.stack(want), torch.stack(size)


CASES = [
    # heads, stored, values, page, lengths, tokens that ask, splits, window, cap, sink
    (32, 576, 512, 16, [1, 64, 65, 200], [1, 1, 1, 1], 1, 0, 0.0, False),
    (32, 576, 512, 16, [129, 16, 700], [1, 1, 1], 5, 0, 0.0, True),
    (32, 576, 512, 32, [129, 16, 300], [1, 3, 40], 3, 0, 0.0, False),
    (64, 576, 512, 16, [333, 90], [2, 1], 64, 0, 20.0, False),
    (16, 576, 448, 16, [70, 131, 40], [7, 1, 40], 1, 50, 0.0, True),
    (20, 400, 384, 48, [70, 131], [7, 1], 2, 33, 0.0, False),
    (4, 288, 272, 16, [300, 300, 17], [1, 9, 17], 4, 0, 0.0, True),
    (3, 32, 16, 16, [65, 1], [65, 1], 1, 0, 0.0, False),
]


@pytest.mark.parametrize("nq,d,wv,page,lengths,spans,splits,window,cap,sunk", CASES)
def test_attention_over_latent_rows(nq, d, wv, page, lengths, spans, splits, window, cap, sunk):
    """Blocks of 64 keys that end inside, on and behind their edge, shares without a block, items of several tokens and of
    part of the heads, widths that fill no piece."""
    rows = [rnd(n, d, seed=i) for i, n in enumerate(lengths)]
    q = rnd(sum(spans), nq * d, seed=50)
    sink = torch.randn(nq, generator=torch.Generator().manual_seed(3)) if sunk else None
    scale = 2.0 * d ** -0.5
    got = attend(q, rows, spans, nq, d, wv, page, splits, window, sink, cap, scale)
    want, size = expected(q, rows, spans, nq, d, wv, window, sink, cap, scale)
    # weights rounded to bfloat16 (2^-9 each, their sum unrounded), sums and exponentials in float32
    assert ((got[..., :wv].to(F64) - want).abs() <= 2.0 ** -8 * size + 1e-4).all(), float((got[..., :wv].to(F64) - want).abs().max())
    assert (got[..., wv:] == 7.0).all()


def test_rows_that_no_item_holds_stay_as_they_are():
    nq, d, wv = 32, 576, 512
    rows, spans = [rnd(n, d, seed=i) for i, n in enumerate([80, 300, 90])], [1, 5, 1]
    q = rnd(sum(spans), nq * d, seed=50)
    got = attend(q, rows, spans, nq, d, wv, splits=3, skip=(1,), scale=0.05)
    want, size = expected(q, rows, spans, nq, d, wv, scale=0.05)
    assert (got[1:6] == 7.0).all()
    for t in (0, 6):
        assert ((got[t, :, :wv].to(F64) - want[t]).abs() <= 2.0 ** -8 * size[t] + 1e-4).all()


def test_a_value_that_is_not_a_number_is_not_hidden():
    """A NaN among the keys that a token sees makes its row NaN, also where its share weighs nothing beside the others."""
    nq, d, wv, n = 32, 576, 512, 512
    rows = [rnd(n, d, seed=1), rnd(n, d, seed=2)]
    rows[1][5, 3] = float("nan")
    q = rnd(2, nq * d, seed=3)
    for splits in (1, 4):
        got = attend(q, rows, [1, 1], nq, d, wv, splits=splits)
        assert not torch.isnan(got[0, :, :wv]).any() and torch.isnan(got[1, :, :wv]).all()


@pytest.mark.parametrize("odd", [float("nan"), float("inf")])
@pytest.mark.parametrize("nq,d,wv,span,splits,window", [(16, 576, 512, 2, 1, 0), (16, 576, 512, 7, 3, 20), (4, 320, 256, 11, 1, 20),
                                                        (4, 576, 512, 16, 2, 0), (1, 288, 256, 40, 1, 0), (32, 576, 512, 3, 1, 20)])
def test_a_value_that_is_not_finite_stays_with_the_tokens_that_see_it(nq, d, wv, span, splits, window, odd):
    """Tokens that share a workgroup with one that sees it and do not see it themselves: of its own position, of one before them
    that their window has left behind, of one that nobody's window holds any more."""
    n = 131
    for place in (n - 1, n - span + 1, n - span // 2, *((n - span - window + 2, n - span - window) if window else ())):
        rows = [rnd(n, d, seed=1), rnd(n - 3, d, seed=2)]
        rows[0][place, 5] = odd
        q = rnd(2 * span, nq * d, seed=3)
        scale = 2.0 * d ** -0.5
        got = attend(q, rows, [span, span], nq, d, wv, splits=splits, window=window, scale=scale)[..., :wv].to(F64)
        want, size = expected(q, rows, [span, span], nq, d, wv, window=window, scale=scale)
        hit = [place <= p and not (window and p - place >= window) for p in range(n - span, n)] + [False] * span
        assert torch.isfinite(want).all((1, 2)).tolist() == [not h for h in hit]
        assert torch.equal(torch.isfinite(got), torch.isfinite(want)), place     # (a score of minus infinity spoils its channel alone)
        rest = torch.isfinite(want)
        assert ((got - want).abs() <= 2.0 ** -8 * size + 1e-4)[rest].all(), place
