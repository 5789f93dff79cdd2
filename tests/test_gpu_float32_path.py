"""The float32 path's kernels where their tiles end: products of every tile shape and the attention of whole rows."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F64 = torch.float64
U = 2.0 ** -24     # unit roundoff of float32


@pytest.fixture(scope="module")
def k():
    from pulse_infer_amd.ops import kernels
    return kernels


def rnd(*shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed))


# rows x weight rows x K: one and sixteen rows with few and many weight rows; every staged tile (the rule's 2 x 2, 2 x 4,
# 3 x 4 and 4 x 4 blocks), with remainders of rows, weight rows and K; shares of K of no, one and unequal numbers of blocks;
# rows that are no multiple of four, which are read value by value: tiles of 16 x 32, 32 x 32 and 32 x 64, K below one block
@pytest.mark.parametrize("shape", [(1, 100, 4), (1, 16400, 20), (16, 33, 68), (17, 40, 16), (40, 90, 300), (49, 2050, 1028),
                                   (97, 2048, 52), (333, 2048, 100), (333, 5000, 84), (1030, 4100, 36), (65, 70, 257), (1, 33, 3), (130, 1010, 67), (129, 100, 1001), (2050, 2100, 18)])
@pytest.mark.parametrize("types", [(torch.float32, torch.float32, torch.float32), (torch.bfloat16, torch.float32, torch.float32),
                                   (torch.float32, torch.bfloat16, torch.bfloat16)])
def test_float32_product_at_the_edges_of_its_tiles(k, shape, types):
    m, n, kk = shape
    a, w = rnd(m, kk, seed=1).to(types[0]), rnd(n, kk, seed=2).to(types[1])
    out = torch.full((m, n), float("nan"), dtype=types[2], device=DEV)
    k.gemm_f32(a.to(DEV), w.to(DEV), out)
    want, size = a.to(F64) @ w.to(F64).T, a.to(F64).abs() @ w.to(F64).abs().T
    # a sum of K products in float32, in any order: |error| <= (K + 2) u sum |a| |w|; a bfloat16 result is rounded once more
    bound = (kk + 2) * U * size + (2.0 ** -8 * want.abs() if types[2] == torch.bfloat16 else 0.0)
    assert ((out.cpu().to(F64) - want).abs() <= bound).all()
    alone = torch.empty(1, n, dtype=types[2], device=DEV)        # a row by itself: the same sums in the same order
    for row in {0, m // 2, m - 1}:
        k.gemm_f32(a[row:row + 1].to(DEV), w.to(DEV), alone)
        assert torch.equal(alone[0], out[row])


def visible(pos, n, window, keep_first, chunk):
    j = torch.arange(n)
    lo = pos - pos % chunk if chunk else max(0, pos - window + 1) if window else 0
    return (j <= pos) & ((j >= lo) | (j < min(keep_first, lo)))


@pytest.mark.parametrize("d,nq,nkv,page", [(32, 5, 1, 16), (64, 8, 2, 32), (128, 16, 4, 16), (128, 20, 1, 16), (256, 4, 4, 48)])
@pytest.mark.parametrize("form", [dict(), dict(window=37, softcap=3.0, sink=True), dict(window=40, keep_first=5, gate=1),
                                  dict(chunk=48, gate=-1)])
def test_float32_attention_of_whole_rows(k, d, nq, nkv, page, form):
    """Portions and single tokens side by side (tiles that hold tokens of several requests), more than 64 tokens (several a
    tile) and fewer (one a tile); slots that were never written hold NaN, and so does a value that early tokens do not see."""
    group, scale = nq // nkv, 0.3
    portions = [(0, 50), (130, 13), (61, 1), (200, 9)]        # (tokens before, tokens of the step)
    bad = 45                                                  # request 0's key of this position has a NaN value
    window, keep, chunk, cap = (form.get(x, 0) for x in ("window", "keep_first", "chunk", "softcap"))
    width = max((b + n + page - 1) // page for b, n in portions)
    table = torch.full((len(portions), width), -1, dtype=torch.int32)
    order = torch.randperm(width * len(portions), generator=torch.Generator().manual_seed(3)).tolist()
    kc = torch.full((width * len(portions), nkv, page, d), float("nan"))
    vc = torch.full((width * len(portions), nkv, d, page), float("nan"))
    keys, values = [], []
    for e, (before, n) in enumerate(portions):
        total = before + n
        ks, vs = rnd(total, nkv, d, seed=10 + e), rnd(total, nkv, d, seed=20 + e)
        if e == 0:
            vs[bad] = float("nan")
        for p in range((total + page - 1) // page):
            table[e, p] = page_id = order.pop()
            for j in range(p * page, min(total, (p + 1) * page)):
                kc[page_id, :, j % page] = ks[j]
                vc[page_id, :, :, j % page] = vs[j]
        keys.append(ks.to(F64))
        values.append(vs.to(F64))
    positions = [b + i for b, n in portions for i in range(n)]
    entry = [e for e, (b, n) in enumerate(portions) for _ in range(n)]
    tokens = len(positions)
    q = rnd(tokens, nq * d + 4, seed=30)
    sink = rnd(nq, seed=31) if form.get("sink") else None
    gate_width = {0: 0, 1: 0, -1: d // 2}[form.get("gate", 0)]
    gate = rnd(tokens, nq * max(1, gate_width), seed=32) if form.get("gate") else None
    on = lambda t: None if t is None else t.to(DEV)

    def run(rows):
        out = torch.full((len(rows), nq * d), 7.0, device=DEV)
        k.attn_generic(q[rows].to(DEV), out, nq, nkv, d, kc.to(DEV), vc.to(DEV),
                       torch.tensor([positions[i] for i in rows], dtype=torch.int32, device=DEV),
                       torch.tensor([entry[i] for i in rows], dtype=torch.int32, device=DEV), table.to(DEV), scale, window,
                       gate=None if gate is None else gate[rows].to(DEV), gate_width=gate_width, sink=on(sink), softcap=cap,
                       keep_first=keep, chunk=chunk)
        return out.cpu()

    whole = run(list(range(tokens)))
    few = list(range(40, 60))
    assert torch.equal(torch.nan_to_num(run(few), 9.0), torch.nan_to_num(whole[few], 9.0))    # whatever shares the tile
    for t in range(tokens):
        e, p = entry[t], positions[t]
        ks, vs = keys[e], values[e]
        see = visible(p, ks.shape[0], window, keep, chunk)
        qt = q[t, :nq * d].to(F64).view(nkv, group, d)
        s = torch.einsum("ghd,jgd->ghj", qt, ks[see]) * scale
        size = torch.einsum("ghd,jgd->ghj", qt.abs(), ks[see].abs()).max() * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        top = s.amax(-1, keepdim=True)
        den = torch.exp(s - top).sum(-1, keepdim=True)
        if sink is not None:
            den = den + torch.exp(sink.to(F64).view(nkv, group, 1) - top)
        want = torch.einsum("ghj,jgd->ghd", torch.exp(s - top) / den, vs[see]).reshape(nq, d)
        if gate is not None:
            g = torch.sigmoid(gate[t].to(F64)).view(nq, -1)
            want = want * g if not gate_width else torch.cat([want[:, :gate_width] * g, want[:, gate_width:]], -1)
        got = whole[t].to(F64).view(nq, d)
        if torch.isnan(vs[see]).any():
            assert torch.isnan(got).all()
            continue
        # scores are off by (d + 8) u of their terms' sizes at most, weights by twice that, sums of weighted values by one
        # more rounding a key and a handful for the exponentials and the gate
        bound = (2 * (d + 8) * U * float(size) + (int(see.sum()) + 64) * U) * float(vs[see].abs().max())
        assert float((got - want).abs().max()) <= bound, (t, e, p)


@pytest.mark.parametrize("requests", [65, 1100])
def test_float32_attention_of_many_requests_at_once(k, requests):
    """A step of single tokens whose tiles hold sixteen requests each, with a workgroup a request and, where the chip has no room
    for that many, with several each; portions of two tokens among them."""
    nq, d, page = 8, 32, 16
    gen = torch.Generator().manual_seed(4)
    last = torch.randint(1, 3 * page, (requests,), generator=gen)
    counts = [2 if i % 7 == 3 else 1 for i in range(requests)]
    entry = [i for i, c in enumerate(counts) for _ in range(c)]
    positions = [int(last[i]) - c + 1 + j for i, c in enumerate(counts) for j in range(c)]
    ks, vs = rnd(requests, 3 * page, nq, d, seed=5), rnd(requests, 3 * page, nq, d, seed=6)
    q = rnd(len(entry), nq * d, seed=7)
    kc = ks.view(requests * 3, page, nq, d).transpose(1, 2).contiguous()
    vc = vs.view(requests * 3, page, nq, d).permute(0, 2, 3, 1).contiguous()
    out = torch.full((len(entry), nq * d), 7.0, device=DEV)
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    k.attn_generic(q.to(DEV), out, nq, nq, d, kc.to(DEV), vc.to(DEV), ints(positions), ints(entry),
                   torch.arange(requests * 3, dtype=torch.int32, device=DEV).view(requests, 3), 0.3)
    e, p = torch.tensor(entry), torch.tensor(positions)
    s = (q.view(-1, 1, nq, d).to(F64) * ks[e].to(F64)).sum(-1) * 0.3                       # [tokens, keys, heads]
    s = s.masked_fill((torch.arange(3 * page).view(1, -1) > p.view(-1, 1)).unsqueeze(-1), float("-inf"))
    want = (torch.softmax(s, 1).unsqueeze(-1) * vs[e].to(F64)).sum(1).reshape(len(entry), nq * d)
    size = float((q.view(-1, 1, nq, d).abs() * ks[e].abs()).sum(-1).max()) * 0.3
    # (as above: scores off by (d + 8) u of their size, weights by twice that, a rounding a key and some for the exponentials)
    bound = (2 * (d + 8) * U * size + (3 * page + 64) * U) * float(vs.abs().max())
    assert float((out.cpu().to(F64) - want).abs().max()) <= bound


@pytest.mark.parametrize("tokens", [1, 70])
def test_float32_attention_hides_no_value_that_is_not_a_number(k, tokens):
    """A query that is NaN, sixteen keys in a row that are (all that one wavefront sees of a request), and a value that is one
    whose weight is nothing beside the others': what a token sees of them makes its row NaN, and no other."""
    nq, nkv, d, page, before = 2, 1, 64, 16, 63
    total = before + tokens
    pages = (total + page - 1) // page
    q = rnd(tokens, nq * d, seed=1)
    ks, vs = rnd(3, total, d, seed=2), rnd(3, total, d, seed=3)
    ks[1, 32:48] = float("nan")                   # request 1: every key of the third block
    ks[2, :16] = 0.0
    ks[2, 16:] = 40.0 * q[0, :d]                  # request 2: its first block's scores lie hundreds below the others
    q[:, d:] = q[:, :d]
    q[1:] = q[0]
    vs[2, 5] = float("nan")
    kc = torch.zeros(3 * pages, nkv, page, d)
    vc = torch.zeros(3 * pages, nkv, d, page)
    for r in range(3):
        for j in range(total):
            kc[r * pages + j // page, 0, j % page] = ks[r, j]
            vc[r * pages + j // page, 0, :, j % page] = vs[r, j]
    table = torch.arange(3 * pages, dtype=torch.int32).view(3, pages)

    def run(entry, queries):
        out = torch.full((tokens, nq * d), 7.0, device=DEV)
        k.attn_generic(queries.to(DEV), out, nq, nkv, d, kc.to(DEV), vc.to(DEV),
                       torch.arange(before, total, dtype=torch.int32, device=DEV),
                       torch.full((tokens,), entry, dtype=torch.int32, device=DEV), table.to(DEV), 1.0)
        return out.cpu().view(tokens, nq, d)

    assert not torch.isnan(run(0, q)).any()
    bad = q.clone()
    bad[tokens - 1, d:] = float("nan")            # (the last token's second head)
    out = run(0, bad)
    assert torch.isnan(out[-1, 1]).all() and not torch.isnan(out[-1, 0]).any() and not torch.isnan(out[:-1]).any()
    assert torch.isnan(run(1, q)).all()
    assert torch.isnan(run(2, q)).all()
