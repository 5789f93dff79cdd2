"""The router on the matrix cores and the experts' products grouped by expert, where their tiles end."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F64 = torch.float64


def rnd(*shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed))


# rows an expert gets: none, one, a tile of 32, 64, 128 and 192 rows and one more and one less; widths of one step of the loop, of
# several, with a remainder of the tile's columns, and inner widths that are no multiple of 64 (the other kernels)
@pytest.mark.parametrize("hidden,ff", [(64, 64), (320, 192), (192, 136), (200, 64)])
@pytest.mark.parametrize("rows", [32, 64, 128, 192])
@pytest.mark.parametrize("form", ["silu", "clamped_on_input"])
def test_grouped_experts_at_the_edges_of_their_tiles(hidden, ff, rows, form):
    from pulse_infer_amd.ops import kernels

    counts = [0, 1, rows - 1, rows, rows + 1, 2 * rows + 5, 0, 17]
    experts, pairs = len(counts), sum(counts)
    chosen = torch.cat([torch.full((c,), e) for e, c in enumerate(counts)])
    chosen = chosen[torch.randperm(pairs, generator=torch.Generator().manual_seed(1))]
    top = 1
    x = rnd(pairs, hidden, seed=2).to(torch.bfloat16)
    wg, wu = ((rnd(experts, ff, hidden, seed=3 + i) * hidden ** -0.5).to(torch.bfloat16) for i in range(2))
    wd = (rnd(experts, hidden, ff, seed=5) * ff ** -0.5).to(torch.bfloat16)
    weight = torch.rand(pairs, 1, generator=torch.Generator().manual_seed(6)) + 0.5
    idx = chosen.to(torch.int32).view(pairs, 1)
    act = torch.full((pairs, ff), float("nan"), dtype=torch.bfloat16, device=DEV)
    y = torch.full((pairs, hidden), float("nan"), device=DEV)
    out = torch.full((pairs, hidden), float("nan"), device=DEV)
    ints = torch.full((2 * pairs + 3 * kernels.moe_max_tiles(pairs, experts, rows) + 1,), -5, dtype=torch.int32, device=DEV)
    limit = 0.8
    kw = dict(weight_on_input=True, activation="clamped_swish", limit=limit) if form != "silu" else {}
    kernels.moe_grouped(x.to(DEV), wg.to(DEV), wu.to(DEV), wd.to(DEV), idx.to(DEV), weight.to(DEV), act, y, out, ints, rows, **kw)
    xd, e = x.to(F64), chosen
    g = torch.einsum("th,tfh->tf", xd, wg.to(F64)[e])
    u = torch.einsum("th,tfh->tf", xd, wu.to(F64)[e])
    if form == "silu":
        want_act = g * torch.sigmoid(g) * u
    else:
        g, u = (g * weight).clamp(max=limit), (u * weight).clamp(-limit, limit)
        want_act = g * torch.sigmoid(1.702 * g) * (u + 1.0)
    got_act = act.cpu().to(F64)
    # float32 sums of `hidden` products of about 1 / sqrt(hidden) each, through an activation of slope 2 at most, rounded once
    assert ((got_act - want_act).abs() <= 2.0 ** -8 * want_act.abs() + 1e-5 * (1.0 + want_act.abs().max())).all()
    want = torch.einsum("tf,thf->th", got_act, wd.to(F64)[e])          # (of the rounded activations)
    size = torch.einsum("tf,thf->th", got_act.abs(), wd.to(F64)[e].abs())
    if form == "silu":
        want, size = want * weight, size * weight
    assert ((out.cpu().to(F64) - want).abs() <= (ff + 4) * 2.0 ** -24 * size).all()


# one block of outputs for all sixteen wavefronts to share, two, five (two wavefronts a block), nine and seventeen (one, and a
# second round); widths of fewer steps of 32 than wavefronts, of a whole round of eight ahead, of a remainder, of several rounds
@pytest.mark.parametrize("n", [8, 17, 65, 130, 257, 1000])
@pytest.mark.parametrize("hidden", [64, 544, 4096, 4128, 5120])
@pytest.mark.parametrize("tokens", [1, 17])
def test_router_logits_at_the_edges_of_its_blocks(n, hidden, tokens):
    """The scores of every output: a correction that is far above all scores names the outputs that are chosen."""
    from pulse_infer_amd.ops import kernels

    x, w = rnd(tokens, hidden, seed=1).to(torch.bfloat16), (rnd(n, hidden, seed=2) * hidden ** -0.5).to(torch.bfloat16)
    z = x.to(F64) @ w.to(F64).T
    # a float32 sum of `hidden` exact products in any order, through a sigmoid of slope 1/4 and a few roundings of its own
    bound = (hidden + 2) * 2.0 ** -24 * (x.to(F64).abs() @ w.to(F64).abs().T) / 4 + 2.0 ** -21
    top = 8
    order = torch.randperm(n, generator=torch.Generator().manual_seed(3)).tolist()
    for first in range(0, n, top):
        some = (order + order[:top])[first:first + top]
        correction = torch.zeros(n)
        correction[some] = 1024.0
        idx = torch.full((tokens, top), -5, dtype=torch.int32, device=DEV)
        weight = torch.full((tokens, top), float("nan"), device=DEV)
        kernels.moe_router(x.to(DEV), w.to(DEV), correction.to(torch.bfloat16).to(DEV), top, idx, weight, score="sigmoid",
                           renormalize=False)
        got, chosen = weight.cpu().to(F64), idx.cpu().long()
        assert (chosen.sort(1).values == torch.tensor(sorted(some))).all()
        want = torch.sigmoid(z).gather(1, chosen)
        assert ((got - want).abs() <= bound.gather(1, chosen)).all()
        if n > 200 and first >= 8 * top:      # (enough of them to meet every block)
            break


@pytest.mark.parametrize("tokens", [3, 40])
@pytest.mark.parametrize("n, top", [(1, 1), (6, 1), (7, 1), (24, 4), (25, 4), (48, 8), (49, 8), (64, 10), (64, 11), (64, 64)])
def test_equal_outputs_are_chosen_in_their_order(n, top, tokens):
    """Ranked (up to six outputs a choice) and searched for: several outputs of the same weights, the lower number first."""
    from pulse_infer_amd.ops import kernels

    hidden = 256
    x = rnd(tokens, hidden, seed=1).to(torch.bfloat16)
    kinds = (rnd(5, hidden, seed=2) * hidden ** -0.5).to(torch.bfloat16)
    of = torch.randint(0, 5, (n,), generator=torch.Generator().manual_seed(n))
    idx = torch.full((tokens, top), -5, dtype=torch.int32, device=DEV)
    weight = torch.full((tokens, top), float("nan"), device=DEV)
    kernels.moe_router(x.to(DEV), kinds[of].to(DEV), None, top, idx, weight)
    z = (x.to(F64) @ kinds.to(F64).T)[:, of]
    order = z.sort(dim=1, descending=True, stable=True).indices[:, :top]
    assert torch.equal(idx.cpu().long(), order)      # (five values a token, further apart than sums in 32 bits err)
    want = torch.softmax(z, 1).gather(1, order)
    want = want / want.sum(1, keepdim=True)
    assert ((weight.cpu().to(F64) - want).abs() <= 1e-5 * want).all()


@pytest.mark.parametrize("tokens", [1, 7, 16])
@pytest.mark.parametrize("n, experts, top, groups", [(2, 2, 1, (0, 0)), (16, 16, 4, (4, 2)), (64, 61, 8, (0, 0)), (65, 65, 6, (5, 3)),
                                                     (256, 256, 64, (0, 0)), (250, 200, 33, (0, 0))])
def test_router_and_groups_in_one_launch(tokens, n, experts, top, groups):
    """The choices and weights of the router alone, bit by bit; every pair of an expert in one of its places, and tiles that hold an
    expert's places one after the other."""
    from pulse_infer_amd.ops import kernels

    hidden, rows = 288, 32
    x, w = rnd(tokens, hidden, seed=1).to(torch.bfloat16), (rnd(n, hidden, seed=2) * hidden ** -0.5).to(torch.bfloat16)
    correction = (rnd(n, seed=3) * 0.1).to(torch.bfloat16).to(DEV)
    x, w = x.to(DEV), w.to(DEV)
    how = dict(score="sigmoid", renormalize=True, groups=groups, weight_scale=1.5)
    idx, idx1 = (torch.full((tokens, top), -5, dtype=torch.int32, device=DEV) for _ in range(2))
    weight, weight1 = (torch.full((tokens, top), float("nan"), device=DEV) for _ in range(2))
    kernels.moe_router(x, w, correction, top, idx, weight, **how)
    pairs = tokens * top
    tiles = kernels.moe_max_tiles(pairs, experts, rows)
    ints = torch.full((2 * pairs + 3 * tiles + 1,), -9, dtype=torch.int32, device=DEV)
    assert kernels.moe_router_groups(x, w, correction)
    kernels.moe_router_grouped(x, w, correction, top, idx1, weight1, experts, rows, ints, **how)
    assert torch.equal(idx, idx1) and torch.equal(weight, weight1)
    chosen, got = idx.cpu().flatten().tolist(), ints.cpu().tolist()
    order, count = got[pairs:2 * pairs], got[-1]
    t_expert, t_row0, t_rows = (got[2 * pairs + i * tiles:2 * pairs + (i + 1) * tiles][:count] for i in range(3))
    want = {e: sorted(a for a, c in enumerate(chosen) if c == e) for e in set(chosen) if e < experts}
    assert sum(t_rows) == sum(len(v) for v in want.values()) and all(0 < r <= rows for r in t_rows)
    held = {}
    for e, row0, r in zip(t_expert, t_row0, t_rows):
        held.setdefault(e, []).extend(order[row0:row0 + r])
    assert {e: sorted(v) for e, v in held.items()} == want
    assert t_row0 == [sum(t_rows[:i]) for i in range(count)] and t_expert == sorted(t_expert)


def test_grouped_experts_with_room_for_more_pairs_than_offsets_reach():
    """Lists with room for so many pairs that their rows may lie more than 4 GB apart take the kernels that go by pointers."""
    from pulse_infer_amd.ops import kernels

    hidden, ff, experts, pairs, rows = 64, 64, 3, 200, 192
    x = rnd(pairs, hidden, seed=2).to(torch.bfloat16).to(DEV)
    wg, wu = ((rnd(experts, ff, hidden, seed=3 + i) * hidden ** -0.5).to(torch.bfloat16).to(DEV) for i in range(2))
    wd = (rnd(experts, hidden, ff, seed=5) * ff ** -0.5).to(torch.bfloat16).to(DEV)
    idx = (torch.arange(pairs, dtype=torch.int32) % experts).to(DEV)
    few = kernels.moe_max_tiles(pairs, experts, rows)
    many = (1 << 25) // rows + few
    rank, order = (torch.empty(pairs, dtype=torch.int32, device=DEV) for _ in range(2))
    tile_expert, tile_row0, tile_rows = (torch.empty(many, dtype=torch.int32, device=DEV) for _ in range(3))
    num = torch.empty(1, dtype=torch.int32, device=DEV)
    p, i32 = kernels._ptr, kernels._i32
    kernels.call("pulse_moe_group", p(idx), i32(pairs), i32(experts), i32(rows), i32(few), p(rank), p(order), p(tile_expert), p(tile_row0),
                 p(tile_rows), p(num), kernels._stream())
    lists = [p(order), p(tile_expert), p(tile_row0), p(tile_rows), p(num)]
    e = idx.long().cpu()
    g = torch.einsum("th,tfh->tf", x.cpu().to(F64), wg.cpu().to(F64)[e])
    want = g * torch.sigmoid(g) * torch.einsum("th,tfh->tf", x.cpu().to(F64), wu.cpu().to(F64)[e])
    for tiles in (few, many):
        act = torch.full((pairs, ff), float("nan"), dtype=torch.bfloat16, device=DEV)
        kernels.call("pulse_moe_gate_up_grouped", p(x), p(wg), p(wu), *lists, i32(tiles), i32(rows), p(act), i32(hidden), i32(ff), i32(1),
                     p(None), i32(0), kernels._f32(0.0), kernels._stream())
        got = act.cpu().to(F64)
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5 * (1.0 + want.abs().max())).all(), tiles
        y = torch.full((pairs, hidden), float("nan"), device=DEV)
        kernels.call("pulse_moe_down_grouped", p(act), p(wd), *lists, i32(tiles), i32(rows), p(y), i32(hidden), i32(ff), kernels._stream())
        out, size = (torch.einsum("tf,thf->th", a, b) for a, b in ((got, wd.cpu().to(F64)[e]), (got.abs(), wd.cpu().to(F64)[e].abs())))
        assert ((y.cpu().to(F64) - out).abs() <= (ff + 4) * 2.0 ** -24 * size).all(), tiles


def test_grouped_experts_of_tokens_four_gigabytes_apart():
    """A list's tokens up to 4.29 GB behind the first, as far as an offset of 32 bits reaches.  (4 GB in front of them, so that an offset
    taken for a negative one finds other values.)"""
    from pulse_infer_amd.ops import kernels

    hidden, ff, experts, rows = 4096, 64, 2, 192
    pairs = ((1 << 31) - 4096) // hidden - (experts + 1) * rows        # (lists have room for a last tile an expert)
    pairs -= pairs % rows
    few = kernels.moe_max_tiles(pairs, experts, rows)
    assert 2 ** 32 - 2 ** 23 < 2 * pairs * hidden < 2 * (few * rows + 1) * hidden + 8192 < 2 ** 32
    x = torch.empty((1 << 31) + pairs * hidden, dtype=torch.bfloat16, device=DEV)[1 << 31:].view(pairs, hidden).normal_()
    wg, wu = ((rnd(experts, ff, hidden, seed=3 + i) * hidden ** -0.5).to(torch.bfloat16).to(DEV) for i in range(2))
    idx = (torch.arange(pairs, dtype=torch.int32) % experts).to(DEV)
    ints = [torch.empty(n, dtype=torch.int32, device=DEV) for n in (pairs, pairs, few, few, few, 1)]
    act = torch.full((pairs, ff), float("nan"), dtype=torch.bfloat16, device=DEV)
    p, i32 = kernels._ptr, kernels._i32
    kernels.call("pulse_moe_group", p(idx), i32(pairs), i32(experts), i32(rows), i32(few), *(p(t) for t in ints), kernels._stream())
    kernels.call("pulse_moe_gate_up_grouped", p(x), p(wg), p(wu), *(p(t) for t in ints[1:]), i32(few), i32(rows), p(act), i32(hidden),
                 i32(ff), i32(1), p(None), i32(0), kernels._f32(0.0), kernels._stream())
    assert not torch.isnan(act).any()
    some = torch.tensor([0, 1, 191, 192, pairs // 2, pairs // 2 + 1, pairs - 2, pairs - 1])
    xs, e = x[some.to(DEV)].cpu().to(F64), some % experts
    g, u = (torch.einsum("th,tfh->tf", xs, w.cpu().to(F64)[e]) for w in (wg, wu))
    want = g * torch.sigmoid(g) * u
    assert ((act[some.to(DEV)].cpu().to(F64) - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5 * (1.0 + want.abs().max())).all()


@pytest.mark.parametrize("hidden,ff", [(64, 64), (1024, 448)])
@pytest.mark.parametrize("form", ["silu", "clamped_on_input"])
def test_grouped_experts_do_not_depend_on_the_tiles_of_their_rows(hidden, ff, form):
    """Lists of 32, 64, 128 and 192 rows, and what their last tiles are rounded up to: the same bits."""
    from pulse_infer_amd.ops import kernels

    counts = [1, 31, 33, 63, 64, 65, 96, 127, 128, 129, 191, 193, 192 + 64, 192 + 65, 320, 321, 0, 384 + 128]
    experts, pairs = len(counts), sum(counts)
    idx = torch.cat([torch.full((c,), e, dtype=torch.int32) for e, c in enumerate(counts)]).view(pairs, 1).to(DEV)
    x = rnd(pairs, hidden, seed=2).to(torch.bfloat16).to(DEV)
    wg, wu = ((rnd(experts, ff, hidden, seed=3 + i) * hidden ** -0.5).to(torch.bfloat16).to(DEV) for i in range(2))
    wd = (rnd(experts, hidden, ff, seed=5) * ff ** -0.5).to(torch.bfloat16).to(DEV)
    weight = torch.rand(pairs, 1, generator=torch.Generator().manual_seed(6)).to(DEV) + 0.5
    kw = dict(weight_on_input=True, activation="clamped_swish", limit=0.8) if form != "silu" else {}
    results = []
    for rows in (32, 64, 128, 192):
        act = torch.full((pairs, ff), float("nan"), dtype=torch.bfloat16, device=DEV)
        y = torch.full((pairs, hidden), float("nan"), device=DEV)
        ints = torch.full((2 * pairs + 3 * kernels.moe_max_tiles(pairs, experts, rows) + 1,), -5, dtype=torch.int32, device=DEV)
        kernels.moe_grouped(x, wg, wu, wd, idx, weight, act, y, None, ints, rows, **kw)
        results.append((act, y))
    assert not torch.isnan(results[0][0]).any() and not torch.isnan(results[0][1]).any()
    for act, y in results[1:]:
        assert torch.equal(act, results[0][0]) and torch.equal(y, results[0][1])


@pytest.mark.parametrize("low,high", [(0.1, 8.0), (-22.0, -15.0)])
def test_activation_of_grouped_experts_is_rounded_once(low, high):
    """silu(gate) * up is a float32 value within 8 units of 2^-24 of the function (the exponential 2 units, the sum, the quotient and the
    product one each) and then rounded to bfloat16: what lies further from a tie than that is rounded as the function itself is.  Gates and ups are
    products of two bfloat16 values, which float32 holds."""
    from pulse_infer_amd.ops import kernels

    hidden, ff, pairs, rows = 64, 448, 1920, 192
    x, wg, wu = torch.zeros(pairs, hidden), torch.zeros(1, ff, hidden), torch.zeros(1, ff, hidden)
    x[:, 0], x[:, 1] = 1.0 + torch.rand(pairs, generator=torch.Generator().manual_seed(1)), 1.0 + torch.arange(pairs) / 128 % 1
    wg[0, :, 0] = torch.linspace(low, high, ff)              # (gates of up to twice that)
    wu[0, :, 1] = rnd(ff, seed=2)
    x, wg, wu = (t.to(torch.bfloat16) for t in (x, wg, wu))
    g, u = (x.to(F64)[:, i:i + 1] * w.to(F64)[0, :, i] for i, w in ((0, wg), (1, wu)))
    want = g * torch.sigmoid(g) * u
    act = torch.full((pairs, ff), float("nan"), dtype=torch.bfloat16, device=DEV)
    y = torch.full((pairs, hidden), float("nan"), device=DEV)
    wd = torch.zeros(1, hidden, ff, dtype=torch.bfloat16)
    idx = torch.zeros(pairs, 1, dtype=torch.int32)
    ints = torch.full((2 * pairs + 3 * kernels.moe_max_tiles(pairs, 1, rows) + 1,), -5, dtype=torch.int32, device=DEV)
    kernels.moe_grouped(x.to(DEV), wg.to(DEV), wu.to(DEV), wd.to(DEV), idx.to(DEV), torch.ones(pairs, 1).to(DEV), act, y, None, ints, rows)
    below, above = (torch.nextafter(act.cpu(), torch.full((), s * float("inf"), dtype=torch.bfloat16)).to(F64) for s in (-1, 1))
    got = act.cpu().to(F64)
    bound = 8 * 2.0 ** -24 * want.abs()
    assert ((want >= (got + below) / 2 - bound) & (want <= (got + above) / 2 + bound)).all()
