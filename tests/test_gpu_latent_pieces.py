"""The kernels around the expanded form of latent attention, in pieces of 16 bytes and value by value: the same results."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16


def bf(*s, seed):
    return torch.randn(s, generator=torch.Generator().manual_seed(seed)).to(BF).to(DEV)


def shifted(t):
    """The same values at an address that is no multiple of 16 (the kernels then go value by value)."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:]
    return flat.view(t.shape).copy_(t)


@pytest.mark.parametrize("heads,d,rot,dv,width", [(1, 8, 16, 8, 32), (3, 128, 64, 128, 192), (5, 24, 16, 56, 64), (2, 64, 32, 8, 96)])
@pytest.mark.parametrize("pairing", [0, 1])
def test_queries_pages_and_results_in_pieces(heads, d, rot, dv, width, pairing):
    from pulse_infer_amd.ops import kernels

    tokens, rank, src_page = 37, 40, 16
    q, angle = bf(tokens, heads * (d + rot), seed=1), torch.randn(tokens, rot // 2, generator=torch.Generator().manual_seed(2)).to(DEV)
    out = [torch.full((tokens, heads * width), float("nan"), dtype=BF, device=DEV) for _ in range(2)]
    kernels.latent_queries(q, 0, out[0], angle.cos(), angle.sin(), pairing, heads, d, rot, width)
    kernels.latent_queries(shifted(q), 0, out[1], angle.cos(), angle.sin(), pairing, heads, d, rot, width)
    # (the compiler may contract the two products' sum differently: a float32 rounding of it before that to bfloat16)
    x = q.double().view(tokens, heads, d + rot)
    a, b = (x[..., d::2], x[..., d + 1::2]) if pairing == 0 else (x[..., d:d + rot // 2], x[..., d + rot // 2:])
    c, s = angle.cos().double().unsqueeze(1), angle.sin().double().unsqueeze(1)
    want = torch.zeros(tokens, heads, width, dtype=torch.float64, device=DEV)
    want[..., :d] = x[..., :d]
    lo, hi = (slice(d, d + rot, 2), slice(d + 1, d + rot, 2)) if pairing == 0 else (slice(d, d + rot // 2), slice(d + rot // 2, d + rot))
    want[..., lo], want[..., hi] = a * c - b * s, b * c + a * s
    bound = 2.0 ** -8 * want.abs() + 2.0 ** -22 * (x.abs().amax() * 2)
    for o in out:
        assert ((o.double().view_as(want) - want).abs() <= bound).all()
    kc = bf(9, 1, src_page, rank + rot, seed=3)
    table = torch.tensor([[3, 7, 1, 8, 0, 5, -1, 2]], dtype=torch.int32, device=DEV)
    pages = torch.tensor([0, 0, 85, 0, 0, 64, 85, 0], dtype=torch.int32, device=DEV)     # 85 cached tokens: the rest is zeros
    up = bf(2 * kernels.EXPANDED_PAGE, heads * (d + dv), seed=4)
    results = []
    for u in (up, shifted(up)):
        k = torch.full((2, heads, kernels.EXPANDED_PAGE, width), float("nan"), dtype=BF, device=DEV)
        v = torch.full((2, heads, width, kernels.EXPANDED_PAGE), float("nan"), dtype=BF, device=DEV)
        kernels.latent_pages(kc, table, pages, u, k, v, d, rot, dv, rank)
        results.append((k, v))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
    assert torch.equal(results[0][1][:, :, :dv].transpose(2, 3).reshape(2, heads, -1, dv),
                       up[:, heads * d:].view(2, kernels.EXPANDED_PAGE, heads, dv).transpose(1, 2))
    y = [torch.empty(tokens, heads * dv, dtype=BF, device=DEV) for _ in range(2)]
    o = bf(tokens, heads * width, seed=5)
    kernels.latent_compact(o, width, y[0], heads, dv)
    kernels.latent_compact(shifted(o), width, y[1], heads, dv)
    assert torch.equal(y[0], y[1]) and torch.equal(y[0], o.view(tokens, heads, width)[..., :dv].reshape(tokens, -1))


@pytest.mark.parametrize("tokens", [1, 5, 700])
@pytest.mark.parametrize("d,stored,rotary,pairing", [(128, 128, 128, 1), (64, 96, 16, 1), (24, 32, 8, 0), (40, 40, 0, 0)])
def test_rows_of_queries_and_keys_in_pieces(tokens, d, stored, rotary, pairing):
    """Queries and keys without biases and norms: 16 bytes a thread, and value by value (from an address that is no multiple of 16)."""
    from pulse_infer_amd.ops import kernels

    nq, nkv, dv, page = 5, 2, 24, 16
    x = bf(tokens, nq * d + nkv * (d + dv), seed=7)
    angle = torch.randn(tokens, max(1, rotary // 2), generator=torch.Generator().manual_seed(8)).to(DEV)
    cos, sin = (angle.cos(), angle.sin()) if rotary else (None, None)
    entries = 3
    width = (tokens + page - 1) // page + 1
    table = torch.randperm(entries * width, generator=torch.Generator().manual_seed(9)).to(torch.int32).view(entries, width).to(DEV)
    table[2, 0] = -1                                        # no page: nothing is written there
    entry = (torch.arange(tokens) % entries).to(torch.int32).to(DEV)
    positions = torch.arange(tokens, dtype=torch.int32, device=DEV)
    got = []
    for src in (x, shifted(x)):
        q = torch.full((tokens, nq * stored), float("nan"), dtype=BF, device=DEV)
        k = torch.full((entries * width, nkv, page, stored), 7.0, dtype=BF, device=DEV)
        v = torch.full((entries * width, nkv, stored, page), 7.0, dtype=BF, device=DEV)
        kernels.qkv_rows(src, q, nq, nkv, d, dv, stored, None, None, 1e-6, cos, sin, rotary, pairing, k, v, positions, entry, table,
                         norm=False)
        got.append((q, k, v))
    # (the two products' sum may be contracted differently: a float32 rounding before that to bfloat16)
    for one, two in zip(*got):
        assert ((one.double() - two.double()).abs() <= 2.0 ** -7 * two.double().abs() + 2.0 ** -20).all()
    if rotary == 0:
        assert torch.equal(got[0][0].view(tokens, nq, stored)[..., :d].reshape(tokens, -1), x[:, :nq * d])
