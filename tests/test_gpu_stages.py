"""The product in stages (some tens to some hundreds of rows) where its tiles and its shares of K end."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F64 = torch.float64


def rnd(*shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed))


# remainders of rows and weight rows, one step of K and many, one row and several panels; bfloat16 results, float32 shares of one
# step each and of the plan's number, SwiGLU (which tile runs is the plan's choice: every one of them, with the stages of K going
# round, is in the tests behind this one)
@pytest.mark.parametrize("shape", [(1, 32, 64), (65, 96, 128), (97, 6144, 192), (97, 24576, 64), (128, 4096, 1024),
                                   (130, 24608, 128), (193, 12288, 64), (256, 4128, 320), (357, 6176, 64), (1030, 2080, 128),
                                   # tiles of 192 and 256 rows of X, panels of them
                                   (357, 24544, 64), (509, 24544, 1024), (357, 24608, 64), (509, 24608, 64), (2100, 8224, 128)])
def test_product_in_stages_at_the_edges_of_its_tiles(shape):
    from pulse_infer_amd.ops import kernels

    m, n, k = shape
    x, w = rnd(m, k, seed=1).to(torch.bfloat16), rnd(n, k, seed=2).to(torch.bfloat16)
    xd, wd = torch.empty(m, k + 8, dtype=torch.bfloat16, device=DEV)[:, :k], w.to(DEV)
    xd.copy_(x)                                         # (rows may lie further apart than they are long)
    want, size = x.to(F64) @ w.to(F64).T, x.to(F64).abs() @ w.to(F64).abs().T
    exact = (k + 2) * 2.0 ** -24 * size                 # a float32 sum of k exact products, in any order
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    kernels.gemm_stages(xd, wd, out)
    assert ((out.cpu().to(F64) - want).abs() <= exact + 2.0 ** -8 * want.abs()).all()
    best = kernels.gemm_stages_shares(m, n, k)
    assert best >= 1 and k % (64 * best) == 0
    for shares in {1, best, k // 64}:
        parts = torch.full((shares, m, n), float("nan"), device=DEV)
        kernels.gemm_stages(xd, wd, parts)
        got = parts.cpu().to(F64)
        assert ((got.sum(0) - want).abs() <= exact).all(), shares
        part = k // shares
        last = x[:, k - part:].to(F64) @ w[:, k - part:].to(F64).T
        assert ((got[-1] - last).abs() <= exact).all(), shares
    slab = torch.arange(n) // 16 % 2
    gate, up = want[:, slab == 0] / k ** 0.5, want[:, slab == 1] / k ** 0.5
    xs = (x.float() / k ** 0.5).to(torch.bfloat16) if (k ** 0.5).is_integer() and k in (64, 1024) else None
    if xs is not None:                                  # (a power of two: the scaled rows are exact)
        act = torch.full((m, n // 2), float("nan"), dtype=torch.bfloat16, device=DEV)
        kernels.gemm_stages(xs.to(DEV), wd, act, swiglu=True)
        wanted = gate * torch.sigmoid(gate) * up
        # hardware exponential and reciprocal (relative 2^-21 each), one rounding to bfloat16
        assert ((act.cpu().to(F64) - wanted).abs() <= 2.0 ** -7.9 * wanted.abs() + 1e-5).all()


STEPS = 13      # more than twice the stages of any tile: every stage is filled, read and filled again


def product(m, n, k):
    x, w = rnd(m, k, seed=1).to(torch.bfloat16).to(DEV), (rnd(n, k, seed=2) * k ** -0.5).to(torch.bfloat16).to(DEV)
    want, size = x.to(F64) @ w.to(F64).T, x.to(F64).abs() @ w.to(F64).abs().T
    return x, w, want, (k + 2) * 2.0 ** -24 * size          # (a float32 sum of k exact products, in any order)


# the tile that the plan takes for these rows and weight rows on 256 compute units, remainders of both
@pytest.mark.parametrize("tile,m,n", [((64, 64), 70, 672), ((64, 128), 70, 8288), ((96, 128), 70, 16928), ((128, 64), 130, 8288),
                                      ((128, 128), 130, 12960), ((192, 128), 130, 16928), ((256, 128), 130, 24864),
                                      ((192, 192), 130, 32800), ((192, 256), 193, 32800), ((256, 192), 300, 24864),
                                      ((256, 256), 600, 16928)])
def test_every_tile_of_the_product_in_stages(tile, m, n):
    from pulse_infer_amd.ops import kernels

    k = 64 * STEPS
    assert kernels.gemm_stages_tile(m, n, k) == tile and m % tile[1] and n % tile[0]
    x, w, want, exact = product(m, n, k)
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    kernels.gemm_stages(x, w, out)
    assert ((out.to(F64) - want).abs() <= exact + 2.0 ** -8 * want.abs()).all()
    act = torch.full((m, n // 2), float("nan"), dtype=torch.bfloat16, device=DEV)
    kernels.gemm_stages(x, w, act, swiglu=True)
    slab = torch.arange(n, device=DEV) // 16 % 2
    gate, up, gate_off, up_off = want[:, slab == 0], want[:, slab == 1], exact[:, slab == 0], exact[:, slab == 1]
    silu = gate * torch.sigmoid(gate)
    # (silu's slope is 1.1 at most; the exponential and the reciprocal, one rounding to bfloat16)
    bound = (2.0 ** -8 + 2.0 ** -16) * (silu * up).abs() + 1.1 * gate_off * (up.abs() + up_off) + silu.abs() * up_off
    assert ((act.to(F64) - silu * up).abs() <= bound).all()


@pytest.mark.parametrize("tile,m,n,shares", [((64, 64), 70, 356, 2), ((64, 128), 70, 4232, 2), ((96, 128), 70, 8336, 2),
                                             ((128, 64), 130, 4232, 2), ((128, 128), 130, 3092, 4), ((192, 128), 130, 8336, 2),
                                             ((256, 128), 130, 12440, 2), ((192, 192), 130, 16544, 2), ((192, 256), 193, 16544, 2),
                                             ((256, 192), 130, 12440, 4), ((256, 256), 193, 12440, 4)])
def test_every_tile_of_the_product_in_stages_in_shares(tile, m, n, shares):
    from pulse_infer_amd.ops import kernels

    k = 64 * STEPS * shares
    assert kernels.gemm_stages_tile(m, n, k, shares) == tile and m % tile[1] and n % tile[0]
    x, w, want, exact = product(m, n, k)
    parts = torch.full((shares, m, n), float("nan"), device=DEV)
    kernels.gemm_stages(x, w, parts)
    assert ((parts.to(F64).sum(0) - want).abs() <= exact).all()
    part = k // shares
    for i in range(shares):
        a, b = x[:, i * part:(i + 1) * part].to(F64), w[:, i * part:(i + 1) * part].to(F64)
        assert ((parts[i].to(F64) - a @ b.T).abs() <= (part + 2) * 2.0 ** -24 * (a.abs() @ b.abs().T)).all(), i


def test_product_in_stages_refuses_what_it_cannot_read():
    from pulse_infer_amd.ops import kernels
    from pulse_infer_amd.ops.library import KernelError

    x, w = torch.zeros(70, 96, dtype=torch.bfloat16, device=DEV), torch.zeros(64, 96, dtype=torch.bfloat16, device=DEV)
    assert not kernels.gemm_stages_takes(70, 64, 96) and kernels.gemm_stages_shares(70, 64, 96) == 0
    with pytest.raises((KernelError, ValueError)):
        kernels.gemm_stages(x, w, torch.empty(70, 64, dtype=torch.bfloat16, device=DEV))


def test_product_in_stages_applies_silu_where_its_exponential_is_largest():
    """Gates down to -88.6, where 1 / (1 + exp(-gate)) is smaller than any normal float32 number: silu(gate) is still one, and
    so is its product with a large up."""
    from pulse_infer_amd.ops import kernels

    m, n, k = 65, 64, 64
    gates = torch.linspace(-88.6, 88.6, m)
    x, w = torch.zeros(m, k, dtype=torch.bfloat16), torch.zeros(n, k, dtype=torch.bfloat16)
    high = gates.to(torch.bfloat16)
    x[:, 0], x[:, 1], x[:, 2] = high, (gates - high.float()).to(torch.bfloat16), 1024.0
    gate_rows = torch.arange(n) // 16 % 2 == 0
    w[gate_rows, 0] = w[gate_rows, 1] = 1.0
    w[~gate_rows, 2] = 1.0
    act = torch.full((m, n // 2), float("nan"), dtype=torch.bfloat16, device=DEV)
    kernels.gemm_stages(x.to(DEV), w.to(DEV), act, swiglu=True)
    g = (x[:, 0].to(F64) + x[:, 1].to(F64)).view(m, 1)
    want = (g / (1.0 + torch.exp(-g)) * 1024.0).expand(m, n // 2)
    # the exponential of a number good to 2^-24 of up to 89 (2^-17), a reciprocal, one rounding to bfloat16
    bound = (2.0 ** -8 + 2.0 ** -16) * want.abs() + 1024.0 * 2.0 ** -149
    assert ((act.cpu().to(F64) - want).abs() <= bound).all()


@pytest.mark.parametrize("n,k", [(4096, 1024), (1028, 4096), (2048, 2048)])
def test_an_update_in_stages_does_not_depend_on_the_rows_beside_it(n, k):
    """65 to 192 rows: the same shares, every tile walks a share in the same order; to the bit."""
    from pulse_infer_amd.parts.base import Workspace
    from pulse_infer_amd.parts.linear import Linear

    lin = Linear((rnd(n, k, seed=3) * k ** -0.5).to(torch.bfloat16).to(DEV), "bfloat16")
    x = rnd(192, k, seed=4).to(torch.bfloat16).to(DEV)
    ws, h = Workspace(torch.device(DEV)), torch.zeros(192, n, device=DEV)
    scratch = torch.empty(192, n, dtype=torch.bfloat16, device=DEV)
    whole = lin.add_into(x, h, scratch, ws).clone()
    assert whole.dim() == 3
    for m in (65, 97, 128, 160, 191):
        assert torch.equal(lin.add_into(x[:m], h[:m], scratch[:m], ws), whole[:, :m])


@pytest.mark.parametrize("m_out,k_in", [(512, 128), (40, 256), (128, 512), (72, 264), (200, 1000)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_a_product_a_head_does_not_depend_on_the_tokens_beside_it(m_out, k_in, dtype):
    """A token by itself, a few, and enough for tiles of 64 tokens: the same bits."""
    from pulse_infer_amd.ops import kernels

    heads, tokens = 5, 1100
    w = (rnd(heads, m_out, k_in, seed=1) * k_in ** -0.5).to(torch.bfloat16).to(DEV)
    x = rnd(tokens, heads * k_in, seed=2).to(dtype).to(DEV)

    def run(rows):
        out = torch.full((rows.shape[0], heads * m_out), float("nan"), dtype=torch.bfloat16, device=DEV)
        kernels.heads_product(rows, k_in, w, None, out, m_out, 0.5)
        return out

    whole = run(x)
    for a, b in ((0, 1), (3, 20), (100, 355), (500, 756), (700, 1001)):
        assert torch.equal(run(x[a:b].contiguous()), whole[a:b]), (a, b)
    xr = x.to(torch.bfloat16).cpu().to(F64).view(tokens, heads, k_in)
    want = 0.5 * torch.stack([xr[:, h] @ w[h].cpu().to(F64).T for h in range(heads)], 1).reshape(tokens, -1)
    size = 0.5 * torch.stack([xr[:, h].abs() @ w[h].cpu().to(F64).abs().T for h in range(heads)], 1).reshape(tokens, -1)
    assert ((whole.cpu().to(F64) - want).abs() <= (k_in + 4) * 2.0 ** -24 * size + 2.0 ** -8 * want.abs()).all()


@pytest.mark.parametrize("policy", ["stages", "none"])
@pytest.mark.parametrize("rows,n", [(193, 256), (257, 256), (513, 768), (1100, 1028), (2560, 256)])
def test_updates_in_shares_make_no_batched_product(rows, n, policy, monkeypatch):
    """The batched product in bfloat16 with a transposed view as its right operand is a call that has faulted: no update
    makes it, whoever makes the shares."""
    from pulse_infer_amd.parts import linear
    from pulse_infer_amd.parts.base import Workspace

    def never(*args, **kwargs):
        raise AssertionError("a batched product was called")
    for name in ("bmm", "baddbmm", "matmul", "einsum"):
        monkeypatch.setattr(torch, name, never)
    monkeypatch.setattr(linear, "OWN_MANY_ROWS", policy)
    k = 8192
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, k, generator=g).bfloat16().to(DEV)
    w = (torch.randn(n, k, generator=g) * k ** -0.5).bfloat16().to(DEV)
    lin = linear.Linear(w, "bfloat16")
    assert lin.library_shares_for(x)
    parts = lin.add_into(x, torch.zeros(rows, n, device=DEV), torch.empty(rows, n, dtype=torch.bfloat16, device=DEV),
                         Workspace(torch.device(DEV)))
    want = torch.mm(x.double(), w.double().t())
    bound = (k + 2) * 2.0 ** -24 * torch.mm(x.double().abs(), w.double().abs().t())     # as above, the shares' sum in 64 bits
    assert parts.dtype == torch.float32 and parts.shape[1:] == (rows, n)
    assert ((parts.double().sum(0) - want).abs() <= bound).all()


def test_gate_and_up_in_stages_do_not_depend_on_the_rows_beside_them():
    """Where a block of weight rows starts its walk along K is a matter of the weight alone: every tile, the same bits."""
    from pulse_infer_amd.ops import kernels

    n, k = 24608, 64 * STEPS
    x, w, _, _ = product(600, n, k)
    whole = torch.empty((600, n // 2), dtype=torch.bfloat16, device=DEV)
    kernels.gemm_stages(x, w, whole, swiglu=True)
    tiles = set()
    for m in (1, 65, 97, 130, 193, 357, 509):
        tiles.add(kernels.gemm_stages_tile(m, n, k))
        act = torch.full((m, n // 2), float("nan"), dtype=torch.bfloat16, device=DEV)
        kernels.gemm_stages(x[:m], w, act, swiglu=True)
        assert torch.equal(act, whole[:m]), m
    assert len(tiles) >= 4


@pytest.mark.parametrize("k", [320, 2560])
@pytest.mark.parametrize("rows", [70, 300])
def test_blocks_of_weight_rows_start_together_where_their_rows_are_no_power_of_two(rows, k):
    """Rows of another length lie on channels of their own: their sums have the one order of K, whichever block they lie in."""
    from pulse_infer_amd.ops import kernels

    x, block = rnd(rows, k, seed=5).to(torch.bfloat16).to(DEV), rnd(768, k, seed=6).to(torch.bfloat16).to(DEV)
    w = block.repeat(4, 1).contiguous()
    act = torch.full((rows, 1536), float("nan"), dtype=torch.bfloat16, device=DEV)
    kernels.gemm_stages(x, w, act, swiglu=True)
    assert not torch.isnan(act).any() and torch.equal(act[:, :768], act[:, 768:])


@pytest.mark.parametrize("far", ["x", "w", "both"])
@pytest.mark.parametrize("apart", [(1 << 22) + 8, 17000008, 34000000, 34100008])
def test_product_in_stages_of_rows_gigabytes_apart(far, apart):
    """A tile's last row (64 a tile) 0.5, 2.1, 4.28 and 4.3 GB behind its first, which is more than offsets of 32 bits reach: the same
    bits as of rows that lie together.  (4 GB in front of the operands, so that an offset taken for a negative one finds other values.)"""
    from pulse_infer_amd.ops import kernels

    m, n, k = 130, 160, 192
    x, w, _, _ = product(m, n, k)
    front = 1 << 31

    def spread(t):
        room = torch.empty(front + t.shape[0] * apart, dtype=t.dtype, device=DEV)
        return room.as_strided(t.shape, (apart, 1), front).copy_(t)
    xf, wf = (spread(t) if far in (name, "both") else t for name, t in (("x", x), ("w", w)))
    for swiglu, width in ((False, n), (True, n // 2)):
        near, out = (torch.full((m, width), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2))
        kernels.gemm_stages(x, w, near, swiglu=swiglu)
        kernels.gemm_stages(xf, wf, out, swiglu=swiglu)
        assert torch.equal(out, near)
    near, out = (torch.full((3, m, n), float("nan"), device=DEV) for _ in range(2))
    kernels.gemm_stages(x, w, near)
    kernels.gemm_stages(xf, wf, out)
    assert torch.equal(out, near)


@pytest.mark.parametrize("rows,gap,contiguous", [(1030, 0, True), (1030, 8, True), (1030, 4, True), (1030, 0, False), (520, 0, True)])
def test_float32_results_of_many_rows(rows, gap, contiguous):
    """16,384 x 1,024 with float32 results: in stages from the estimate's line on, elsewhere as before (fewer rows, rows that are
    not 16 bytes aligned, results further apart), the same sums within float32 in any order."""
    from pulse_infer_amd.parts.linear import Linear

    n, k = 16384, 1024
    lin = Linear((rnd(n, k, seed=2) * k ** -0.5).to(torch.bfloat16).to(DEV), "bfloat16")
    x = torch.empty(rows, k + gap, dtype=torch.bfloat16, device=DEV)[:, :k]
    x.copy_(rnd(rows, k, seed=1))
    assert lin.takes_stages_float32(x, lin.weight) == (rows > 1024 and gap % 8 == 0)
    out = torch.full((rows, n if contiguous else n + 4), float("nan"), device=DEV)[:, :n]
    lin.forward(x, out)
    some = [0, 1, 255, 256, 511, rows - 1]
    xs, ws = x[some].cpu().to(F64), lin.weight.cpu().to(F64)
    assert bool(out.isfinite().all())
    assert ((out[some].cpu().to(F64) - xs @ ws.T).abs() <= (k + 2) * 2.0 ** -24 * (xs.abs() @ ws.abs().T)).all()
