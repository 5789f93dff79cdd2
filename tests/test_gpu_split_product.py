"""The product of float32 operands as bfloat16 parts: the edges of its tiles, shares and chunks of rows, its order of sums, and
values outside the range in which parts are exact."""
import ctypes

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


def bound(a, w):
    """A sum of K products in float32, in any order: |error| <= (K + 2) u sum |a| |w|, which the parts keep (measured: a
    fiftieth of it)."""
    return (a.shape[1] + 2) * U * (a.abs().to(F64) @ w.abs().to(F64).T)


def without_scratch(a, w, out):
    from pulse_infer_amd.ops.library import call
    p, i, j = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
    call("pulse_gemm_f32", p(a.data_ptr()), i(0), p(w.data_ptr()), i(0), p(out.data_ptr()), i(0), i(a.shape[0]), i(w.shape[0]),
         i(a.shape[1]), j(a.stride(0)), j(w.stride(0)), j(out.stride(0)), p(torch.cuda.current_stream().cuda_stream))


# rows x weight rows x K (all past the line of 6 x 2^20 values of the weight): each way for few rows, tiles of 32, 64 and 96 rows with
# one and several workgroups along K and their remainders; K of less than a block, of fewer blocks than shares, of unequal shares
# and no whole block at the end; weight rows past a tile of 256 and no multiple of four; more rows than a chunk
@pytest.mark.parametrize("shape", [(16, 160000, 40), (17, 1600000, 4), (32, 100000, 64), (33, 3100, 2052), (64, 25000, 260),
                                   (65, 48000, 132), (96, 1537, 4096), (97, 2048, 4100), (129, 1057, 6000), (200, 16384, 516),
                                   (333, 6150, 1028), (400, 790, 7972), (2017, 47700, 132), (2100, 11500, 548)])
def test_parts_at_the_edges(k, shape):
    m, n, kk = shape
    a, w = rnd(m, kk, seed=1).to(DEV), rnd(n, kk, seed=2).to(DEV)
    out = torch.full((m, n), float("nan"), device=DEV)
    k.gemm_f32(a, w, out)
    assert ((out.to(F64) - a.to(F64) @ w.to(F64).T).abs() <= bound(a, w)).all()
    plain = torch.full((m, n), float("nan"), device=DEV)
    without_scratch(a, w, plain)
    assert torch.equal(plain, out)
    for first, rows in ((0, 1), (m // 2, 1), (m - 1, 1), (max(0, m - 20), 20), (m // 3, min(70, m - m // 3))):
        part = torch.empty(min(rows, m - first), n, device=DEV)      # whatever is in the batch: the same bits
        k.gemm_f32(a[first:first + rows], w, part)
        assert torch.equal(part, out[first:first + rows])


@pytest.mark.parametrize("m", [1, 20, 70, 333])
def test_parts_of_strided_operands_and_results(k, m):
    """Rows further apart than they are long, results that are a column range, results in bfloat16, and operands that cannot be
    read four values at a time (the float32 instruction: the same result to rounding)."""
    n, kk = 3070, 2052
    wide_a, wide_w = rnd(m, kk + 12, seed=3).to(DEV), rnd(n, kk + 8, seed=4).to(DEV)
    a, w = wide_a[:, 8:8 + kk], wide_w[:, 4:4 + kk]
    want, limit = a.to(F64) @ w.to(F64).T, bound(a, w)
    out = torch.full((m, n + 7), 5.0, device=DEV)
    k.gemm_f32(a, w, out[:, 3:3 + n])
    assert ((out[:, 3:3 + n].to(F64) - want).abs() <= limit).all() and (out[:, :3] == 5.0).all() and (out[:, 3 + n:] == 5.0).all()
    whole = torch.empty(m, n, device=DEV)
    k.gemm_f32(a.contiguous(), w.contiguous(), whole)
    assert torch.equal(out[:, 3:3 + n], whole)
    rounded = torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
    k.gemm_f32(a, w, rounded)
    assert torch.equal(rounded, whole.to(torch.bfloat16))
    k.gemm_f32(wide_a[:, 7:7 + kk], wide_w[:, 3:3 + kk], whole)
    off = wide_a[:, 7:7 + kk].to(F64) @ wide_w[:, 3:3 + kk].to(F64).T
    assert ((whole.to(F64) - off).abs() <= bound(wide_a[:, 7:7 + kk], wide_w[:, 3:3 + kk])).all()


@pytest.mark.parametrize("shape", [(5, 9800, 644), (30, 9800, 644), (200, 9800, 644), (333, 3080, 2052)])
def test_values_outside_the_range_of_parts(k, shape):
    """Infinities, NaN, the largest finite values, values whose parts would vanish, and rows of zeros, in either operand: what
    float32 arithmetic makes of them, in their rows and columns alone."""
    m, n, kk = shape
    a, w = rnd(m, kk, seed=5), rnd(n, kk, seed=6)
    clean = torch.empty(m, n, device=DEV)
    k.gemm_f32(a.to(DEV), w.to(DEV), clean)
    inf, nan, most = float("inf"), float("nan"), torch.finfo(torch.float32).max
    a[0, 3], a[1, kk - 1], a[2], a[3, kk // 2] = inf, nan, a[2] * 1e-36, most
    a[4] = 0.0
    w[5, 3], w[6, 7], w[7, kk - 2], w[8] = 0.0, -inf, 2.0 ** 70, w[8] * 2.0 ** -110
    w[9] = 0.0
    w[6, 3] = 1.0                                        # (with the infinity of row 0: +inf - inf)
    out = torch.full((m, n), 3.0, device=DEV)
    k.gemm_f32(a.to(DEV), w.to(DEV), out)
    plain = torch.empty(m, n, device=DEV)
    without_scratch(a.to(DEV), w.to(DEV), plain)
    assert torch.equal(torch.nan_to_num(plain, nan=7.0), torch.nan_to_num(out, nan=7.0))
    got, want = out.cpu(), (a.to(F64) @ w.to(F64).T)
    limit = bound(a, w) + kk * 2.0 ** -126     # (a product or sum below the smallest normal number may be flushed to zero)
    special = torch.isnan(want) | torch.isinf(want) | (want.abs() > most)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got[special & ~torch.isnan(want)], want[special & ~torch.isnan(want)].to(torch.float32))
    assert ((got.to(F64) - want).abs()[~special] <= limit[~special]).all()
    assert torch.equal(got[5 if m > 5 else 4:, 10:], (clean.cpu()[5:, 10:] if m > 5 else torch.zeros(1, n - 10)))


def test_parts_are_no_less_exact_than_the_float32_instruction(k):
    """Error against 64 bits beside that of the same product on the float32 instruction (the path of operands that are not
    aligned): smaller, for operands as activations and weights are, positive ones, and ones of very unequal sizes."""
    m, n, kk = 200, 3080, 2048
    for seed, make in ((1, lambda x: x), (2, torch.abs), (3, lambda x: x * torch.exp(3 * rnd(*x.shape, seed=9)))):
        wide_a, wide_w = make(rnd(m, kk + 4, seed=seed)).to(DEV), make(rnd(n, kk + 4, seed=seed + 10)).to(DEV)
        errors = []
        for at in (4, 3):
            a, w = wide_a[:, at:at + kk], wide_w[:, at:at + kk]
            out = torch.empty(m, n, device=DEV)
            k.gemm_f32(a, w, out)
            want = a.to(F64) @ w.to(F64).T
            errors.append(float((out.to(F64) - want).norm() / want.norm()))
        assert errors[0] <= 0.8 * errors[1]        # (measured 0.4 to 0.6)


# weights past the line whose rows and K end inside tiles and blocks, long and short of both
@pytest.mark.parametrize("n,kk", [(3074, 2052), (16390, 516), (1030, 8196), (6150, 1028), (40003, 164), (4099, 4100)])
def test_parts_of_some_rows_are_the_same_bits_whatever_the_tile(k, n, kk):
    """Every number of rows up to some hundreds goes its own way (tiles of 16 to 64 rows by 16 to 64 weight rows, of 64 and 96 by 256,
    with K in one go or over workgroups): each row's results are those of the largest batch, and within a float32 sum's bound."""
    most = 200
    a, w = rnd(most, kk, seed=11).to(DEV), rnd(n, kk, seed=12).to(DEV)
    whole = torch.full((most, n), float("nan"), device=DEV)
    k.gemm_f32(a, w, whole)
    assert ((whole.to(F64) - a.to(F64) @ w.to(F64).T).abs() <= bound(a, w)).all()
    for m in (1, 4, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 96, 97, 129, 160, 161):
        some = torch.full((m, n), float("nan"), device=DEV)
        k.gemm_f32(a[most - m:], w, some)
        assert torch.equal(some, whole[most - m:]), m
        without_scratch(a[:m], w, some)
        assert torch.equal(some, whole[:m]), m


# members whose third part, second part, all parts but the first are below the smallest normal number
@pytest.mark.parametrize("e", [-60, -108, -112, -118, -124])
def test_members_far_below_their_row_s_largest(k, e):
    """A row whose largest value is in range is taken apart whatever its other members are: of these, parts below 2^-126 are lost
    (less than 2^-126 of a value), and products and sums below it may be flushed, six a pair of values.  It shows where
    the large values meet zeros."""
    n, kk = 3074, 2052
    w = rnd(n, kk, seed=14)
    w[:, 0] = 0.0
    for m in (1, 33, 333):
        a = rnd(m, kk, seed=13) * 2.0 ** e
        a[:, 0] = 1.0
        out = torch.empty(m, n, device=DEV)
        k.gemm_f32(a.to(DEV), w.to(DEV), out)
        small = a.clone()
        small[:, 0] = 0.0
        limit = bound(small, w) + 2.0 ** -126 * (w.abs().to(F64).sum(1) + 6 * kk)
        assert ((out.cpu().to(F64) - small.to(F64) @ w.to(F64).T).abs() <= limit).all(), m
