"""Decoded tokens, short portions and prompt portions in one attention launch: the bits of the two launches it stands for."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class Entry:
    def __init__(self, start, count, first_row):
        self.start, self.count, self.first_row = start, count, first_row


# head sizes with a kernel for both and without; whole walks and splits of the tokens' keys, one item and many, a window, chunks
@pytest.mark.parametrize("d", [128, 64, 32, 192, 80])
@pytest.mark.parametrize("nq,nkv,splits,window,chunk", [(8, 2, 1, 0, 0), (32, 8, 4, 0, 0), (4, 4, 3, 0, 0), (8, 2, 1, 40, 0),
                                                       (8, 2, 1, 0, 96)])
def test_tokens_and_portions_in_one_launch(d, nq, nkv, splits, window, chunk):
    from pulse_infer_amd.ops import attention_mfma as am

    page, lengths = 16, [(0, 1), (300, 1), (77, 3), (0, 200), (130, 33), (511, 1), (5, 16)]
    gen = torch.Generator().manual_seed(d + nq)
    entries, rows = [], 0
    for start, count in lengths:
        entries.append(Entry(start, count, rows))
        rows += count
    width = max((e.start + e.count + page - 1) // page for e in entries)
    pages = len(entries) * width
    table = torch.randperm(pages, generator=gen).to(torch.int32).view(len(entries), width).to(DEV)
    bf = lambda *s: torch.randn(s, generator=gen).to(torch.bfloat16).to(DEV)
    q, kc, vc = bf(rows, nq * d), bf(pages, nkv, page, d), bf(pages, nkv, d, page)
    positions = torch.tensor([e.start + i for e in entries for i in range(e.count)], dtype=torch.int32, device=DEV)
    group = nq // nkv
    short, long = am.split_entries(entries)
    dev = lambda flat: torch.tensor(flat, dtype=torch.int32, device=DEV)
    short_items = dev(am.build_items(short, am.tokens_per_item(group)))
    long_items = dev(am.build_items(long, am.portion_tokens(group, d)))
    context = max(e.start + e.count for _, e in short)
    size = ((context + splits - 1) // splits + 31) // 32 * 32
    part_o, part_ml = torch.empty(rows * nq * splits * d, device=DEV), torch.empty(rows * nq * splits * 2, device=DEV)
    one, two = (torch.full((rows, nq * d), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    tail = (d ** -0.5, window, size, splits, context, part_o, part_ml)
    am.attn_prefill(q, two, nq, nkv, d, kc, vc, positions, table, long_items, d ** -0.5, window, chunk=chunk)
    am.attn_mfma(q, two, nq, nkv, d, kc, vc, positions, table, short_items, *tail, chunk=chunk)
    am.attn_mfma(q, one, nq, nkv, d, kc, vc, positions, table, short_items, *tail, chunk=chunk, long_items=long_items)
    assert not torch.isnan(two).any() and torch.equal(one, two)


@pytest.mark.parametrize("values", [1, 96, 128, 129, 192])
@pytest.mark.parametrize("splits,window,gated", [(1, 0, False), (3, 0, True), (1, 90, False)])
def test_portions_of_heads_whose_values_are_narrower(values, splits, window, gated):
    """Heads of 192 channels whose values fill ``values`` of them: the bits of the kernel that computes them all, stale values
    (not a number) under keys that nobody sees among it."""
    from pulse_infer_amd.ops import attention_mfma as am

    page, nq, d, lengths = 16, 6, 192, [(0, 333), (70, 64), (500, 17)]
    gen = torch.Generator().manual_seed(values)
    entries, rows = [], 0
    for start, count in lengths:
        entries.append(Entry(start, count, rows))
        rows += count
    width = max((e.start + e.count + page - 1) // page for e in entries)
    pages = len(entries) * width
    table = torch.randperm(pages, generator=gen).to(torch.int32).view(len(entries), width).to(DEV)
    bf = lambda *s: torch.randn(s, generator=gen).to(torch.bfloat16).to(DEV)
    q, kc, vc = bf(rows, nq * d), bf(pages, nq, page, d), bf(pages, nq, d, page)
    vc[:, :, values:] = 0.0
    for i, e in enumerate(entries):                         # behind a request's last position
        end = e.start + e.count
        if end % page:
            vc[int(table[i, end // page]), :, :values, end % page:] = float("nan")
    positions = torch.tensor([e.start + i for e in entries for i in range(e.count)], dtype=torch.int32, device=DEV)
    items = torch.tensor(am.build_items(list(enumerate(entries)), am.portion_tokens(1, d)), dtype=torch.int32, device=DEV)
    size = 192 if splits > 1 else 0
    part_o, part_ml = torch.zeros(rows * nq * splits * d, device=DEV), torch.empty(rows * nq * splits * 2, device=DEV)
    gate = bf(rows, nq) if gated else None
    one, two = (torch.zeros((rows, nq * d), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    args = (nq, nq, d, kc, vc, positions, table, items, d ** -0.5, window, size, splits, part_o, part_ml)
    am.attn_prefill(q, two, *args, gate=gate)
    am.attn_prefill(q, one, *args, gate=gate, values=values)
    wanted = lambda t: t.view(rows, nq, d)[:, :, :values]
    assert not torch.isnan(wanted(two)).any() and torch.equal(wanted(one), wanted(two))


def test_options_of_other_entry_points_are_not_read_here():
    """``plain_norm`` of the options is for decoded tokens that are prepared on the way: whatever it holds, the entry points of prepared
    queries do as without it, and read nothing behind the options."""
    import ctypes

    from pulse_infer_amd.ops import attention_mfma as am
    from pulse_infer_amd.ops.library import call_in
    from pulse_infer_amd.ops.kernels import _f32, _i32, _i64, _ptr, _stream

    d, nq, nkv, page, context = 64, 4, 2, 16, 50
    gen = torch.Generator().manual_seed(3)
    bf = lambda *s: torch.randn(s, generator=gen).to(torch.bfloat16).to(DEV)
    pages = (context + page - 1) // page
    q, kc, vc = bf(context, nq * d), bf(pages, nkv, page, d), bf(pages, nkv, d, page)
    positions = torch.arange(context, dtype=torch.int32, device=DEV)
    table = torch.arange(pages, dtype=torch.int32, device=DEV).view(1, pages)
    entry = [(0, Entry(0, context, 0))]
    lib = am.load_variant("attn_mfma", {"PULSE_HEAD_DIM": d})
    for name, per, tail in (("pulse_attn_mfma", am.tokens_per_item(nq // nkv), (_i32(context),)),
                            ("pulse_attn_prefill", am.portion_tokens(nq // nkv, d), ())):
        items = torch.tensor(am.build_items(entry, per), dtype=torch.int32, device=DEV)
        results = []
        for plain_norm in (0, 1, 2, 3, -1):
            ex = am._Extras()
            ex.plain_norm, ex.v_head0 = plain_norm, -1
            out = torch.full((context, nq * d), float("nan"), dtype=torch.bfloat16, device=DEV)
            split = (_i32(64), _i32(1)) if tail else (_i32(0), _i32(1))
            call_in(lib, name, _ptr(q), _i64(nq * d), _ptr(out), _i64(nq * d), _ptr(kc), _ptr(vc), _ptr(positions), _ptr(table),
                    _i32(pages), _ptr(items), _i32(items.numel() // am.ITEM_INTS), _i32(context), _i32(nq), _i32(nkv), _i32(page),
                    _i32(pages), _f32(d ** -0.5), _i32(0), *split, *tail, _ptr(None), _ptr(None),
                    *((_ptr(None), _ptr(None)) if tail else ()), ctypes.byref(ex), _stream())
            results.append(out)
        assert not torch.isnan(results[0]).any() and all(torch.equal(results[0], r) for r in results[1:])
