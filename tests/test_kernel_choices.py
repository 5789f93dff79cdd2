"""Decisions the host takes for the kernels (no GPU needed): what must hold of every choice, whatever the
numbers the cost rules currently prefer, and for another count of compute units than the MI355X's."""
import itertools
import types

import pytest


class E:
    def __init__(self, start, count):
        self.start, self.count = start, count


@pytest.fixture(params=[256, 304, 64])
def units(request, monkeypatch):
    from pulse_infer_amd.ops import device

    monkeypatch.setattr(device, "_units", request.param)
    assert device.compute_units() == request.param
    return request.param


def test_decode_splits_cover_the_context_in_whole_blocks(units):
    from pulse_infer_amd.ops import attention_mfma as M

    for items, nkv, group, context in itertools.product((1, 2, 8, 24, 64, 200), (1, 8), (1, 4, 20),
                                                        (1, 31, 500, 1024, 4096, 40000)):
        size, n = M.choose_splits(items, nkv, group, context)
        assert n >= 1 and size % M.BLOCK_KEYS == 0 and size > 0
        assert size * n >= context and size * (n - 1) < max(context, 1)          # every key once, no empty last split
        assert n <= 2 * M.MAX_CHOSEN_SPLITS
        if n > 1:
            assert size >= M.MIN_SPLIT_KEYS                                      # a split is worth its workgroup
    # more work than the chip has units is never cut finer than one split a unit would need
    size, n = M.choose_splits(4 * units, 8, 4, 2048)
    assert n == 1


def test_a_plan_for_uneven_contexts_has_room_for_every_pair(units):
    from pulse_infer_amd.ops import attention_mfma as M

    for nkv, group in ((8, 4), (1, 6), (2, 20), (16, 1)):
        slots, first = M.plan_slots(nkv, group)
        heads = nkv * ((group + 15) // 16)
        assert first >= 1 and slots == 2 * first and first * heads <= max(units, heads)   # one round fills the units once
    for items, splits in ((1, 8), (64, 8), (128, 8), (200, 5), (1024, 1)):
        assert M.plan_fits(items, splits)
        assert M.plan_ints(items, splits) == 1 + items * splits + items                    # count, pairs, split sizes
    assert not M.plan_fits(129, 8) and not M.plan_fits(0, 8)


def test_a_step_counts_as_uneven_by_its_longest_context_over_the_mean():
    from pulse_infer_amd.parts.base import UNEVEN_CONTEXTS, EntryMeta, contexts_uneven

    def metas(contexts):
        return [EntryMeta(i, i, c - 1, 1, i) for i, c in enumerate(contexts)]

    assert not contexts_uneven(metas([4096] * 8))
    assert not contexts_uneven(metas([9000, 10]))                     # two requests: nothing to order
    assert contexts_uneven(metas([4096, 200, 200, 200]))
    assert contexts_uneven(metas([1500, 1000, 500]))                  # exactly 1.5 times the mean
    assert not contexts_uneven(metas([1499, 1000, 500]))
    assert UNEVEN_CONTEXTS == 1.5
    # portions count with what they bring: a context is start + count
    assert contexts_uneven([EntryMeta(0, 0, 0, 900, 0), EntryMeta(1, 1, 99, 1, 900), EntryMeta(2, 2, 49, 1, 901)])


def test_prefill_splits_are_chosen_for_long_walks(units):
    from pulse_infer_amd.ops import attention_mfma as M

    choose = lambda entries, **kw: M.choose_prefill_splits(list(enumerate(entries)), 32, 8, 4, 128, kw.get("window", 0))
    assert choose([E(0, 128)]) == (0, 1)                      # short walks: nothing to gain
    assert choose([E(0, 2048)], window=256) == (0, 1)         # a window keeps them short
    assert M.choose_prefill_splits([(0, E(0, 4096))], 16, 8, 4, 96, 0) == (0, 1)     # no split variant for this head size
    for entries in ([E(16384 - 512, 512)], [E(4032, 64)], [E(0, 2048)], [E(0, 8192)], [E(100, 700), E(3000, 40)],
                    [E(39000, 1000)]):
        size, n = choose(entries)
        longest = max(e.start + e.count for e in entries)
        tokens = sum(e.count for e in entries)
        if n == 1:
            assert size == 0
            continue
        assert size % M.PREFILL_SPLIT_KEYS == 0 and size >= 8 * M.PREFILL_SPLIT_KEYS
        assert size * n >= longest and size * (n - 1) < longest + M.PREFILL_SPLIT_KEYS
        assert n <= M.PREFILL_MAX_SPLITS and tokens * 8 * 4 * 128 * 4 * n <= M.PREFILL_SCRATCH_BYTES
    assert choose([E(16384 - 64, 64)])[1] > 1                 # few items over a long context are cut
    # a full chip's walks are never cut
    if 2048 // 32 * 8 >= 2 * units:
        for entries in ([E(0, 2048)], [E(0, 8192)], [E(0, 4096), E(0, 8192)], [E(8192 - 512, 512)] * 8, [E(0, 30000)]):
            assert choose(entries) == (0, 1)


def test_library_products_share_out_a_wide_inner_dimension(units):
    import torch
    from pulse_infer_amd.parts.linear import Linear

    rows = lambda m, k: torch.empty(m, k, dtype=torch.bfloat16)
    for n, k in ((5120, 17408), (4096, 12288), (5120, 25600), (5120, 5120), (96, 8192)):
        lin = Linear(torch.empty(n, k, dtype=torch.bfloat16), "bfloat16")
        for m in (100, 192, 272, 544, 2048):
            shares = lin.library_shares_for(rows(m, k))
            assert shares in (0, 2, 4)
            if shares:
                assert m > Linear.SHARES_ROWS[1] and k >= Linear.LIBRARY_SHARES_MIN_K
                assert k % shares == 0 and (k // shares) % 64 == 0
    down = Linear(torch.empty(5120, 17408, dtype=torch.bfloat16), "bfloat16")
    assert down.library_shares_for(rows(272, 17408)) >= down.library_shares_for(rows(2048, 17408))   # fewer tiles, more shares
    assert Linear(torch.empty(64, 8192), "float32").library_shares_for(torch.empty(300, 8192)) == 0


def test_own_products_share_out_their_inner_dimension_evenly(units):
    import torch
    from pulse_infer_amd.parts.linear import Linear

    shape = lambda n, k: Linear(torch.empty(n, k, dtype=torch.bfloat16, device="meta"), "bfloat16")
    for n, k in ((4096, 12288), (4096, 4096), (5120, 17408), (5120, 25600), (96, 224), (1000, 384)):
        lin = shape(n, k)
        for m in (1, 12, 13, 64, 192, 193):
            x = torch.empty(m, k, dtype=torch.bfloat16)
            shares, waves = lin.shares_and_waves_for(x)
            if not Linear.SHARES_ROWS[0] <= m <= Linear.SHARES_ROWS[1] or n % 4:
                assert (shares, waves) == (0, 0)
            elif shares:
                assert k % shares == 0 and (k // shares) % 128 == 0 and waves in (4, 6) and 1 <= shares <= 16
    for n, k in ((24576, 4096), (34816, 5120), (51200, 5120), (448, 96), (12288, 2048)):
        lin = shape(n, k)
        for m in (17, 32, 64):
            waves = lin.swiglu_waves_for(m)
            assert waves in (0, 2, 4, 6, 10)
            if waves and n > 64 * units:
                # chosen only where no compute unit gets much more than its share of the weight rows
                groups = -(-n // (16 * waves))
                fullest = -(-groups // units) * 16 * waves
                assert fullest * units < 1.5 * n + 1.5 * units * (m // 2)


def test_which_products_of_many_rows_the_option_decides(units, monkeypatch):
    """Up to 255 rows the product in stages whatever the option says; from 256 on as it says: none of this package's, the tiled
    product for gate and up or for all, the product in stages where it takes them."""
    import torch
    from pulse_infer_amd.parts import linear
    from pulse_infer_amd.parts.linear import Linear

    gate_up = Linear(torch.empty(24576, 4096, dtype=torch.bfloat16, device="meta"), "bfloat16")
    o = Linear(torch.empty(4096, 4096, dtype=torch.bfloat16, device="meta"), "bfloat16")
    rows = lambda m: torch.empty(m, 4096, dtype=torch.bfloat16, device="meta")
    for policy in ("none", "stages", "swiglu", "all"):
        monkeypatch.setattr(linear, "OWN_MANY_ROWS", policy)
        for m in (64, 65, 255):
            assert gate_up.takes_stages(rows(m), swiglu=True) == (m >= 65) and not gate_up.takes_tiles(rows(m), swiglu=True)
            assert bool(o.stage_shares_for(rows(m))) == (m >= 65)
        for m in (256, 257, 512, 513, 768, 769, 1024, 1536, 1537):
            assert gate_up.takes_tiles(rows(m), swiglu=True) == (policy in ("swiglu", "all"))
            assert o.takes_tiles(rows(m)) == (policy == "all") == bool(o.tile_shares_for(rows(m)))
            if policy != "stages":
                assert not gate_up.takes_stages(rows(m), swiglu=True)
            if policy in ("none", "all"):
                assert not o.takes_stages(rows(m)) and not o.stage_shares_for(rows(m))
            if m > Linear.STAGE_ROWS_SHARES:
                assert not o.stage_shares_for(rows(m))
    monkeypatch.setattr(linear, "OWN_MANY_ROWS", "stages")
    small = Linear(torch.empty(4096, 1024, dtype=torch.bfloat16, device="meta"), "bfloat16")
    for m in (256, 257, 512, 513, 768, 769, 1536, 1537, 2048, 8192, 100000):
        assert gate_up.takes_stages(rows(m), swiglu=True)
        assert small.takes_stages(torch.empty(m, 1024, dtype=torch.bfloat16, device="meta"), swiglu=True)


def test_updates_of_many_rows_go_in_two_shares_while_these_fill_the_chip_once(monkeypatch):
    """As many tiles of 256 x 256 as half the compute units; with the library's products up to a hundred."""
    import torch
    from pulse_infer_amd.ops import device
    from pulse_infer_amd.parts import linear
    from pulse_infer_amd.parts.linear import Linear

    monkeypatch.setattr(device, "_units", 256)
    down = Linear(torch.empty(4096, 12288, dtype=torch.bfloat16, device="meta"), "bfloat16")      # (16 tiles a tile of rows)
    for policy, last in (("stages", 2048), ("swiglu", 2048), ("none", 1536)):
        monkeypatch.setattr(linear, "OWN_MANY_ROWS", policy)
        shares = [down.library_shares_for(torch.empty(m, 12288, dtype=torch.bfloat16, device="meta")) for m in (768, 769, last, last + 1, 8192)]
        assert shares == [4, 2, 2, 0, 0]


def test_shares_of_an_update_depend_on_the_weight_alone_up_to_192_rows(units):
    """17 to 64 rows (shared out over workgroups) and 65 to 192 (in stages): one cut each."""
    import torch
    from pulse_infer_amd.parts.linear import Linear

    for n, k in ((4096, 4096), (4096, 12288), (2560, 9728), (5120, 17408), (2048, 8192), (7168, 2048), (1000, 8192)):
        lin = Linear(torch.empty(n, k, dtype=torch.bfloat16, device="meta"), "bfloat16")
        rows = lambda m: torch.empty(m, k, dtype=torch.bfloat16, device="meta")
        assert len({lin.shares_and_waves_for(rows(m)) for m in (17, 33, 64, 100, 192)}) == 1
        cuts = {lin.stage_shares_for(rows(m)) for m in range(65, 193)}
        assert len(cuts) == 1 and cuts != {0}
        for m in (193, 255, 256, 300, 512):
            shares = lin.stage_shares_for(rows(m))
            assert 0 <= shares <= 16 and (shares == 0 or k % (64 * shares) == 0)


def test_a_projections_shares_depend_on_the_weight_alone_up_to_256_rows(monkeypatch):
    """One cut of q, k and v from 65 rows on, none to be had on one row and not on the next, wherever the whole product had one
    order of its sums; beyond 256 rows whole again where shares are no gain."""
    import torch
    from pulse_infer_amd.ops import device
    from pulse_infer_amd.parts import linear
    from pulse_infer_amd.parts.linear import Linear

    monkeypatch.setattr(device, "_units", 256)
    monkeypatch.setattr(linear, "OWN_MANY_ROWS", "stages")
    meta = lambda *shape: torch.empty(*shape, dtype=torch.bfloat16, device="meta")
    shares = lambda rows, n, k: Linear(meta(n, k), "bfloat16").parts_shares_for(meta(rows, k))
    for n, k in ((6144, 4096), (7168, 5120), (8192, 4096), (12288, 4096), (8192, 8192)):
        cuts = {shares(m, n, k) for m in range(65, 257)}
        assert len(cuts) == 1 and cuts != {0}, (n, k, cuts)
        cut = cuts.pop()
        assert k % (64 * cut) == 0
    for n, k in ((5120, 4096), (10240, 8192), (3072, 4096)):      # (some rows of these are the library's when whole)
        assert len({shares(m, n, k) for m in range(65, 257)} - {0}) == 1
    assert shares(128, 5120, 4096) and not shares(129, 5120, 4096) and not shares(192, 5120, 4096) and shares(193, 5120, 4096)
    assert not shares(64, 6144, 4096) and not shares(513, 6144, 4096)
    assert shares(357, 6144, 4096) == 4 and shares(384, 6144, 4096) == 4 and not any(shares(m, 6144, 4096) for m in (385, 448, 509, 512))
    assert shares(512, 7168, 5120) and shares(256, 18432, 7168) and not any(shares(m, 18432, 7168) for m in (257, 300, 512))
    assert not shares(97, 6144, 2560) and not shares(97, 6142, 4096) and not shares(97, 1000, 4096)
    monkeypatch.setattr(linear, "OWN_MANY_ROWS", "none")
    assert shares(255, 6144, 4096) == 4 and not shares(256, 6144, 4096) and not shares(357, 6144, 4096)


def test_updates_in_shares_of_many_rows_are_this_packages(units, monkeypatch):
    """Wherever an update beyond 192 rows is worth making in shares, the product in stages makes them, also of small
    weights, unless the option gives it to the tiled product or to the library."""
    import torch
    from pulse_infer_amd.parts import linear
    from pulse_infer_amd.parts.linear import Linear

    for n, k in ((4096, 12288), (5120, 17408), (2560, 9728), (1024, 8192), (256, 8192), (100, 8192)):
        lin = Linear(torch.empty(n, k, dtype=torch.bfloat16, device="meta"), "bfloat16")
        for m in (193, 256, 257, 357, 512, 513, 1024, 1536, 2048, 6400, 30000):
            x = torch.empty(m, k, dtype=torch.bfloat16, device="meta")
            for policy in ("stages", "swiglu"):
                monkeypatch.setattr(linear, "OWN_MANY_ROWS", policy)
                shares = lin.stage_shares_for(x)
                assert shares or not lin.library_shares_for(x)
                assert shares <= 16 and (not shares or k % (64 * shares) == 0)
                if m > Linear.STAGE_ROWS_SHARES:
                    assert bool(shares) == bool(lin.library_shares_for(x))
            monkeypatch.setattr(linear, "OWN_MANY_ROWS", "none")
            assert m < 256 or not lin.stage_shares_for(x)


def test_plain_products_in_stages_keep_the_compute_units_busy(monkeypatch):
    """Narrow weights whose tiles leave most units idle stay with the library, whose product can cut their inner dimension;
    what fills the chip goes in stages, beyond 512 rows where the library's own tiles do not fill it better."""
    import torch
    from pulse_infer_amd.ops import device, kernels
    from pulse_infer_amd.parts import linear
    from pulse_infer_amd.parts.linear import Linear

    monkeypatch.setattr(device, "_units", 256)
    monkeypatch.setattr(linear, "OWN_MANY_ROWS", "stages")
    takes = lambda m, n, k: Linear(torch.empty(n, k, dtype=torch.bfloat16, device="meta"), "bfloat16").takes_stages(
        torch.empty(m, k, dtype=torch.bfloat16, device="meta"))
    for n, k in ((576, 8192), (1536, 7168), (2048, 4096), (1024, 4096)):
        assert not any(takes(m, n, k) for m in (65, 97, 128, 192, 255))
    for n, k in ((6144, 4096), (7168, 4096), (8192, 2048), (12288, 4096)):
        assert all(takes(m, n, k) for m in (65, 97, 128, 192, 255))
    assert takes(357, 6144, 4096) and takes(512, 6144, 4096) and not takes(700, 4096, 4096) and not takes(1100, 6144, 4096)
    assert not takes(64, 6144, 4096) and not takes(300, 12288, 4096)
    # beyond 512 rows by the estimate (1,152 and 840, 941 and 922 flops a picosecond), but for tiles of 256 x 256 that fill every round ...
    assert takes(1300, 6144, 4096) and not takes(1280, 5120, 17408) and takes(1024, 7168, 5120) and not takes(1024, 8192, 4096)
    assert takes(2048, 6144, 4096) and not takes(8192, 6144, 4096) and not takes(4096, 4096, 4096) and not takes(1800, 8192, 4096)
    assert takes(4096, 4096, 12288) and takes(8192, 5120, 5120)
    assert takes(2048, 8192, 512) and takes(4096, 8192, 512) and not takes(8192, 8192, 512) and not takes(2048, 8192, 576)
    # ... and long inner dimensions in tiles of 192 x 256
    assert takes(1536, 5120, 17408) and not takes(1800, 5120, 17408) and not takes(4096, 5120, 25600) and takes(2560, 5120, 17408)
    for m in (65, 255, 256, 1024):
        for n, k in ((2112, 7168), (5120, 8192), (3072, 2048), (24576, 1536)):
            tile = kernels.gemm_stages_tile(m, n, k)
            if takes(m, n, k):
                tiles = -(-n // tile[0]) * -(-m // tile[1])
                assert tiles >= 0.33 * 256


def test_keys_of_four_steps_are_not_cut_over_workgroups(units):
    """attn_wide's splits: none up to a step of 32 keys for each of a workgroup's wavefronts; beyond, two to three steps or more each."""
    from pulse_infer_amd.ops import kernels as K

    assert all(K.attn_wide_splits(items, 2, keys) == 1 for items in (1, 4, 8, 32, 1000) for keys in (1, 32, 96, 97, 128))
    for items, keys in itertools.product((1, 4, 8, 32), (129, 160, 161, 256, 600, 1500, 40000)):
        n, steps = K.attn_wide_splits(items, 2, keys), (keys + 31) // 32
        assert 1 <= n <= 16 and (steps + n - 1) // n >= 3
        assert n == 1 or items * 2 * (n - 1) < 2 * units


def test_latent_rows_are_shared_out_in_whole_blocks(units):
    """attn_latent's splits: no more workgroups than units where an item is cut, none without a block, at most 64; its items hold
    every (token, head) of the entries once."""
    from pulse_infer_amd.ops import kernels as K

    for items, keys in itertools.product((1, 3, 8, 32, 200, 256, 1000), (1, 64, 65, 128, 600, 4097, 40000)):
        n, blocks = K.attn_latent_splits(items, keys), (keys + 63) // 64
        assert 1 <= n <= 64 and (n == 1 or items * n <= units)
        each = -(-blocks // n)
        assert (n - 1) * each < blocks <= n * each
    entries = [types.SimpleNamespace(first_row=a, count=n) for a, n in ((0, 1), (1, 7), (8, 64))]
    for nq in (1, 4, 12, 16, 20, 32, 40, 64):
        flat, hp = K.attn_latent_items(entries, nq)
        held = [(t, h) for t0, nt, h0, nh in zip(*[iter(flat)] * 4) for t in range(t0, t0 + nt) for h in range(h0, h0 + nh)]
        assert sorted(held) == [(t, h) for t in range(72) for h in range(nq)]
        assert all(nt * hp <= 32 and nh <= hp for nt, nh in zip(flat[1::4], flat[3::4]))


def test_nothing_but_the_copies_own_statement_touches_m0():
    """The check of the build: it passes a statement that sets the copies' place, and finds every other use."""
    from pulse_infer_amd.csrc import build

    place = "\ts_mov_b32 m0, s41                                           // 000000002A00: BEFC0029\n\ts_nop 0   // 0\n"
    copies = "\tglobal_load_lds_dwordx4 v1, s[2:3] offset:-4096 // 0\n\tv_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3] // 0\n"
    assert build.m0_misuses((place + copies) * 2) == []
    for wrong in ("\ts_mov_b32 m0, s3 // 0\n", "\ts_mov_b32 m0, -1 // 0\n\ts_nop 0\n", "\ts_set_gpr_idx_on s3, gpr_idx(SRC0) // 0\n",
                  "\tv_movrels_b32_e32 v1, v2 // 0\n", "\ts_add_u32 s1, m0, s2 // 0\n", "\ts_sendmsg sendmsg(MSG_INTERRUPT) // 0\n",
                  "\ts_mov_b32 m0, s3 // 0\n\tv_readlane_b32 s3, v1, m0 // 0\n"):
        assert build.m0_misuses(place + wrong + copies)
    if (lib := build.existing_library()) is not None:
        assert len(build.device_code(lib)) > 10 and build.device_code(__file__) == []


def test_walks_of_prompts_turn_only_where_two_workgroups_share_a_unit():
    """Shortest beside longest: where a launch's workgroups find a place at once, two a compute unit, whole walks, none in front."""
    from pulse_infer_amd.ops.library import load_variant

    turn = lambda d, items, heads, splits=1, values=0: load_variant("attn_mfma", {"PULSE_HEAD_DIM": d}).pulse_attn_prefill_turn(
        items, heads, splits, values or d)
    for d in (32, 64, 128):
        assert [turn(d, n, 8) for n in (1, 32, 33, 64, 65, 4096)] == [0, 0, 32, 32, 0, 0]
        assert turn(d, 3, 100) == 2 and turn(d, 1, 300) == 0 and turn(d, 40, 8, 2) == 0 and turn(d, 1 << 30, 60000) == 0
    assert turn(192, 12, 32) == 0 == turn(192, 12, 32, values=160) and turn(192, 12, 32, values=128) == 8 == turn(192, 12, 32, values=64)
    assert turn(96, 40, 8) == 0      # (a head size whose kernel takes its items in order)


def test_items_of_several_prompts_stand_in_the_order_of_their_walks():
    """The same items, the longest walks last; a single prompt's, and those of kernels that take them in order, as they were."""
    from pulse_infer_amd.ops import attention_mfma as M

    lists = [[(0, 2048)], [(0, 4096), (0, 512)], [(0, 512), (0, 4096)], [(3000, 70), (0, 513), (7000, 512), (100, 31)], [(0, 300)] * 5]
    for spans in lists:
        entries, row = [], 7
        for index, (start, count) in enumerate(spans):
            entries.append((index + 2, E(start, count)))
            entries[-1][1].first_row = row
            row += count
        for d, per in ((128, 32), (64, 8), (192, 128)):
            plain, made = M.build_items(entries, per), M.build_portions(entries, per, d)
            fours = lambda flat: [tuple(flat[i:i + 4]) for i in range(0, len(flat), 4)]
            assert sorted(fours(plain)) == sorted(fours(made)) and (len(spans) > 1 or plain == made)
            of = dict(entries)
            walks = [of[i].start + row0 - of[i].first_row + n for row0, n, i, _ in fours(made)]
            assert walks == sorted(walks)
            assert M.build_portions(entries, per, 96) == plain


def test_both_routers_refuse_rows_that_are_too_wide():
    """What the router alone refuses is refused also where few tokens' choices are grouped in its launch."""
    import ctypes
    from pulse_infer_amd.ops import library

    lib = library.load()
    room = ctypes.create_string_buffer(64)
    here = ctypes.c_void_p(ctypes.addressof(room) + 15 & ~15)
    i, f = ctypes.c_int, ctypes.c_float
    for hidden in (15360, 1 << 20):
        assert lib.pulse_moe_router(here, i(1), here, None, i(1), here, here, i(8), i(hidden), i(16), i(4), i(0), i(1), i(0), i(0), f(1.0), None)
        assert b"do not fit" in lib.pulse_last_error()
        assert lib.pulse_moe_router_grouped(here, here, None, here, here, i(8), i(hidden), i(16), i(4), i(0), i(1), i(0), i(0), f(1.0), i(16),
                                            i(32), i(17), here, here, here, here, here, None)
        assert b"moe_router_grouped" in lib.pulse_last_error() and b"do not fit" in lib.pulse_last_error()
