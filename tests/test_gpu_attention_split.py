"""GPU parity of the variants of the split-KV decode attention, at the sizes where the choice between
them changes, against the CPU oracle (float64 accumulation) with the tolerances of
test_gpu_attention.py: 2e-2 of the peak for bf16 KV, 6e-2 for FP8 KV."""
import ctypes as C
import math

import numpy as np
import pytest

import kv_testing as kt
import mlakv_ffi as ffi
import oracle_ffi as orc

pytestmark = pytest.mark.gpu

LATENT, ROPE = kt.LATENT, kt.ROPE
SCALE = 1.0 / math.sqrt(192.0)
TOL_BF16, TOL_FP8 = 2e-2, 6e-2


def _cache(ctxs, bs, seed, fp8=False, grow=None):
    """A filled one-layer cache and its table; `grow(position)` scales the rows of a sequence."""
    blocks = sum(-(-c // bs) for c in ctxs) + 3
    table = kt.build_tables(ctxs, bs, blocks, seed=seed).table()
    cache = kt.PagedCache(1, blocks, bs, fp8=fp8)
    total = sum(ctxs)
    latent, rope = kt.randn_bf16((1, total, LATENT), seed=seed + 1), kt.randn_bf16((1, total, ROPE), seed=seed + 2)
    if grow is not None:
        at = np.concatenate([np.arange(n) for n in ctxs])
        factor = kt.torch.as_tensor(grow(at), dtype=kt.torch.float32)[None, :, None]
        latent, rope = (latent.float() * factor).bfloat16(), (rope.float() * factor).bfloat16()
    kt.append(cache, latent.cuda(), rope.cuda(), kt.dev_i32(kt.slots_for(table, ctxs, bs)))
    return cache, table


def _check(cache, table, ctxs, heads, seed, fp8=False, sparse=None, **options):
    q = kt.randn_bf16((len(ctxs), heads, LATENT + ROPE), seed=seed).cuda()
    expected, expected_lse = kt.oracle_attention(cache, 0, q, table, ctxs, SCALE, sparse_indices=sparse)
    if sparse is None:
        out, lse, _ = kt.attention(cache, 0, q, kt.dev_i32(table), kt.dev_i32(ctxs), SCALE, **options)
    else:
        out, lse, _ = kt.sparse_attention(cache, 0, q, kt.dev_i32(table), kt.dev_i32(ctxs), kt.dev_i32(sparse), SCALE, **options)
    got, peak = out.float().cpu().numpy(), np.abs(expected).max()
    assert np.isfinite(got).all()
    assert np.abs(got - expected).max() <= (TOL_FP8 if fp8 else TOL_BF16) * peak
    live = np.asarray(ctxs) > 0
    assert np.abs(lse.cpu().numpy()[live] - expected_lse[live]).max() <= 2e-2


# Partials per sequence on average (256 units on a full chip): 85 (eight waves per head in the merge),
# 36 with 128 heads in two groups, 19 and 12 (four), 10 (one); empty sequences and sequences of one
# unit among them.
@pytest.mark.parametrize("ctxs,heads,fp8", [([3000, 1, 1900], 64, True), ([900, 2100, 40], 128, False), ([4096], 16, False),
                                            ([300] * 12 + [0], 48, False), ([130] * 21, 64, True), ([200] * 24 + [1700], 32, False)])
def test_merge_with_several_waves_per_head(ctxs, heads, fp8):
    cache, table = _cache(ctxs, 64, seed=901, fp8=fp8)
    # units of one tile as well: more partials than one round of the waves takes
    for options in ({"selection_units": 1}, {"chunk_tiles": 1}):
        _check(cache, table, ctxs, heads, seed=905, fp8=fp8, **options)


# The same merge in plans made for longer contexts, as a server's are: how many waves share a head goes by the
# partials that a sequence has, several from 9 partials on (1000 and 1100 tokens in units of 128: 8 and 9), with more
# than 1024 heads in the batch from 25 (1500 and 1620 tokens in units of 64: 24 and 26). Sequences with nothing to
# merge among them, and second head groups of 16 and 48 heads (80 and 112 in all).
@pytest.mark.parametrize("ctxs,heads,fp8,capacity", [([1000, 1100, 90], 64, False, 32768), ([896, 900, 1152, 1160], 112, True, 16384),
                                                     ([2000, 2100] * 6, 64, False, 8192), ([30, 0, 600], 48, True, 4096),
                                                     ([700, 2300, 33] * 4, 80, True, 8192),
                                                     ([1500, 1620, 300, 2600] * 5, 64, False, 8192)])
def test_merge_in_plans_of_longer_contexts(ctxs, heads, fp8, capacity):
    cache, table = _cache(ctxs, 64, seed=991, fp8=fp8)
    wide = np.zeros((len(ctxs), capacity // 64), dtype=table.dtype)
    wide[:, :table.shape[1]] = table
    for options in ({"selection_units": 1}, {"chunk_tiles": 2}, {"chunk_tiles": 4}):
        _check(cache, wide, ctxs, heads, seed=995, fp8=fp8, max_seq_len=capacity, **options)


# Rows that grow or fall along the context: the reference maxima of a head's waves lie far apart, and the weights of
# whole partials vanish beside those of others. Eight, four and one wave per head.
@pytest.mark.parametrize("rising", [True, False])
@pytest.mark.parametrize("ctxs,heads,fp8", [([3000, 5000], 64, False), ([2000, 600] * 6, 64, True), ([1500] * 24, 16, False)])
def test_merge_of_partials_with_unequal_weights(ctxs, heads, fp8, rising):
    longest = max(ctxs)
    cache, table = _cache(ctxs, 64, seed=985, fp8=fp8, grow=lambda at: 0.1 + 4.0 * (at if rising else longest - at) / longest)
    for options in ({"selection_units": 1}, {"chunk_tiles": 2}):
        _check(cache, table, ctxs, heads, seed=987, fp8=fp8, **options)


# Units of 16 heads shared by four workgroups (whole contexts and selections of 257 tokens and more while four
# per unit fit the 256 CUs): fewer tiles than workgroups, shares of different sizes, the last batch
# that fits (16 x 64 heads) and the first that is shared by two (17).
@pytest.mark.parametrize("ctxs,heads,fp8", [([768, 1, 0, 32, 33, 65, 96, 97, 129, 300], 64, True), ([257, 600, 40], 128, False),
                                            ([400, 31, 700], 16, True), ([320 + 7 * i for i in range(16)], 64, False),
                                            ([280] * 17, 64, False)])
def test_units_shared_by_four_workgroups(ctxs, heads, fp8):
    cache, table = _cache(ctxs, 64, seed=911, fp8=fp8)
    _check(cache, table, ctxs, heads, seed=915, fp8=fp8)
    rng = np.random.default_rng(917)
    for k in (257, 704):
        sparse = np.full((len(ctxs), k), -1, dtype=np.int32)
        for s, n in enumerate(ctxs):
            sparse[s, :min(n, k)] = rng.permutation(n)[:k]
        _check(cache, table, ctxs, heads, seed=919, fp8=fp8, sparse=sparse)


# A row of NaN spoils every head of its sequence, also where the merge's waves take one partial each
# and the one that holds it holds nothing else (three partials of the short sequence, eight waves).
# No tolerance: NaN everywhere in that sequence, the other sequence as without it.
@pytest.mark.parametrize("ctxs", [[32000, 300], [9000, 900] + [9000] * 10])
def test_merge_keeps_a_nan(ctxs):
    cache, table = _cache(ctxs, 64, seed=921)
    q = kt.randn_bf16((len(ctxs), 64, LATENT + ROPE), seed=925).cuda()
    arguments = (q, kt.dev_i32(table), kt.dev_i32(ctxs), SCALE)
    clean = kt.attention(cache, 0, *arguments, selection_units=1)[0]
    block, slot = int(table[1, 0]), 10
    cache.latent[0, block, slot, :] = float("nan")
    out, lse, _ = kt.attention(cache, 0, *arguments, selection_units=1)
    others = [s for s in range(len(ctxs)) if s != 1]
    assert kt.torch.isnan(out[1].float()).all() and kt.torch.isnan(lse[1]).all()
    assert kt.torch.equal(out[others], clean[others])


# A launch of four workgroups per unit holds sequences of two and three tiles too, whose last workgroups do not
# exist. With q = 0 every row has the same weight, and 32 rows of 3e38 add up to an infinity in fp32:
# infinite in the output whatever the number of workgroups, never 0 x infinity.
@pytest.mark.parametrize("tokens", [64, 96])
def test_workgroups_without_a_tile_leave_infinities_alone(tokens):
    ctxs = [300, tokens]
    cache, table = _cache(ctxs, 64, seed=931)
    last = (tokens - 32) // 64, (tokens - 32) % 64
    cache.latent[0, int(table[1, last[0]]), last[1]:last[1] + 32, 7] = 3e38
    q = kt.torch.zeros(2, 64, LATENT + ROPE, dtype=kt.torch.bfloat16, device="cuda")
    for options in ({}, {"selection_units": kt.ffi.ATTN_UNITS_HEAD_BLOCK_HALVES}):
        out, lse, _ = kt.attention(cache, 0, q, kt.dev_i32(table), kt.dev_i32(ctxs), SCALE, **options)
        assert kt.torch.isposinf(out[1, :, 7].float()).all(), options
        rest = [c for c in range(LATENT) if c != 7]
        assert kt.torch.isfinite(out[1][:, rest].float()).all() and kt.torch.isfinite(lse).all()


# Sharing a unit between four workgroups must not cost precision against two: error (2-norm, against the
# oracle's float64 sums) over rows that grow or fall along the context, where the parts' weights differ and
# every rounding of a part's rows shows (with bf16 slices it was 1.10 to 1.15 x that of two), and over equal
# ones. No margin: four parts of fp32 round once less than two of bf16.
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("shape", ["grow", "fall", "equal"])
def test_four_workgroups_are_as_precise_as_two(shape, fp8):
    ctxs, heads = [768, 500, 300, 257, 90], 64
    factor = {"grow": lambda at: 0.1 + at / 180.0, "fall": lambda at: 4.5 - at / 180.0, "equal": None}[shape]
    cache, table = _cache(ctxs, 64, seed=941, fp8=fp8, grow=factor)
    q = kt.randn_bf16((len(ctxs), heads, LATENT + ROPE), seed=945).cuda()
    expected, _ = kt.oracle_attention(cache, 0, q, table, ctxs, SCALE)
    errors = []
    for units in (kt.ffi.ATTN_UNITS_AUTO, kt.ffi.ATTN_UNITS_HEAD_BLOCK_HALVES):
        out, _, _ = kt.attention(cache, 0, q, kt.dev_i32(table), kt.dev_i32(ctxs), SCALE, selection_units=units)
        errors.append(np.linalg.norm(out.double().cpu().numpy() - expected) / np.linalg.norm(expected))
    assert errors[0] <= errors[1], errors


# A NaN query row gives a NaN output row and LSE, whatever merges it: one, four or eight waves per head (10, 16
# and 85 partials per sequence on average), the merge inside the launch, and a sequence that is not split.
@pytest.mark.parametrize("ctxs,options", [([900] * 24, {"selection_units": 1}), ([2000] * 16, {"selection_units": 1}),
                                          ([3000, 2000, 1000], {"selection_units": 1}),
                                          ([900, 400, 700], {"chunk_tiles": 2, "merge_mode": 1}), ([900, 400, 30], {"chunk_tiles": 100})])
def test_a_nan_query_head_gives_a_nan_row(ctxs, options):
    cache, table = _cache(ctxs, 64, seed=951)
    q = kt.randn_bf16((len(ctxs), 64, LATENT + ROPE), seed=955).cuda()
    arguments = (kt.dev_i32(table), kt.dev_i32(ctxs), SCALE)
    clean, clean_lse, _ = kt.attention(cache, 0, q, *arguments, **options)
    spoiled = q.clone()
    spoiled[1, 5] = float("nan")
    out, lse, _ = kt.attention(cache, 0, spoiled, *arguments, **options)
    assert kt.torch.isnan(out[1, 5].float()).all() and kt.torch.isnan(lse[1, 5])
    out[1, 5], lse[1, 5] = clean[1, 5], clean_lse[1, 5]
    assert kt.torch.equal(out, clean) and kt.torch.equal(lse, clean_lse)


# NaN rows that fill exactly the first group of eight partials of a sequence, with finite partials behind them:
# NaN from one wave per head (24 sequences; units of four tiles, the first of the long one with two of its
# own), from eight, and from the merge inside the launch.
@pytest.mark.parametrize("ctxs,options", [([40] * 23 + [20000], {"selection_units": 1}), ([600], {"chunk_tiles": 1}),
                                          ([600, 64], {"chunk_tiles": 1, "merge_mode": 1})])
def test_leading_nan_partials_spoil_the_row(ctxs, options):
    cache, table = _cache(ctxs, 64, seed=961)
    at = max(range(len(ctxs)), key=lambda s: ctxs[s])
    spoiled = 32 * (2 + 7 * 4) if ctxs[at] > 600 else 32 * 8
    for position in range(0, spoiled, 64):
        rows = min(64, spoiled - position)
        cache.latent[0, int(table[at, position // 64]), :rows] = float("nan")
    q = kt.randn_bf16((len(ctxs), 64, LATENT + ROPE), seed=965).cuda()
    out, lse, _ = kt.attention(cache, 0, q, kt.dev_i32(table), kt.dev_i32(ctxs), SCALE, **options)
    assert kt.torch.isnan(out[at].float()).all() and kt.torch.isnan(lse[at]).all()
    others = [s for s in range(len(ctxs)) if s != at]
    assert kt.torch.isfinite(out[others].float()).all()


SENTINEL = 0xA5


def _workspace_after(cache, table, ctxs, heads, sparse=None, selection_units=0):
    """The plan, and its workspace (filled with SENTINEL before) after one launch."""
    lib, batch, row = kt.ffi.load(), len(ctxs), 2 * (LATENT + ROPE)
    plan = kt.make_plan(batch, heads, max(ctxs) if sparse is None else sparse.shape[1], cache.block_size, cache.fp8,
                        selection=sparse is not None, selection_units=selection_units)
    workspace = kt.torch.full((int(plan.workspace_bytes),), SENTINEL, dtype=kt.torch.uint8, device="cuda")
    q = kt.randn_bf16((batch, heads, LATENT + ROPE), seed=975).cuda()
    out = kt.torch.zeros(batch, heads, LATENT, dtype=kt.torch.bfloat16, device="cuda")
    table_d, lens_d = kt.dev_i32(table), kt.dev_i32(ctxs)
    before = (C.byref(plan), C.byref(cache.view), 0, q.data_ptr(), heads * row, row, q.data_ptr() + 2 * LATENT, heads * row, row,
              table_d.data_ptr(), table_d.shape[1], lens_d.data_ptr())
    after = (SCALE, out.data_ptr(), 2 * heads * LATENT, 2 * LATENT, None, workspace.data_ptr(), int(plan.workspace_bytes), kt.stream_ptr())
    if sparse is None:
        kt.ffi.check(lib.mlakvAttnDecode(*before, *after))
    else:
        selection = kt.dev_i32(sparse)
        kt.ffi.check(lib.mlakvAttnDecodeSparse(*before, selection.data_ptr(), sparse.shape[1], *after))
    kt.torch.cuda.synchronize()
    return plan, workspace


# What halved units write: two workgroups per unit (asked for by the options) the first 2112 bytes x batch x heads
# that the header gives them, four (the plan's own choice) 8256 and more than 2112, where four per unit fit.
@pytest.mark.parametrize("k", [257, 512, 768])
def test_halved_units_keep_to_their_part_of_the_workspace(k):
    ctxs, heads = [k + 100, 900, k], 64
    cache, table = _cache(ctxs, 64, seed=971)
    sparse = np.stack([np.random.default_rng(973).permutation(n)[:k] for n in ctxs]).astype(np.int32)
    plan, workspace = _workspace_after(cache, table, ctxs, heads, sparse, kt.ffi.ATTN_UNITS_HEAD_BLOCK_HALVES)
    assert plan.reserved == 1 and (workspace[:1024 * heads] != SENTINEL).any()
    assert (workspace[2112 * len(ctxs) * heads:] == SENTINEL).all()
    plan, workspace = _workspace_after(cache, table, ctxs, heads, sparse)
    assert plan.reserved == 3 and (workspace[2112 * len(ctxs) * heads:] != SENTINEL).any()
    assert (workspace[8256 * len(ctxs) * heads:] == SENTINEL).all()


# Four workgroups per unit only where the XCD with the most sequences holds them all at once (32 CUs, sequence s on
# XCD s % 8), with more than 64 heads from 385 tokens on (FP8 289): seen in the workspace, where four write beyond
# the 2080 bytes x batch x heads of two.
@pytest.mark.skipif(not kt.torch.cuda.is_available() or kt.torch.cuda.get_device_properties(0).multi_processor_count != 256,
                    reason="the sizes are those of 256 CUs")
@pytest.mark.parametrize("batch,heads,most,fp8,parts", [
    (16, 64, 415, False, 4), (17, 64, 416, False, 2), (8, 128, 407, False, 4), (9, 128, 408, False, 2), (16, 48, 415, False, 4),
    (17, 48, 416, False, 2), (21, 48, 420, False, 2), (8, 80, 407, False, 4), (12, 80, 411, False, 2), (8, 112, 407, False, 4),
    (9, 112, 408, False, 2), (64, 16, 463, False, 4), (2, 128, 384, False, 2), (2, 128, 385, False, 4), (2, 80, 288, True, 2),
    (2, 80, 289, True, 4), (2, 64, 257, False, 4), (2, 64, 256, False, 1)])
def test_four_workgroups_only_where_an_xcd_holds_them(batch, heads, most, fp8, parts):
    ctxs = [most - i for i in range(batch)]
    cache, table = _cache(ctxs, 64, seed=981, fp8=fp8)
    _, workspace = _workspace_after(cache, table, ctxs, heads)
    assert bool((workspace[2112 * batch * heads:] != SENTINEL).any()) == (parts == 4)
    sparse = np.stack([np.r_[:n, [-1] * (most - n)] for n in ctxs]).astype(np.int32)
    plan, workspace = _workspace_after(cache, table, ctxs, heads, sparse)
    assert plan.reserved == (3 if parts == 4 else 1)
    assert bool((workspace[2112 * batch * heads:] != SENTINEL).any()) == (parts == 4)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("bs", [16, 32, 64])
def test_rows_of_zeros_inside_long_segments(bs, fp8):
    """Block-table entries that name no block inside segments of many more tiles than the ring holds:
    the tiles they reach are staged with an unknown number of loads, full waits until they have landed, and
    the counted waits of whole tiles resume behind them. Holes in the first tiles, alone, in a row, a ring
    apart and a few tiles before the end. A table that names a block of zeros instead gives the same bits (blocks
    of 16 slots: half a tile each)."""
    heads, tile = 64, 32
    ctxs = [1700, 900, 3000, 70, 640, 1311]
    cache, table = _cache(ctxs, bs, seed=1101, fp8=fp8)
    spare = sorted(set(range(cache.blocks)) - {int(b) for s, n in enumerate(ctxs) for b in table[s, :-(-n // bs)]})[0]
    broken, zeroed = table.copy(), table.copy()
    for s, tiles in enumerate([(9, 20, 21, 35, 39, 43), (0, 27), (2, 8, 9, 10, 11, 40, 88), (1,), (3, 7, 11, 15, 19), (1, 6, 30, 37)]):
        for n, at in enumerate(tiles):
            broken[s, at * tile // bs] = (-1, cache.blocks, 2 ** 31 - 1)[n % 3]
            zeroed[s, at * tile // bs] = spare
    q = kt.randn_bf16((len(ctxs), heads, LATENT + ROPE), seed=1105).cuda()
    expected, expected_lse = kt.oracle_attention(cache, 0, q, zeroed, ctxs, SCALE)
    # units of 100 tiles of the 64-head kernel: a sequence is one or two segments
    options = {"selection_units": ffi.ATTN_UNITS_SPLIT, "chunk_tiles": 100}
    out, lse, plan = kt.attention(cache, 0, q, kt.dev_i32(broken), kt.dev_i32(ctxs), SCALE, **options)
    assert plan.selection_units == ffi.ATTN_UNITS_SPLIT and plan.chunk_tiles == 100
    assert np.abs(out.float().cpu().numpy() - expected).max() <= (TOL_FP8 if fp8 else TOL_BF16) * np.abs(expected).max()
    assert np.abs(lse.cpu().numpy() - expected_lse).max() <= 2e-2
    whole, whole_lse, _ = kt.attention(cache, 0, q, kt.dev_i32(zeroed), kt.dev_i32(ctxs), SCALE, **options)
    assert kt.torch.equal(out, whole) and kt.torch.equal(lse, whole_lse)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("bs", [16, 48, 80, 24, 8])
def test_half_tiles_in_blocks_of_their_own(bs, fp8):
    """Blocks that hold whole half tiles (multiples of 16 slots that are none of 32): each half is fetched as a run of
    rows. The same bits as from blocks of 24 slots, where every row is located on its own (as in blocks of 8), for
    lengths that end on, before and behind a half; with holes in first and second halves the bits of a table that names a
    block of zeros there. The row scales of a block start off any 16-byte boundary."""
    heads = 64
    ctxs = [1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 700, 1296, 1311, 2000]
    caches = {}
    for size in (bs, 24):
        cache, table = _cache(ctxs, size, seed=1201, fp8=fp8)
        if fp8:
            padded = kt.torch.zeros(cache.blocks, size + 1, device="cuda")
            padded[:, :size] = cache.scale[0]
            cache.view.scale, cache.view.scale_block_stride = padded.data_ptr(), 4 * (size + 1)
            cache.padded = padded
        caches[size] = (cache, table)
    cache, table = caches[bs]
    general, general_table = caches[24]
    q = kt.randn_bf16((len(ctxs), heads, LATENT + ROPE), seed=1205).cuda()
    expected, _ = kt.oracle_attention(cache, 0, q, table, ctxs, SCALE)
    lens = kt.dev_i32(ctxs)
    spare = sorted(set(range(cache.blocks)) - {int(b) for s, n in enumerate(ctxs) for b in table[s, :-(-n // bs)]})[0]
    broken, zeroed = table.copy(), table.copy()
    for s, n in enumerate(ctxs):
        for at in range(s % 2, -(-n // bs), 5 if n > 100 else 2):
            broken[s, at] = (-1, cache.blocks, 2 ** 31 - 1)[at % 3]
            zeroed[s, at] = spare
    for options in ({"selection_units": ffi.ATTN_UNITS_SPLIT}, {"chunk_tiles": 100}, {"chunk_tiles": 3}):
        out, lse, _ = kt.attention(cache, 0, q, kt.dev_i32(table), lens, SCALE, **options)
        assert np.abs(out.float().cpu().numpy() - expected).max() <= (TOL_FP8 if fp8 else TOL_BF16) * np.abs(expected).max()
        if "chunk_tiles" in options:  # (the automatic cap of a unit goes by the block size)
            same, same_lse, _ = kt.attention(general, 0, q, kt.dev_i32(general_table), lens, SCALE, **options)
            assert kt.torch.equal(out, same) and kt.torch.equal(lse, same_lse)
        holes = [kt.attention(cache, 0, q, kt.dev_i32(t), lens, SCALE, quant=True, **options) for t in (broken, zeroed)]
        for got, want in zip(holes[0], holes[1]):
            assert not isinstance(got, kt.torch.Tensor) or kt.torch.equal(got, want)


# Units of 16 heads shared by five to eight workgroups, whole contexts: sequences of fewer tiles than workgroups, empty ones,
# shares of different sizes, the batches with the fewest and the most workgroups per unit (12, 9 and 8 x 64 heads: five, seven,
# eight), and every line of the rule from both sides. The workspace shows them: eight leave what lies behind their rows as it was,
# the split (13 x 64: four do not fit; lengths beyond a line) gives the bits of a plan that asks for it.
@pytest.mark.skipif(not kt.torch.cuda.is_available() or kt.torch.cuda.get_device_properties(0).multi_processor_count != 256,
                    reason="the sizes are those of 256 CUs")
@pytest.mark.parametrize("ctxs,heads,bs,fp8,many", [
    ([1760, 1, 0, 33, 1025, 257, 1500, 31], 64, 64, False, True), ([1761, 1, 0, 33, 1025, 257, 1500, 31], 64, 64, False, False),
    ([1760, 900, 40], 128, 16, True, True), ([1664, 900, 40], 128, 64, False, True), ([1665, 900, 40], 128, 64, False, False),
    ([1984, 5], 64, 64, False, True), ([1985, 5], 64, 64, False, False), ([1025], 16, 48, True, True), ([1024, 700], 64, 64, False, False),
    ([1100, 40, 224], 128, 16, True, True), ([1300 - 100 * i for i in range(12)], 64, 64, False, True),
    ([1760] + [50] * 11, 64, 64, True, True), ([1761] + [50] * 11, 64, 64, True, False), ([1856] + [70] * 9, 64, 64, True, True),
    ([1857] + [70] * 9, 64, 64, True, False), ([1984] + [70] * 9, 64, 64, False, True), ([1030 + 31 * i for i in range(9)], 64, 128, True, True),
    ([1300 - 90 * i for i in range(13)], 64, 64, True, False), ([1152, 3, 1100, 700, 65, 32], 80, 64, False, True),
    ([1153, 3, 1100, 700, 65, 32], 80, 64, False, False), ([1760, 900, 33], 80, 64, False, True), ([1536] + [60] * 24, 32, 64, False, True),
    ([1537] + [60] * 24, 32, 64, False, False), ([1984] + [60] * 24, 32, 64, True, True), ([1664] + [60] * 7, 96, 64, True, True),
    ([1665] + [60] * 7, 96, 64, True, False), ([1984] + [60] * 50, 16, 64, False, True)])
def test_contexts_in_units_shared_by_five_to_eight_workgroups(ctxs, heads, bs, fp8, many):
    cache, table = _cache(ctxs, bs, seed=1301, fp8=fp8)
    _check(cache, table, ctxs, heads, seed=1305, fp8=fp8)
    if many:
        _, workspace = _workspace_after(cache, table, ctxs, heads)
        used = 16512 * len(ctxs) * heads
        assert bool((workspace[8256 * len(ctxs) * heads:used] != SENTINEL).any())
        assert (workspace[used:] == SENTINEL).all()
    q = kt.randn_bf16((len(ctxs), heads, LATENT + ROPE), seed=1305).cuda()
    out, split = [kt.attention(cache, 0, q, kt.dev_i32(table), kt.dev_i32(ctxs), SCALE, selection_units=units)[0]
                  for units in (ffi.ATTN_UNITS_AUTO, ffi.ATTN_UNITS_SPLIT)]
    assert kt.torch.equal(out, split) == (not many)


# The same of selections: which plans share their units so (`reserved` 5; 3: between four, 1: otherwise), at the lines of the rule
# from both sides, and what the units and the split give for sequences shorter than the selection, empty ones and full ones.
@pytest.mark.skipif(not kt.torch.cuda.is_available() or kt.torch.cuda.get_device_properties(0).multi_processor_count != 256,
                    reason="the sizes are those of 256 CUs")
@pytest.mark.parametrize("batch,heads,fp8,expected", [
    (8, 64, False, {512: 3, 768: 3, 769: 5, 1536: 5, 1537: 1, 2048: 1}), (8, 64, True, {1024: 3, 1025: 5, 1536: 5, 1537: 1}),
    (4, 64, False, {769: 1, 1100: 1}), (2, 64, False, {769: 5, 1408: 5, 1409: 1}), (1, 16, True, {1024: 3, 1025: 5, 1280: 5, 1281: 1}),
    (9, 64, True, {1025: 5, 2048: 5}), (12, 64, False, {769: 5, 2048: 5}), (13, 64, False, {769: 1, 2048: 1}),
    (25, 32, False, {769: 5, 1664: 5, 1665: 1}), (25, 32, True, {2048: 5}), (8, 32, False, {1100: 1}), (16, 16, False, {2048: 5}),
    (12, 16, False, {1280: 5, 1281: 1}), (6, 128, False, {769: 5, 1408: 5, 1409: 1}), (4, 128, False, {1100: 1}), (9, 80, True, {1408: 5, 1409: 1})])
def test_selections_in_units_shared_by_five_to_eight_workgroups(batch, heads, fp8, expected):
    assert {k: kt.make_plan(batch, heads, k, 64, fp8, selection=True).reserved for k in expected} == expected
    ctxs = [2100 - 150 * i for i in range(min(batch, 12))] + [33] * (batch - 12)
    ctxs[batch // 2] = 0 if batch > 2 else ctxs[batch // 2]
    cache, table = _cache(ctxs, 64, seed=1307, fp8=fp8)
    rng = np.random.default_rng(1309)
    for k in (min(expected), max(k for k, how in expected.items() if how == max(expected.values()))):
        sparse = np.full((batch, k), -1, dtype=np.int32)
        for s, n in enumerate(ctxs):
            sparse[s, :min(n, k)] = rng.permutation(n)[:k]
        _check(cache, table, ctxs, heads, seed=1311, fp8=fp8, sparse=sparse)
        plan, workspace = _workspace_after(cache, table, ctxs, heads, sparse)
        if plan.reserved == 5:
            assert (workspace[16512 * batch * heads:] == SENTINEL).all()


# The slices of up to eight parts are fp32: no further from float64 than the split units' bf16 partials, over rows that grow
# along the context (the parts' weights lie far apart).
@pytest.mark.parametrize("fp8", [False, True])
def test_many_workgroups_are_as_precise_as_the_split(fp8):
    ctxs, heads = [1700, 1200, 1025, 300], 64
    cache, table = _cache(ctxs, 64, seed=1321, fp8=fp8, grow=lambda at: 0.1 + 4.0 * at / 1700)
    q = kt.randn_bf16((len(ctxs), heads, LATENT + ROPE), seed=1323).cuda()
    expected, _ = kt.oracle_attention(cache, 0, q, table, ctxs, SCALE)
    errors = []
    for options in ({}, {"selection_units": ffi.ATTN_UNITS_SPLIT}):
        out, _, _ = kt.attention(cache, 0, q, kt.dev_i32(table), kt.dev_i32(ctxs), SCALE, **options)
        errors.append(np.linalg.norm(out.float().cpu().numpy() - expected) / np.linalg.norm(expected))
    print(errors)
    assert errors[0] <= 1.02 * errors[1]


# The same of selections, whose rows the split locates one by one: over rows that grow or fall along the selection, and equal ones.
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("shape", ["grow", "fall", "equal"])
def test_selections_of_many_workgroups_are_as_precise_as_the_split(shape, fp8):
    ctxs, heads, k = [2100, 1500, 1400, 1700, 1450, 900, 1600, 33, 2000], 64, 1400
    factor = {"grow": lambda at: 0.1 + at / 500.0, "fall": lambda at: 4.3 - at / 500.0, "equal": None}[shape]
    cache, table = _cache(ctxs, 64, seed=1331, fp8=fp8, grow=factor)
    q = kt.randn_bf16((len(ctxs), heads, LATENT + ROPE), seed=1333).cuda()
    rng = np.random.default_rng(1335)
    sparse = np.full((len(ctxs), k), -1, dtype=np.int32)
    for s, n in enumerate(ctxs):
        sparse[s, :min(n, k)] = np.sort(rng.permutation(n)[:k])
    expected, _ = kt.oracle_attention(cache, 0, q, table, ctxs, SCALE, sparse_indices=sparse)
    errors, reserved = [], []
    for options in ({}, {"selection_units": ffi.ATTN_UNITS_SPLIT}):
        out, _, plan = kt.sparse_attention(cache, 0, q, kt.dev_i32(table), kt.dev_i32(ctxs), kt.dev_i32(sparse), SCALE, **options)
        errors.append(np.linalg.norm(out.double().cpu().numpy() - expected) / np.linalg.norm(expected))
        reserved.append(plan.reserved)
    assert reserved == [5, 1]
    assert errors[0] <= errors[1], errors


# Block-table entries that name no block, in units of 16 heads of one, two, four and eight workgroups, in blocks so small that a
# hole is some of a wavefront's rows and not all: in the first, the last and a middle share, over a whole share, at the ends of a
# sequence and in all of a short one; in a selection wherever its tokens lie. A table that names a block of
# zeros gives the same bits.
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("bs", [16, 64, 48, 8])
@pytest.mark.parametrize("parts", [1, 2, 4, 8])
def test_holes_in_units_of_16_heads(parts, bs, fp8):
    heads = 64
    ctxs = {1: [256, 200, 33, 129, 1], 2: [768, 257, 33, 640], 4: [768, 257, 33, 640], 8: [1700, 1025, 33, 640, 1311, 1696]}[parts]
    k = {1: 200, 2: 600, 4: 600, 8: 1100}[parts]
    options = {"selection_units": ffi.ATTN_UNITS_HEAD_BLOCK_HALVES} if parts == 2 else {}
    cache, table = _cache(ctxs, bs, seed=1341, fp8=fp8)
    spare = sorted(set(range(cache.blocks)) - {int(b) for s, n in enumerate(ctxs) for b in table[s, :-(-n // bs)]})[0]
    broken, zeroed = table.copy(), table.copy()
    for s, n in enumerate(ctxs):
        holes = [(20, n // 2, n - 1), (n - 1,), (0, n - 1), (), range(n // 8, n // 4), (n // 3, n // 2, n // 2 + 1, n - 5)][s]
        for at, position in enumerate(holes):
            broken[s, position // bs] = (-1, cache.blocks, 2 ** 31 - 1)[at % 3]
            zeroed[s, position // bs] = spare
    q = kt.randn_bf16((len(ctxs), heads, LATENT + ROPE), seed=1343).cuda()
    rng = np.random.default_rng(1345)
    sparse = np.full((len(ctxs), k), -1, dtype=np.int32)
    for s, n in enumerate(ctxs):
        sparse[s, :min(n, k)] = rng.permutation(n)[:k]
    lens, chosen = kt.dev_i32(ctxs), kt.dev_i32(sparse)
    expected, expected_lse = kt.oracle_attention(cache, 0, q, zeroed, ctxs, SCALE)
    got = [kt.attention(cache, 0, q, kt.dev_i32(t), lens, SCALE, **options)[:2] for t in (broken, zeroed)]
    split = kt.attention(cache, 0, q, kt.dev_i32(zeroed), lens, SCALE, selection_units=ffi.ATTN_UNITS_SPLIT)[0]
    assert not kt.torch.equal(got[1][0], split)  # (the units ran)
    assert np.abs(got[0][0].float().cpu().numpy() - expected).max() <= (TOL_FP8 if fp8 else TOL_BF16) * np.abs(expected).max()
    assert np.abs(got[0][1].cpu().numpy() - expected_lse).max() <= 2e-2
    assert kt.torch.equal(got[0][0], got[1][0]) and kt.torch.equal(got[0][1], got[1][1])
    got = [kt.sparse_attention(cache, 0, q, kt.dev_i32(t), lens, chosen, SCALE, **options) for t in (broken, zeroed)]
    assert got[0][2].reserved == {1: 1, 2: 1, 4: 3, 8: 5}[parts]
    assert kt.torch.equal(got[0][0], got[1][0]) and kt.torch.equal(got[0][1], got[1][1])


# A NaN query head gives a NaN row and a NaN cache row spoils its own sequence, whichever share of it holds the row; the others
# keep their bits. Units shared by eight workgroups, whole contexts and selections.
@pytest.mark.parametrize("fp8", [False, True])
def test_units_shared_by_five_to_eight_workgroups_keep_a_nan(fp8):
    ctxs, heads, k = [1700, 1300, 1025, 1400, 40, 1200], 64, 1100
    cache, table = _cache(ctxs, 64, seed=1351, fp8=fp8)
    q = kt.randn_bf16((len(ctxs), heads, LATENT + ROPE), seed=1353).cuda()
    sparse = np.stack([np.r_[:min(n, k), [-1] * (k - min(n, k))] for n in ctxs]).astype(np.int32)
    arguments = (kt.dev_i32(table), kt.dev_i32(ctxs))

    def both(query):
        return [kt.attention(cache, 0, query, *arguments, SCALE)[:2], kt.sparse_attention(cache, 0, query, *arguments, kt.dev_i32(sparse), SCALE)[:2]]

    clean = both(q)
    spoiled = q.clone()
    spoiled[1, 5] = float("nan")
    for (out, lse), (want, want_lse) in zip(both(spoiled), clean):
        assert kt.torch.isnan(out[1, 5].float()).all() and kt.torch.isnan(lse[1, 5])
        out[1, 5], lse[1, 5] = want[1, 5], want_lse[1, 5]
        assert kt.torch.equal(out, want) and kt.torch.equal(lse, want_lse)
    if fp8:
        cache.scale[0, int(table[3, 900 // 64]), 900 % 64] = float("nan")
    else:
        cache.latent[0, int(table[3, 900 // 64]), 900 % 64] = float("nan")
    others = [s for s in range(len(ctxs)) if s != 3]
    for (out, lse), (want, want_lse) in zip(both(q), clean):
        assert kt.torch.isnan(out[3].float()).all()
        assert kt.torch.equal(out[others], want[others]) and kt.torch.equal(lse[others], want_lse[others])


# Every way to say how long the contexts are leads to the same units shared by eight workgroups, and so does the quantising entry
# point: the lengths by value and a bound of them under a plan for 8192 tokens, a plan of the longest context, and the
# codes of that output with and without it.
@pytest.mark.parametrize("fp8", [False, True])
def test_units_shared_by_five_to_eight_workgroups_from_every_entry_point(fp8):
    lib, bs, heads = ffi.load(), 64, 64
    ctxs = [1700, 1, 0, 1030, 512]
    table = kt.build_tables(ctxs, bs, sum(-(-n // bs) for n in ctxs) + 3, seed=1361, max_blocks=8192 // bs).table()
    cache = kt.PagedCache(1, sum(-(-n // bs) for n in ctxs) + 3, bs, fp8=fp8)
    kt.append(cache, kt.randn_bf16((1, sum(ctxs), LATENT), seed=1362).cuda(), kt.randn_bf16((1, sum(ctxs), ROPE), seed=1363).cuda(),
              kt.dev_i32(kt.slots_for(table, ctxs, bs)))
    q = kt.randn_bf16((len(ctxs), heads, LATENT + ROPE), seed=1364).cuda()
    table_d, lens_d, row = kt.dev_i32(table), kt.dev_i32(ctxs), (LATENT + ROPE) * 2
    want, want_lse, _ = kt.attention(cache, 0, q, table_d, lens_d, SCALE)
    split = kt.attention(cache, 0, q, table_d, lens_d, SCALE, selection_units=ffi.ATTN_UNITS_SPLIT)[0]
    assert not kt.torch.equal(want, split)
    plan = kt.make_plan(len(ctxs), heads, 8192, bs, fp8)
    workspace = kt.torch.empty(int(plan.workspace_bytes), dtype=kt.torch.uint8, device="cuda")
    host = (C.c_int32 * len(ctxs))(*ctxs)
    head = (C.byref(plan), C.byref(cache.view), 0, q.data_ptr(), heads * row, row, q.data_ptr() + LATENT * 2, heads * row, row,
            table_d.data_ptr(), table_d.shape[1])
    for call, lengths in ((lib.mlakvAttnDecodeHostLens, (C.cast(host, C.c_void_p),)), (lib.mlakvAttnDecodeBounded, (lens_d.data_ptr(), 1700))):
        out, lse = kt.torch.full_like(want, float("nan")), kt.torch.full_like(want_lse, float("nan"))
        ffi.check(call(*head, *lengths, SCALE, out.data_ptr(), heads * LATENT * 2, LATENT * 2, lse.data_ptr(), workspace.data_ptr(),
                       workspace.numel(), kt.stream_ptr()))
        kt.torch.cuda.synchronize()
        assert kt.torch.equal(out, want) and kt.torch.equal(lse, want_lse)
    want_codes, want_scales = orc.mx_quant_rows(kt.bits16(want).reshape(-1, LATENT))
    for want_out in (False, True):
        out, lse, _, codes, scales = kt.attention(cache, 0, q, table_d, lens_d, SCALE, quant=True, want_out=want_out)
        assert (out is None or kt.torch.equal(out, want)) and kt.torch.equal(lse, want_lse)
        assert np.array_equal(codes.cpu().numpy().reshape(-1, LATENT), want_codes)
        assert np.array_equal(scales.cpu().numpy().reshape(-1, LATENT // 32), want_scales)


# Batches at the edges of a window of 64 sequences and with a window in the middle, whose lengths a workgroup asks for
# ahead: units that begin in every window (one workgroup goes through all of them, 300 take a few tiles each), empty
# sequences at the edges, a window without any tile. The same for selections, whose lengths are all the list's.
@pytest.mark.parametrize("batch", [64, 65, 128, 129, 192, 200])
@pytest.mark.parametrize("options", [{"selection_units": 1}, {"chunk_tiles": 3, "work_groups": 1}, {"chunk_tiles": 2, "work_groups": 7},
                                     {"chunk_tiles": 1, "work_groups": 300}])
def test_units_that_begin_in_every_window_of_sequences(batch, options):
    heads, fp8 = 16, batch % 2 == 1
    rng = np.random.default_rng(1401)
    ctxs = [int(n) for n in rng.integers(1, 150, batch)]
    for at in (0, 63, 64, 127, 128, 191):
        if at < batch - 1:
            ctxs[at] = 0
    if batch == 192:
        ctxs[64:128] = [0] * 64
    cache, table = _cache(ctxs, 16, seed=1403, fp8=fp8)
    _check(cache, table, ctxs, heads, seed=1405, fp8=fp8, **options)
    sparse = np.full((batch, 40), -1, dtype=np.int32)
    for s, n in enumerate(ctxs):
        sparse[s, :min(n, 40)] = rng.permutation(n)[:40]
    _check(cache, table, ctxs, heads, seed=1409, fp8=fp8, sparse=sparse, **options)


# One to ten partials per sequence, around the merge's groups of four, six and eight: the bits of the merge inside the
# launch, which takes eight at a time, and the oracle's values. (Units of 128 tokens, so few per sequence on average that no
# waves share a head.)
@pytest.mark.parametrize("heads,fp8,quant", [(64, False, False), (80, True, False), (16, True, True), (128, False, True)])
def test_groups_of_four_six_and_eight_partials(heads, fp8, quant):
    ctxs = [128 * i - i % 3 for i in range(1, 11)] + [0, 512, 513, 768, 769]
    cache, table = _cache(ctxs, 48, seed=1501, fp8=fp8, grow=lambda at: 0.1 + 3.0 * at / 1280)
    q = kt.randn_bf16((len(ctxs), heads, LATENT + ROPE), seed=1503).cuda()
    second, inside = [kt.attention(cache, 0, q, kt.dev_i32(table), kt.dev_i32(ctxs), SCALE, quant=quant, chunk_tiles=4, merge_mode=mode)
                      for mode in (ffi.ATTN_MERGE_SECOND_LAUNCH, ffi.ATTN_MERGE_IN_LAUNCH)]
    for got, want in zip(second, inside):
        assert not isinstance(got, kt.torch.Tensor) or kt.torch.equal(got, want)
    _check(cache, table, ctxs, heads, seed=1503, fp8=fp8, chunk_tiles=4)
