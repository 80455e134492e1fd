"""Which launches lkv_prefill_attn makes for the sequences above 64 query rows per kv head (lkv_prefill_plan),
by the rules its comments state.  The query reads no device memory, so it runs without a GPU (the library then
counts 256 CUs, an MI355X's)."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from lastkv_amd import _lib

PTR = 4096  # stands for an aligned device address


def plan(lengths, hq=32, hkv=8, older=0, local=0, num_splits=0, tile_waves=0, device_lengths=False, host=True, paged=False,
         ring=None, room=None):
    """(waves, splits, halves, mixed) of a call: ``lengths`` an int (one sequence), (batch, tokens) or a list of a
    ragged call's counts, over ``older`` + ``local`` keys, in the workspace lkv_prefill_workspace_bytes asks for, in
    that and ``room`` more bytes, or in the smallest (room -1)."""

    lib = _lib.load()
    a = _lib.PrefillArgs()
    a.struct_size = ctypes.sizeof(a)
    ragged = isinstance(lengths, list)
    B, L = (len(lengths), sum(lengths)) if ragged else lengths if isinstance(lengths, tuple) else (1, lengths)
    a.batch, a.tokens, a.num_q_heads, a.num_kv_heads, a.head_dim, a.causal = B, L, hq, hkv, 128, 1
    a.sm_scale = 128 ** -0.5
    a.q = a.out = PTR
    a.q_stride_t = a.out_stride_t = hq * 128
    a.q_stride_b = a.out_stride_b = L * hq * 128
    a.num_splits, a.tile_waves = num_splits, tile_waves
    if ragged:
        cu = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
        a.cu_seqlens_q, a.max_seqlen_q = PTR, max(lengths)
        if host:
            a.cu_seqlens_q_host = cu.ctypes.data
    blocks = lambda n: -(-n // 32)  # noqa: E731
    if older:
        a.older_k = a.older_v = PTR
        a.older_capacity_tokens, a.older_num_slots, a.older_num_pages = blocks(older) * 32, B, 1
        a.older_len_const = older
        if device_lengths:
            a.older_len = PTR
    if local:
        a.local_k = a.local_v = PTR
        a.local_ring_blocks, a.local_num_slots, a.local_num_pages = blocks(ring or local), B, 1
        a.local_len_const = local
        if device_lengths:
            a.local_len = PTR
    if paged:
        for seg, width in (("older", blocks(older)), ("local", blocks(ring or local))):
            setattr(a, f"{seg}_block_table", PTR)
            setattr(a, f"{seg}_table_stride", width)
            setattr(a, f"{seg}_page_stride", 4096)
    a.workspace = PTR
    a.workspace_bytes = (lib.lkv_prefill_workspace_min_bytes(ctypes.byref(a)) if room == -1 else
                         lib.lkv_prefill_workspace_bytes(ctypes.byref(a)) + (room or 0))
    info = _lib.PrefillPlanInfo()
    _lib.check(lib.lkv_prefill_plan(ctypes.byref(a), ctypes.byref(info)), "lkv_prefill_plan")
    return info.tile_waves, info.tile_splits, info.key_halves, info.rows_beside_tiles


def test_refused_arguments_are_refused_and_short_calls_have_no_tiles():
    with pytest.raises(_lib.LastKVNativeError, match="tile_waves"):
        plan(100, older=1024, tile_waves=3)
    assert _lib.load().lkv_prefill_plan(None, None) == 1
    assert plan(16, older=1024) == plan([16, 1, 3], older=1024) == (0, 0, 0, 0)


def test_waves_splits_and_the_smallest_workspace():
    assert plan((4, 1024), older=6144, local=2048) == (8, 1, 0, 0)  # 1024 4-wave tiles
    assert plan((3, 200), older=2048, local=1024) == (4, 3, 0, 0)  # 168 tiles: three in one round of 512 slots
    assert plan((3, 200), older=2048, local=1024, room=-1) == (4, 1, 0, 0)
    assert plan((3, 200), older=2048, local=1024, num_splits=1) == (4, 1, 0, 0)
    assert plan((3, 200), older=64, local=2048) == (4, 1, 0, 0)  # no equal split starts inside two older blocks
    assert plan((3, 200), local=2048) == (4, 3, 0, 0)
    assert plan(20, older=2048, local=1024) == (4, 4, 1, 0)  # 8 tiles: four splits of two halves
    assert plan(512, older=6144, local=1024) == (4, 2, 1, 0)  # 128 tiles
    assert plan(512, older=6144, local=1024, device_lengths=True, paged=True) == (4, 2, 1, 0)


@pytest.mark.parametrize("tokens,tiles,splits", [(544, 136, 3), (672, 168, 3), (704, 176, 4), (768, 192, 4), (800, 200, 2),
                                                 (896, 224, 2)])
def test_split_counts_of_one_round(tokens, tiles, splits):
    """Over 8K keys: as many splits as fit 512 slots, 4 instead of 2 while those are three workgroups a CU; a ragged
    call (with the decode rows' padding of the grid out of the count) 4 instead of 2 up to 223 tiles."""

    assert plan(tokens, older=6144, local=2048) == (4, splits, 0, 0)
    assert plan([tokens], older=6144, local=2048)[:3] == (4, 4 if 171 <= tiles < 224 else splits, 0)


@pytest.mark.parametrize("lengths,blocks,tiles", [((1, 160), 14, 40), ((1, 256), 22, 64), ((1, 512), 43, 128),
                                                  ((1, 672), 56, 168), ((1, 704), 71, 176), ((1, 864), 87, 216),
                                                  ((1, 896), 90, 224), ([700], 71, 176), ((2, 160), 27, 80), ((2, 360), 55, 192),
                                                  ((3, 100), 24, 96), ((4, 100), 32, 128), ((3, 200), 42, 168),
                                                  ((4, 180), 55, 192), ((4, 200), 64, 224)])
def test_key_splits_need_keys_for_their_states(lengths, blocks, tiles):
    """Tiles split from one key block per three of them on (per 2.5 above two thirds of the CUs; per four and 3.5 in
    calls of several sequences); first chunks and short contexts below run unsplit."""

    for n in (blocks - 1, blocks):
        for kw in ({}, dict(device_lengths=True)):  # (a device length counts as its capacity)
            got = plan(lengths, local=n * 32, **kw)
            assert (got[1] > 1) == (n == blocks), (n, got)


@pytest.mark.parametrize("lengths,hq,hkv,tiles,pairs", [
    ((1, 896), 32, 8, 224, 0), ((1, 900), 32, 8, 232, 1), ((1, 928), 32, 8, 232, 1), ((1, 1024), 32, 8, 256, 1),
    ((2, 470), 32, 8, 240, 1), ((1, 2560), 12, 12, 240, 1), ((3, 160), 64, 8, 240, 1), ((1, 1024), 28, 4, 224, 0),
    ((1, 480), 64, 8, 240, 1)])
def test_two_splits_run_as_pairs_when_they_fill_the_round(lengths, hq, hkv, tiles, pairs):
    """Grids of 224 to 256 tiles take two key splits (512 workgroup slots); as pairs in one workgroup each when
    that fills more than 7/8 of 256 CUs, at any split of the tiles over sequences and heads."""

    for kw in (dict(older=4096, local=lengths[1]), dict(older=4096, local=3000, device_lengths=True, paged=True)):
        got = plan(lengths, hq=hq, hkv=hkv, **kw)
        assert got == ((4, 1, 1, 0) if pairs else (4, 2, 0, 0)), (tiles, got)


def _step(rows, tokens, keys=8192, hq=32, hkv=8, **kw):
    """Whether a step of ``rows`` decode rows and one ``tokens``-token piece over ``keys`` keys (paged, lengths on the
    device, the recent 2048 in the ring) runs in one launch."""

    return plan([1] * rows + [tokens], hq=hq, hkv=hkv, older=keys - 2048, local=2048, device_lengths=True, paged=True, **kw)[3]


@pytest.mark.parametrize("rows,tokens,keys,hq,hkv,one", [
    (17, 64, 8192, 32, 8, 0), (20, 256, 8192, 32, 8, 0), (31, 512, 8192, 32, 8, 0), (32, 256, 8192, 32, 8, 0),
    (17, 1024, 8192, 32, 8, 1), (31, 1024, 8192, 32, 8, 1), (32, 1024, 8192, 32, 8, 1), (32, 1023, 8192, 32, 8, 0),
    (33, 64, 8192, 32, 8, 1), (250, 64, 8192, 32, 8, 1),  # more items than CUs
    (17, 64, 3072, 32, 8, 1), (17, 64, 3104, 32, 8, 0),  # few keys
    (17, 1024, 6144, 64, 8, 0), (31, 1024, 6144, 64, 8, 1), (14, 1024, 6144, 12, 12, 0), (22, 1024, 6144, 12, 12, 1)])
def test_decode_rows_share_the_tiles_launch_where_it_pays(rows, tokens, keys, hq, hkv, one):
    """One round of unsplit decode items (pairs of row and kv head above half the CUs, at most all of them) shares the
    launch over few keys or beside tiles of 128 to 288 query rows per decode row, larger classes always."""

    assert _step(rows, tokens, keys, hq, hkv) == one
    assert _step(rows, tokens, keys, hq, hkv, host=False) == 0  # (the class's size is not known)
    assert _step(rows, tokens, keys, hq, hkv, num_splits=1) == 0
    assert _step(rows, tokens, keys, hq, hkv, tile_waves=8) == 0


def test_split_decode_rows_share_the_launch_with_room_for_their_states():
    """Up to half as many items as CUs take key splits: their states must fit behind the tiles'."""

    for rows in (1, 9, 16):
        assert _step(rows, 256, room=64 << 20) == 1 and _step(rows, 256, room=-1) == 0
