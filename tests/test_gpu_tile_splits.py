"""Key splits of the prefill tile kernel (GPU).

A call whose tile grid would leave CUs idle (few sequences, few query tiles) splits each tile's keys
over up to 4 workgroups when it leaves the split counts to the library (num_splits 0) and its
workspace holds the splits' states (lkv_prefill_workspace_bytes); each split writes its rows'
normalised fp32 O and base-2 LSE, and a merge kernel combines them.  In uniform calls two splits can
share a workgroup as its two halves, merged in LDS.  4-wave tiles split anywhere in their keys, unless
the older segment has 1 to 7 blocks: those calls take only equal splits that start inside it (one of 3
blocks runs unsplit, with the num_splits = 1 bits, as does a call with the minimum workspace).  The
bar is the north-star one against the oracle (outputs and LSE), on contiguous and paged caches, causal
and bidirectional; a ragged step (one long row among decode rows and a short row) takes the split too.
Each test asserts the route its calls take (lkv_prefill_plan).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from lastkv_amd import ops
from oracle import attention as A
from oracle import bf16

from test_gpu_decode import MAX_ABS, REL_L2, _bf, _t
from test_gpu_varlen import _ragged_case

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(rng, B, Hkv, T0, L, paged):
    """B sequences with an older segment of T0 tokens and a ring of L + 300 tokens from a random
    start; returns the kernel segments and the composed K / V (older V as bf16(V * s))."""

    R = (-(-(L + 300) // 32) + 2) * 32
    n1, start = L + 300, int(rng.integers(0, R))
    ok, ov = _bf(rng, (B, Hkv, T0, 128)), _bf(rng, (B, Hkv, T0, 128))
    lk, lv = _bf(rng, (B, Hkv, n1, 128)), _bf(rng, (B, Hkv, n1, 128))
    s = bf16.round_bf16(rng.uniform(0.4, 1.4, Hkv).astype(np.float32))
    older = ops.TiledKV.zeros(B, Hkv, -(-T0 // 32) * 32, DEV)
    ops.pack_kv(_t(ok), _t(ov), older)
    ring = ops.TiledKV.zeros(B, Hkv, R, DEV)
    first = min(n1, R - start)
    ops.pack_kv(_t(lk[:, :, :first]), _t(lv[:, :, :first]), ring, token0=start)
    if first < n1:
        ops.pack_kv(_t(lk[:, :, first:]), _t(lv[:, :, first:]), ring, token0=0)
    seg = dict(older_len=T0, vscale=torch.from_numpy(s).to(DEV), local_len=n1, local_start=start)
    if paged:
        ob, rb = older.k.shape[2], ring.k.shape[2]
        pool = ops.PagedKV.zeros(B * (ob + rb) + 1, Hkv, DEV)
        perm = torch.randperm(B * (ob + rb), generator=torch.Generator().manual_seed(5)).to(DEV, torch.int32)
        otab, rtab = perm[:B * ob].view(B, ob).contiguous(), perm[B * ob:].view(B, rb).contiguous()
        for b in range(B):
            for j in range(ob):
                pool.k[:, otab[b, j]], pool.v[:, otab[b, j]] = older.k[b, :, j], older.v[b, :, j]
            for j in range(rb):
                pool.k[:, rtab[b, j]], pool.v[:, rtab[b, j]] = ring.k[b, :, j], ring.v[b, :, j]
        seg.update(older=pool, older_table=otab, local=pool, local_table=rtab, local_ring_blocks=rb)
    else:
        seg.update(older=older, local=ring)
    k = np.concatenate([ok, lk], 2)
    v = np.concatenate([bf16.mul(ov, s.reshape(1, -1, 1, 1)), lv], 2)
    return seg, k, v


@pytest.mark.parametrize("T0", [3000, 70])
@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("causal", [True, False])
def test_key_splits_match_oracle_and_minimum_workspace_runs_unsplit(T0, paged, causal, prefill_plans):
    rng = np.random.default_rng(11 + 2 * paged + causal + T0)
    B, Hkv, G, L = 1, 2, 4, 512
    seg, k, v = _case(rng, B, Hkv, T0, L, paged)
    q = _bf(rng, (B, L, Hkv * G, 128))
    want, want_lse = A.attention(q.transpose(0, 2, 1, 3), k, v, causal_bottom_right=causal)
    want = bf16.round_bf16(want.transpose(0, 2, 1, 3).astype(np.float32))
    lse = torch.empty((B, L, Hkv * G), dtype=torch.float32, device=DEV)
    split = ops.prefill_attention(_t(q), causal=causal, lse=lse, **seg)  # automatic: 4 splits for T0 = 3000, none for 70
    got = split.float().cpu().numpy()
    ma, rl = A.max_abs(got, want), A.rel_l2(got, want)
    print(f"T0={T0} paged={paged} causal={causal}: key splits max_abs {ma:.2e} rel_l2 {rl:.2e}", flush=True)
    assert ma <= MAX_ABS and rl <= REL_L2
    np.testing.assert_allclose(lse.cpu().numpy(), want_lse.transpose(0, 2, 1), rtol=1e-4, atol=1e-4)
    unsplit = ops.prefill_attention(_t(q), causal=causal, num_splits=1, **seg)
    if T0 == 70:  # 3 older blocks: no equal split starts inside them
        assert torch.equal(split, unsplit)
    else:
        assert not torch.equal(split, unsplit)  # (the split merge rounds differently somewhere)
    # the minimum workspace (no room for the states): the same arithmetic as num_splits = 1
    need = ops.prefill_workspace_bytes(B, Hkv, T0, seg["local_len"], seg["local_start"] % 32)
    small = ops.prefill_attention(_t(q), causal=causal, workspace=torch.empty(need, dtype=torch.uint8, device=DEV),
                                  **seg)
    assert torch.equal(small, unsplit)
    assert prefill_plans == [(4, 1, 0, 0) if T0 == 70 else (4, 4, 1, 0), (4, 1, 0, 0), (4, 1, 0, 0)]


def test_ragged_step_long_row_takes_key_splits(prefill_plans):
    """One 300-token row among eleven one-token rows and a 7-token row: the long row's tiles split
    their keys (its older segment is not empty); every row within the bar of the oracle."""

    rng = np.random.default_rng(23)
    Hkv, G = 2, 4
    lengths = [1] * 5 + [300] + [1] * 6 + [7]
    seg, ks, vs, _ = _ragged_case(rng, lengths, Hkv, G, True, True)
    cu = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    q = _bf(rng, (int(cu[-1]), Hkv * G, 128))
    out = ops.prefill_attention(_t(q), causal=True, cu_seqlens_q=torch.from_numpy(cu).to(DEV),
                                max_seqlen_q=max(lengths), **seg)
    worst = 0.0
    for b in range(len(lengths)):
        rows = slice(int(cu[b]), int(cu[b + 1]))
        want, _ = A.attention(q[rows].transpose(1, 0, 2)[None], ks[b], vs[b], causal_bottom_right=True)
        want = bf16.round_bf16(want[0].transpose(1, 0, 2).astype(np.float32))
        got = out[rows].float().cpu().numpy()
        worst = max(worst, A.rel_l2(got, want))
        assert A.max_abs(got, want) <= MAX_ABS and A.rel_l2(got, want) <= REL_L2, f"sequence {b}"
    assert prefill_plans == [(4, 4, 0, 0)]
    print(f"ragged step with a long row: worst rel_l2 {worst:.2e}", flush=True)


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("T0,L,causal,wide,route", [
    (1500, 1024, True, False, (4, 1, 1)), (1500, 1024, False, False, (4, 1, 1)), (1501, 1021, True, False, (4, 1, 1)),
    (1500, 921, True, False, (4, 1, 1)), (1500, 897, False, True, (4, 1, 1)), (33, 1024, True, False, (4, 1, 0)),
    (-33, 1024, True, False, (4, 1, 1)), (1500, 1024, True, True, (4, 1, 1)), (800, 513, True, False, (4, 3, 0)),
    (800, 512, True, False, (4, 2, 1)), (801, 500, False, False, (4, 2, 1))])
def test_key_halves_of_one_workgroup_match_oracle(T0, L, causal, wide, route, paged, prefill_plans):
    """Uniform calls whose pairs of key splits share a workgroup (226 to 256 tiles of 128 rows: two halves; 126 and
    128 tiles with two splits: two halves of each; 130 tiles take three plain splits): equal and unequal halves, a
    ragged last block, an older segment too short to split (unsplit; with its length on the device, T0 < 0 here,
    the halves launch all the same and the second is empty) and a V value fp16 cannot hold (whose tiles run on
    the wide instance)."""

    on_device, T0 = T0 < 0, abs(T0)
    rng = np.random.default_rng(31 + T0 + L + causal + 2 * paged)
    B, Hkv, G = 1, 2, 16
    seg, k, v = _case(rng, B, Hkv, T0, L, paged)
    if on_device:
        seg.update({n: torch.tensor([seg[n]], dtype=torch.int32, device=DEV) for n in ("older_len", "local_len", "local_start")})
    if wide:
        seg["vscale"] = seg["vscale"] * 2.0 ** 17
        v = v.copy()
        v[:, :, :T0] *= 2.0 ** 17  # (a power of two: bf16(V s 2^17) = 2^17 bf16(V s))
    q = _bf(rng, (B, L, Hkv * G, 128))
    lse = torch.empty((B, L, Hkv * G), dtype=torch.float32, device=DEV)
    got = ops.prefill_attention(_t(q), causal=causal, lse=lse, **seg).float()
    assert prefill_plans == [(*route, 0)]
    kt, vt, qt = (torch.from_numpy(np.ascontiguousarray(x)).to(DEV).double() for x in (k[0], v[0], q[0]))
    n = kt.shape[1]
    hide = torch.arange(n, device=DEV)[None, :] > (n - L + torch.arange(L, device=DEV))[:, None]
    for h in range(0, Hkv * G, 5):
        s = qt[:, h] @ kt[h // G].t().contiguous() / 128 ** 0.5
        if causal:
            s = s.masked_fill(hide, float("-inf"))
        want = torch.softmax(s, -1) @ vt[h // G]
        torch.testing.assert_close(lse[0, :, h].double(), torch.logsumexp(s, -1), rtol=1e-4, atol=1e-4)
        want = want.bfloat16().double()
        assert float((got[0, :, h].double() - want).norm() / want.norm()) <= REL_L2


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("T0,n1,L,Hkv,G,shift,route", [
    (0, 1200, 100, 2, 4, 0.0, (4, 4, 1)), (0, 1201, 130, 3, 1, 8.0, (4, 4, 1)), (256, 900, 70, 1, 7, 8.0, (4, 4, 1)),
    (640, 1500, 257, 2, 2, 8.0, (4, 4, 1)), (1024, 33, 33, 2, 4, 8.0, (4, 4, 1)), (0, 129, 129, 2, 1, 8.0, (4, 1, 0))])
def test_key_splits_that_start_in_the_local_segment(T0, n1, L, Hkv, G, shift, route, paged, prefill_plans):
    """Few tiles over a short (or no) older segment: key splits start in the causal local segment, so some rows see
    no key in a split, row tiles end in padding, and halves get unequal blocks.  With ``shift`` every score sits
    near -90 (2^-130 against a zero reference: a row whose reference were not taken from the first block it sees
    would lose all of its probabilities)."""

    g = torch.Generator(device=DEV).manual_seed(T0 + n1 + L)
    rnd = lambda *shape: torch.randn(shape, generator=g, device=DEV)  # noqa: E731
    u = rnd(128)
    u = u / u.norm() * 128 ** 0.5
    q = (rnd(1, L, Hkv * G, 128) - shift * u).bfloat16()
    k = ((0.2 if shift else 1.0) * rnd(1, Hkv, T0 + n1, 128) + (u if shift else 0.0)).bfloat16()
    v = rnd(1, Hkv, T0 + n1, 128).bfloat16()
    R = -(-n1 // 32) * 32 + 64
    start = 45
    if paged:
        blocks = max(1, T0 // 32) + R // 32
        pool = ops.PagedKV.zeros(blocks, Hkv, DEV)
        table = torch.randperm(blocks, generator=torch.Generator().manual_seed(1)).to(DEV, torch.int32)[None]
        ot, rt = table[:, :max(1, T0 // 32)], table[:, max(1, T0 // 32):]
        if T0:
            ops.append_paged(k[:, :, :T0].transpose(1, 2), v[:, :, :T0].transpose(1, 2), pool, ot, token0=0)
        ops.append_paged(k[:, :, T0:].transpose(1, 2), v[:, :, T0:].transpose(1, 2), pool, rt, token0=start, wrap_tokens=R)
        i32 = lambda x: torch.tensor([x], dtype=torch.int32, device=DEV)  # noqa: E731
        seg = dict(older=pool, older_table=ot, older_len=i32(T0), local=pool, local_table=rt, local_len=i32(n1),
                   local_start=i32(start))
    else:
        ring = ops.TiledKV.zeros(1, Hkv, R, DEV)
        first = min(n1, R - start)
        ops.pack_kv(k[:, :, T0:T0 + first], v[:, :, T0:T0 + first], ring, token0=start)
        if first < n1:
            ops.pack_kv(k[:, :, T0 + first:], v[:, :, T0 + first:], ring, token0=0)
        seg = dict(local=ring, local_len=n1, local_start=start)
        if T0:
            older = ops.TiledKV.zeros(1, Hkv, T0, DEV)
            ops.pack_kv(k[:, :, :T0], v[:, :, :T0], older)
            seg.update(older=older, older_len=T0)
    lse = torch.empty((1, L, Hkv * G), dtype=torch.float32, device=DEV)
    got = ops.prefill_attention(q, causal=True, lse=lse, tile_waves=4, **seg)[0].float()
    # (129 keys: room for one split by the host's lengths, for more by the paged call's capacities)
    assert prefill_plans == [(4, 4, 0, 0) if paged and n1 == 129 else (*route, 0)]
    n = T0 + n1
    hide = torch.arange(n, device=DEV)[None, :] > (n - L + torch.arange(L, device=DEV))[:, None]
    want = torch.empty(L, Hkv * G, 128, dtype=torch.float64, device=DEV)
    for h in range(Hkv * G):
        s = (q[0, :, h].double() @ k[0, h // G].double().t().contiguous() / 128 ** 0.5).masked_fill(hide, float("-inf"))
        torch.testing.assert_close(lse[0, :, h].double(), torch.logsumexp(s, -1), rtol=1e-4, atol=1e-4)
        want[:, h] = torch.softmax(s, -1) @ v[0, h // G].double()
    want = want.bfloat16().double()
    assert float((got.double() - want).norm() / want.norm()) <= REL_L2
    assert float((got.double() - want).abs().max()) <= MAX_ABS


@pytest.mark.parametrize("B,L,T0,tile_waves,route", [
    (1, 40, 1500, 4, (4, 4, 1)), (1, 512, 1500, 0, (4, 2, 1)), (2, 300, 1500, 0, (4, 3, 0)), (1, 130, 0, 4, (4, 3, 0)),
    (1, 900, 1500, 0, (4, 1, 1))])
def test_a_nan_key_reaches_every_row_that_sees_it(B, L, T0, tile_waves, route, prefill_plans):
    """One NaN key in the local segment: exactly the rows that see it are NaN, with key splits (as halves of a
    workgroup, as states in memory, or both) as without, whichever split holds the key."""

    g = torch.Generator(device=DEV).manual_seed(B + L + T0)
    Hkv, G, n1 = 8, 4, L + 300
    rnd = lambda *shape: torch.randn(shape, generator=g, device=DEV).bfloat16()  # noqa: E731
    q, lk, lv = rnd(B, L, Hkv * G, 128), rnd(B, Hkv, n1, 128), rnd(B, Hkv, n1, 128)
    ring = ops.TiledKV.zeros(B, Hkv, -(-n1 // 32) * 32, DEV)
    seg = dict(local=ring, local_len=n1)
    if T0:
        older = ops.TiledKV.zeros(B, Hkv, -(-T0 // 32) * 32, DEV)
        ops.pack_kv(rnd(B, Hkv, T0, 128), rnd(B, Hkv, T0, 128), older)
        seg.update(older=older, older_len=T0)
    for at in (0, 299, n1 - 5, n1 - 1):  # (query row r sees keys up to r + 300)
        bad = lk.clone()
        bad[0, 1, at] = float("nan")
        ops.pack_kv(bad, lv, ring)
        want = torch.zeros(B, L, Hkv * G, 128, dtype=torch.bool, device=DEV)
        want[0, max(0, at - 300):, G:2 * G] = True
        for splits in (0, 1):
            got = ops.prefill_attention(q, causal=True, tile_waves=tile_waves, num_splits=splits, **seg)
            assert torch.equal(torch.isnan(got), want), f"key {at}, num_splits {splits}"
            assert prefill_plans.pop() == ((*route, 0) if splits == 0 else (4, 1, 0, 0))


def test_a_split_whose_first_scores_overflow_keeps_its_later_keys(prefill_plans):
    """4-wave tiles with key splits, every key range's first block at scores of -infinity (their fp32 sums
    overflow) and all later keys at one finite score of -1.02e33: the output is the mean of V over the later keys, as
    no finite score is lower than the reference of a row that has none yet.  (Every split holds as many keys: in an
    fp32 LSE of this magnitude the logarithm of their number is lost.)"""

    B, Hkv, G, L, n = 1, 2, 2, 64, 1024  # 32 blocks: four splits of two halves of 4
    q = torch.full((B, L, Hkv * G, 128), 8.0, dtype=torch.bfloat16, device=DEV)
    k = torch.full((B, Hkv, n, 128), -1e30, dtype=torch.bfloat16, device=DEV)
    v = torch.randn((B, Hkv, n, 128), generator=torch.Generator(device=DEV).manual_seed(2), device=DEV).bfloat16()
    first = (torch.arange(n, device=DEV) // 32) % 4 == 0
    k[:, :, first] = -3e38
    cache = ops.TiledKV.zeros(B, Hkv, n, DEV)
    ops.pack_kv(k, v, cache)
    # sm_scale log2(e) = 1: the scaled scores are the sums themselves
    got = ops.prefill_attention(q, local=cache, local_len=n, causal=False, sm_scale=float(np.log(2.0)), tile_waves=4)[0].double()
    assert prefill_plans == [(4, 4, 1, 0)]
    want = torch.stack([v[0, h // G, ~first].double().mean(0) for h in range(Hkv * G)]).bfloat16().double()[None]
    assert float((got - want).norm() / want.expand_as(got).norm()) <= REL_L2
