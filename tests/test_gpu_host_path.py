"""The native launch path (lastkv_amd._host) against the Python bodies of ops.py, over the argument
forms both take: same bits, same refusals."""

from __future__ import annotations

import array

import numpy as np
import pytest
import torch

from lastkv_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
B, HQ, HKV, D = 3, 8, 2, 128


class _Python:
    """Stands for _host and handles nothing, so that the Python bodies run."""

    def __getattr__(self, name):
        return lambda *args: None


class _Recorder:
    """_host, remembering for each call whether it was handled."""

    def __init__(self, host):
        self.host, self.handled = host, []

    def __getattr__(self, name):
        fn = getattr(self.host, name)

        def call(*args):
            out = fn(*args)
            self.handled.append(out is not None)
            return out

        return call


def _both(monkeypatch, make, native=True):
    """Runs make() (fresh state, then the call; returns tensors) natively and in Python; asserts equal bits
    and that the native path took the call (``native``)."""

    results = []
    ops._bind_host()
    ops._cu_count(torch.device(DEV, torch.cuda.current_device()))  # (a device's first call reads it in Python)
    real = ops._host
    for host in (_Recorder(real), _Python()):
        monkeypatch.setattr(ops, "_host", host)
        results.append(make())
        if isinstance(host, _Recorder):
            assert all(host.handled) == native and host.handled, host.handled
    monkeypatch.setattr(ops, "_host", real)
    for a, b in zip(*results):
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)


def _randn(seed, *shape):
    return torch.randn(shape, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV).bfloat16()


def _i32(*x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


def _tiled(seed, slots, blocks):
    return ops.TiledKV(_randn(seed, slots, HKV, blocks, 4096), _randn(seed + 1, slots, HKV, blocks, 4096))


def _paged(seed, pages):
    return ops.PagedKV(_randn(seed, HKV, pages, 4096), _randn(seed + 1, HKV, pages, 4096))


def _segments(form):
    if form == "tiled":
        return dict(older=_tiled(1, B, 8), older_len=200, local=_tiled(3, B, 4), local_len=70, local_start=40,
                    vscale=torch.tensor([0.5, 1.5], device=DEV))
    if form == "slots":  # slots, device lengths, no scale
        return dict(older=_tiled(1, 5, 8), older_len=_i32(200, 31, 0), older_slot=_i32(4, 0, 2), local=_tiled(3, 6, 4),
                    local_len=_i32(70, 65, 80), local_start=_i32(40, 0, 127), local_slot=_i32(5, 1, 0))
    if form == "older":
        return dict(older=_tiled(1, B, 8), older_len=256)
    if form == "local":
        return dict(local=_tiled(3, B, 4), local_len=128, local_start=5)
    pool = _paged(5, 64)
    table = torch.randperm(64, generator=torch.Generator().manual_seed(7)).to(DEV, torch.int32)
    wide = table[:45].view(B, 15)  # (tables as column ranges of a wider one)
    return dict(older=pool, older_table=wide[:, :8], older_len=_i32(200, 31, 256), vscale=torch.tensor([0.5, 1.5], device=DEV),
                local=pool, local_table=wide[:, 8:13], local_ring_blocks=4, local_len=_i32(70, 65, 128),
                local_start=_i32(40, 0, 100), out_scale=torch.tensor([0.75, 1.25], device=DEV))


@pytest.mark.parametrize("form", ["tiled", "slots", "older", "local", "paged"])
@pytest.mark.parametrize("call", ["plain", "strided4d", "outputs"])
def test_decode_forms(form, call, monkeypatch):
    seg = _segments(form)

    def make():
        q = _randn(11, B, HQ, D)
        kw = {}
        if call == "strided4d":
            q = _randn(11, B, HQ + 2, 1, D)[:, 1:HQ + 1]
            kw = dict(num_splits=2, sm_scale=0.1, kv_cache_hint=2)
        if call == "outputs":
            kw = dict(num_splits=3, out=torch.zeros(B, HQ + 1, D, dtype=torch.bfloat16, device=DEV)[:, :HQ],
                      lse=torch.zeros(B, HQ, device=DEV), workspace=torch.empty(1 << 20, dtype=torch.uint8, device=DEV))
        out = ops.decode_attention(q, **kw, **seg)
        return [out] + ([kw["lse"], kw["out"]] if call == "outputs" else [])

    _both(monkeypatch, make)


@pytest.mark.parametrize("form", ["tiled", "slots", "older", "paged"])
@pytest.mark.parametrize("call", ["plain", "strided", "ragged", "ragged_host"])
@pytest.mark.parametrize("tokens", [3, 40])
def test_prefill_forms(form, call, tokens, monkeypatch):
    seg = _segments(form)

    def make():
        if call.startswith("ragged"):
            lengths = [tokens, 1, 2]
            cu = np.array([0, tokens, tokens + 1, tokens + 3], dtype=np.int32)
            q = _randn(12, tokens + 3, HQ + 1, D)[:, :HQ]
            lse = torch.zeros(tokens + 3, HQ, device=DEV)
            return [ops.prefill_attention(q, lse=lse, cu_seqlens_q=_i32(*cu.tolist()), max_seqlen_q=max(lengths),
                                          cu_seqlens_q_host=cu if call == "ragged_host" else None, **seg), lse]
        if call == "plain":
            return [ops.prefill_attention(_randn(12, B, tokens, HQ, D), causal=False, **seg)]
        out = torch.zeros(B, tokens + 1, HQ, D, dtype=torch.bfloat16, device=DEV)[:, :tokens]
        ws = torch.empty(64 << 20, dtype=torch.uint8, device=DEV)
        return [ops.prefill_attention(_randn(12, B, 2 * tokens, HQ, D)[:, ::2], out=out, workspace=ws, num_splits=1,
                                      tile_waves=4 if tokens > 3 else 0, **seg)]

    _both(monkeypatch, make)


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("form", ["fused", "heads", "ragged", "ragged2d"])
@pytest.mark.parametrize("rounding", ["torch", "vllm"])
def test_epilogue_forms(paged, form, rounding, monkeypatch):
    L = 1 if form == "heads" else 20

    def make():
        ragged = form.startswith("ragged")
        lead = (L,) if ragged else (B, L)
        qkv = _randn(13, *lead, (HQ + 2 * HKV) * D)
        q, k, v = qkv.split([HQ * D, HKV * D, HKV * D], dim=-1)
        if form == "heads":
            q, k, v = (t.reshape(*lead, -1, D) for t in (q, k, v))
        cos, sin = (_randn(s, 1 if ragged or form == "fused" else B, L, D) for s in (14, 15))
        if form == "ragged2d":
            cos, sin = cos[0], sin[0]
        kw = dict(cu_seqlens=_i32(0, 1, 18, 20), max_seqlen=17) if ragged else {}
        pos = _i32(3, 60, 31)
        if paged:
            ring = deep = _paged(16, 40)
            tables = torch.arange(40, dtype=torch.int32, device=DEV)
            kw.update(ring_table=tables[:12].view(B, 4), ring_tokens=96, deep_table=tables[12:36].view(B, 8))
        else:
            ring, deep = _tiled(16, 4, 3), _tiled(18, B, 8)
            kw.update(ring_slot=_i32(3, 0, 1))
            pos = pos if ragged else 40
        w = _randn(20, 2, D)
        out = ops.qkv_epilogue(q, k, v, cos, sin, num_q_heads=HQ, num_kv_heads=HKV, q_norm_weight=w[0],
                               k_norm_weight=None if form == "heads" else w[1], eps=1e-5, positions=pos, ring=ring, deep=deep,
                               rounding=rounding, ring_v_mul=torch.tensor([0.5, 3.0], device=DEV) if rounding == "vllm" else None,
                               **kw)
        return [out, ring.k, ring.v, deep.k, deep.v]

    _both(monkeypatch, make)


@pytest.mark.parametrize("shape", [(64,), (5, 64), (2, 3, 64), (1, 4, 64), (4, 1, 64)])
def test_norm_and_silu_forms(shape, monkeypatch):
    wide = shape[:-1] + (3 * shape[-1],)

    def make():
        x = _randn(21, *wide)[..., :64] if len(shape) < 3 or shape[0] == 1 else _randn(21, *shape)
        r, w = _randn(22, *shape), _randn(23, 64)
        out = torch.zeros(shape, dtype=torch.bfloat16, device=DEV)
        a = ops.rmsnorm(x, w, 1e-5, residual=r)
        b = ops.rmsnorm(x, w, 1e-5, out=out)
        return [a, r, b, out, ops.silu_mul(x, r), ops.silu_mul(r, x, out=torch.zeros_like(out))]

    _both(monkeypatch, make)


def test_other_forms_reach_the_python_bodies(monkeypatch):
    """Forms only the Python bodies take: numpy lengths, a list of host offsets, four-dim rows."""

    seg = _segments("tiled")
    seg["older_len"] = np.int64(200)
    _both(monkeypatch, lambda: [ops.decode_attention(_randn(11, B, HQ, D), **seg)], native=False)
    rag = _segments("older")
    _both(monkeypatch, lambda: [ops.prefill_attention(_randn(12, 5, HQ, D), cu_seqlens_q=_i32(0, 1, 3, 5), max_seqlen_q=2,
                                                      cu_seqlens_q_host=[0, 1, 3, 5], **rag)], native=False)
    _both(monkeypatch, lambda: [ops.silu_mul(_randn(1, 2, 2, 2, 64), _randn(2, 2, 2, 2, 64))], native=False)


@pytest.mark.parametrize("bad", ["dtype", "heads", "len", "table", "workspace", "cpu", "norm", "silu", "aligned"])
def test_refused_calls_raise_as_before(bad):
    seg, q = _segments("tiled"), _randn(11, B, HQ, D)
    with pytest.raises((ValueError, _lib.LastKVNativeError)):
        if bad == "dtype":
            ops.decode_attention(q.float(), **seg)
        elif bad == "heads":
            ops.decode_attention(q[:, :7], **seg)
        elif bad == "len":
            ops.decode_attention(q, **dict(seg, local_len=129))
        elif bad == "table":
            ops.decode_attention(q, **dict(_segments("paged"), older_table=None))
        elif bad == "workspace":
            ops.decode_attention(q, num_splits=4, workspace=torch.empty(8, dtype=torch.uint8, device=DEV), **seg)
        elif bad == "cpu":
            ops.decode_attention(q.cpu(), **seg)
        elif bad == "norm":
            ops.rmsnorm(q, _randn(1, 64), 1e-5)
        elif bad == "silu":
            ops.silu_mul(q, q[:, :4])
        else:
            ops.rmsnorm(_randn(1, 4, 65)[:, 1:], _randn(1, 64), 1e-5)


@pytest.mark.parametrize("op", ["rmsnorm", "rmsnorm_in_place", "silu_in_place", "decode", "prefill", "epilogue"])
def test_a_reported_hip_error_raises_and_issues_the_call_once(op):
    """A HIP error that an earlier call left on the thread is reported by the next launch, whose kernel runs all
    the same: the call raises, as the Python bodies do, and its work is not issued a second time (in-place
    results would take it twice)."""

    x, r, w = _randn(1, 3, 64), _randn(2, 3, 64), _randn(3, 64)
    seg, q = _segments("tiled"), _randn(11, B, HQ, D)
    rows = [_randn(s, B, 1, n * D) for s, n in ((13, HQ), (14, HKV), (15, HKV))] + [_randn(s, 1, 1, D) for s in (16, 17)]
    ring = _tiled(18, B, 3)
    calls = {
        "rmsnorm": lambda: ops.rmsnorm(x, w, 1e-5, residual=r),
        "rmsnorm_in_place": lambda: ops.rmsnorm(x, w, 1e-5, out=x),
        "silu_in_place": lambda: ops.silu_mul(x, r, out=x),
        "decode": lambda: ops.decode_attention(q, num_splits=1, **seg),
        "prefill": lambda: ops.prefill_attention(q[:, None], **seg),
        "epilogue": lambda: ops.qkv_epilogue(*rows, num_q_heads=HQ, num_kv_heads=HKV, q_norm_weight=None, k_norm_weight=None,
                                             eps=1e-5, positions=3, ring=ring),
    }
    once = [x.clone(), r.clone()]
    if op == "rmsnorm":
        ops.rmsnorm(once[0], w, 1e-5, residual=once[1])
    elif op == "rmsnorm_in_place":
        ops.rmsnorm(once[0], w, 1e-5, out=once[0])
    elif op == "silu_in_place":
        ops.silu_mul(once[0], once[1], out=once[0])
    torch.cuda.synchronize()
    assert _lib.load().hipSetDevice(9999) != 0  # (resolved from the HIP runtime the library is linked with)
    with pytest.raises(_lib.LastKVNativeError, match="status 4"):
        calls[op]()
    torch.cuda.synchronize()
    assert torch.equal(x, once[0]) and torch.equal(r, once[1])


@pytest.mark.parametrize("what", ["norm_out", "residual", "silu_out", "decode", "prefill", "epilogue"])
def test_outputs_detach_copy_on_write_tensors(what):
    """A lazily cloned tensor shares its storage until one of the two is written: what a call writes (outputs, LSE,
    residual, caches, workspace) is the written tensor's own memory."""

    def lazy(t):
        return t, t.clone(), torch._lazy_clone(t)

    x, w = _randn(1, 3, 64), _randn(3, 64)
    q, seg = _randn(11, B, HQ, D), _segments("tiled")
    shared = []

    def out(t):
        shared.append(lazy(t))
        return shared[-1][2]

    if what == "norm_out":
        ops.rmsnorm(x, w, 1e-5, out=out(_randn(2, 3, 64)))
    elif what == "residual":
        ops.rmsnorm(x, w, 1e-5, residual=out(_randn(2, 3, 64)))
    elif what == "silu_out":
        ops.silu_mul(x, x, out=out(_randn(2, 3, 64)))
    elif what in ("decode", "prefill"):
        ws = torch.zeros(1 << 20, dtype=torch.uint8, device=DEV)
        if what == "decode":
            ops.decode_attention(q, num_splits=2, out=out(_randn(2, B, HQ, D)), lse=out(torch.zeros(B, HQ, device=DEV)),
                                 workspace=out(ws), **seg)
        else:
            ops.prefill_attention(_randn(12, B, 40, HQ, D), out=out(_randn(2, B, 40, HQ, D)),
                                  lse=out(torch.zeros(B, 40, HQ, device=DEV)),
                                  workspace=out(torch.zeros(4 << 20, dtype=torch.uint8, device=DEV)), **seg)
    else:
        ring, deep = (ops.TiledKV(*(out(t) for t in (kv.k, kv.v))) for kv in (_tiled(16, B, 3), _tiled(18, B, 8)))
        ops.qkv_epilogue(*(_randn(s, B, 20, n * D) for s, n in ((13, HQ), (14, HKV), (15, HKV))),
                         *(_randn(s, 1, 20, D) for s in (16, 17)), num_q_heads=HQ, num_kv_heads=HKV, q_norm_weight=None,
                         k_norm_weight=None, eps=1e-5, positions=3, ring=ring, deep=deep, q_out=out(_randn(2, B, 20, HQ, D)))
    torch.cuda.synchronize()
    for original, before, written in shared:
        assert torch.equal(original, before) and not torch.equal(written, before)


def test_a_failed_allocation_gives_the_host_offsets_back():
    """cu_seqlens_q_host is read through the buffer protocol: a call whose workspace cannot be allocated raises and
    keeps no hold of the caller's array (an array.array that is exported cannot grow)."""

    cu = array.array("i", [0, 40, 41, 43])
    q = _randn(12, 43, HQ, D)
    # (1.6 GB of workspace: the table could name that many blocks; more than any hole the allocator still has)
    table = (torch.arange(B * 32768, dtype=torch.int32, device=DEV) % 64).view(B, 32768)
    seg = dict(older=_paged(5, 64), older_table=table, older_len=_i32(200, 31, 256))
    out, cu_dev = torch.empty_like(q), _i32(*cu)
    ops.prefill_attention(q, out=out, cu_seqlens_q=cu_dev, max_seqlen_q=40, cu_seqlens_q_host=cu, **seg)
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction(1e-6)
    try:
        with pytest.raises(torch.cuda.OutOfMemoryError):
            ops.prefill_attention(q, out=out, cu_seqlens_q=cu_dev, max_seqlen_q=40, cu_seqlens_q_host=cu, **seg)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    cu.append(43)
