"""The work that a program has this framework do, as cases that can be timed and checked.

Sizes come from the repository's benchmark and tests: the 8B attention shape (32 query heads, 8 kv
heads, head_dim 128, hidden 4096, MLP 14336, chunks of 1024 tokens), 8K and 128K contexts, and the
video model's 12 heads and 4,680-token blocks; a few other head counts stand for other models.

Kinds of cases:
  decode    one layer's one-token attention over [shared history | local ring], tiled caches, as the
            drop-in model's layers call it
  graph     several layers' fused QKV epilogue + paged decode attention, replayed from one HIP graph:
            a serving decode step without its projections
  prefill   one layer's chunked-prefill attention
  ragged    one layer's attention of a mixed serving step (decode rows and prefill pieces in one call)
  video     one layer's block attention through WanKVCache (bidirectional, paged history)
  epilogue  RoPE + q/k RMSNorm + K/V append of one layer's projections
  commit    the chunk-boundary blend of every layer's ring
  glue      the residual add + RMSNorm and the SwiGLU product of one decoder layer
  model     a whole call of the drop-in causal LM: a prompt from an empty cache, logits out
"""

import math
import random

import numpy as np
import torch
import torch.nn.functional as F

from lastkv_amd import ops
from lastkv_amd.llm import LastKVCache
from lastkv_amd.llm.configuration import CustomRecurrentMarinAKV254ReuseKVConfig
from lastkv_amd.llm.modeling import CustomRecurrentMarinAKV254ReuseKVForCausalLM
from lastkv_amd.videogen import WanKVCache

DEV = "cuda"
D = 128
BF16 = torch.bfloat16
EPS = 1e-5


# ------------------------------------------------------------------------------------------ cases
def listed():
    shape = dict(hq=32, hkv=8, chunk=1024)
    return [
        # one user's token a few thousand tokens into a chat: the smallest attention call, latency
        dict(name="decode_b1_2k", kind="decode", batch=1, position=2500, vscale=True, **shape),
        # the headline decode call: 32 sequences over 8K shared tokens
        dict(name="decode_b32_8k", kind="decode", batch=32, position=8192, vscale=False, all_older=True, **shape),
        # long context, few sequences: split keys, ring of one token beyond the previous chunk
        dict(name="decode_b4_128k", kind="decode", batch=4, position=131072, vscale=True, **shape),
        # a serving decode step of 8 sequences at 8K, 8 layers replayed from a graph (no host work)
        dict(name="graph_b8_8k", kind="graph", batch=8, position=8300, layers=8, vllm=False, **shape),
        # one user's 1024-token prompt piece at 7K
        dict(name="prefill_b1_8k", kind="prefill", batch=1, tokens=1024, position=7168, vscale=True, paged=False, **shape),
        # the last 1024-token piece of 32 prompts of 8K: the largest listed case
        dict(name="prefill_b32_8k", kind="prefill", batch=32, tokens=1024, position=7168, vscale=True, paged=False, **shape),
        # a serving step: 31 decode rows, one prefill piece and a 7-token row
        dict(name="ragged_31_1024_7", kind="ragged", decode_rows=31, long_tokens=1024, short_tokens=7, position=8192,
             **shape),
        # a video rollout's block 7 over its whole history
        dict(name="video_block7", kind="video", heads=12, block=4680, index=7),
        # the projections of 32 sequences' 1024-token pieces, final layer's shared append included
        dict(name="epilogue_32x1024", kind="epilogue", batch=32, tokens=1024, position=7168, vllm=False, deep=True,
             paged=True, **shape),
        # the boundary commit of 4 sequences, 32 layers
        dict(name="commit_b4_32l", kind="commit", layers=32, batch=4, hkv=8, chunk=1024, position=7168, vscale=True),
        # one layer's norm and SwiGLU over a 4096-token prefill step
        dict(name="glue_4096", kind="glue", rows=4096, hidden=4096, width=14336),
        # a 2300-token prompt through a two-layer model of the 8B layer shape: three chunks, every region
        dict(name="model_2300", kind="model", batch=1, tokens=2300, layers=2, hidden=4096, width=14336, vocab=32000,
             **shape),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


HEADS = [(32, 8), (32, 8), (16, 4), (32, 4), (8, 8), (64, 8), (28, 4), (12, 12)]


def draw(rng):
    kind = rng.choice(["decode", "decode", "graph", "prefill", "prefill", "ragged", "video", "epilogue", "epilogue",
                       "commit", "glue", "glue", "model"])
    hq, hkv = rng.choice(HEADS)
    chunk = rng.choice([256, 1024, 1024, 2048])
    shape = dict(hq=hq, hkv=hkv, chunk=chunk)
    if kind == "decode":
        batch = _log_int(rng, 1, 64)
        return dict(kind=kind, batch=batch, position=_log_int(rng, 100, min(131072, 2 ** 21 // (batch * hkv) * 2)),
                    vscale=rng.random() < 0.7, **shape)
    if kind == "graph":
        batch = _log_int(rng, 1, 32)
        return dict(kind=kind, batch=batch, position=_log_int(rng, 500, min(32768, 2 ** 21 // (batch * hkv))),
                    layers=rng.randint(2, 8), vllm=rng.random() < 0.5, **shape)
    if kind == "prefill":
        batch = _log_int(rng, 1, 16)
        tokens = _log_int(rng, 2, chunk)
        position = rng.randint(0, 16384) // chunk * chunk
        while batch * tokens * hq * (position + tokens) > 8e9:  # (the largest listed case: 8.6e9)
            batch, position = max(1, batch // 2), position // 2 // chunk * chunk
        return dict(kind=kind, batch=batch, tokens=tokens, position=position + rng.randint(0, chunk - tokens),
                    vscale=rng.random() < 0.7, paged=rng.random() < 0.5, **shape)
    if kind == "ragged":
        return dict(kind=kind, decode_rows=rng.randint(1, 40), long_tokens=_log_int(rng, 64, chunk),
                    short_tokens=rng.randint(2, 15), position=_log_int(rng, 500, 8192), **shape)
    if kind == "video":
        return dict(kind=kind, heads=rng.choice([12, 12, 24]), block=_log_int(rng, 500, 4680) // rng.choice([1, 2]),
                    index=rng.randint(1, 7))
    if kind == "epilogue":
        batch = _log_int(rng, 1, 32)
        tokens = min(chunk, _log_int(rng, 1, 1024))
        return dict(kind=kind, batch=batch, tokens=tokens, position=rng.randint(0, 8) * chunk + rng.randint(0, chunk - tokens),
                    vllm=rng.random() < 0.5, deep=rng.random() < 0.3, paged=rng.random() < 0.7, **shape)
    if kind == "commit":
        chunk = rng.choice([256, 1000, 1024])
        return dict(kind=kind, layers=_log_int(rng, 1, 32), batch=rng.randint(1, 4), hkv=hkv if hkv < 12 else 8,
                    chunk=chunk, position=rng.randint(0, 7) * chunk, vscale=rng.random() < 0.7)
    if kind == "glue":
        hidden = rng.choice([1536, 2048, 4096, 5120, 8192])
        return dict(kind=kind, rows=_log_int(rng, 1, 8192), hidden=hidden, width=8 * rng.randint(hidden // 4, hidden // 2))
    return dict(kind="model", batch=rng.randint(1, 2), tokens=rng.randint(64, 1800), layers=2, hidden=2048, width=5632,
                vocab=16000, hq=16, hkv=4, chunk=rng.choice([256, 1024]))


# ------------------------------------------------------------------------------------------ inputs
def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed((int(seed) * 1000003 + salt * 7919) % (1 << 62))


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV, dtype=BF16)


def _unit(g, *shape):
    """Gates and scales around 1: bf16 values carried as fp32."""

    return (torch.rand(shape, generator=g, device=DEV) + 0.5).to(BF16).float()


def _regions(c, tokens=1):
    """(older keys, local keys) of a call whose last token is position + tokens - 1: the recent chunk and
    the current one are local, what lies before them is the shared history."""

    last = c["position"] + tokens - 1
    if c.get("all_older"):
        return c["position"], 0
    older = max(0, last // c["chunk"] * c["chunk"] - c["chunk"])
    return older, last + 1 - older


def _kv(g, batch, heads, tokens):
    return _randn(g, batch, heads, tokens, D), _randn(g, batch, heads, tokens, D)


def _blocks(tokens):
    return -(-tokens // 32)


def _ring_tiled(k, v, start, ring_tokens):
    """A ring holding k / v [B, H, n, 128] at ring tokens start, start + 1, ... (wrapping)."""

    ring = ops.TiledKV.zeros(k.shape[0], k.shape[1], ring_tokens, DEV)
    first = min(k.shape[2], ring_tokens - start)
    if first:
        ops.pack_kv(k[:, :, :first], v[:, :, :first], ring, token0=start)
    if first < k.shape[2]:
        ops.pack_kv(k[:, :, first:], v[:, :, first:], ring, token0=0)
    return ring


def _page_tables(batch, older_tokens, rings, ring_tokens):
    """(pages, older table [B, W], ring tables [rings, B, R / 32]): shared pages in runs of 32 per
    sequence, interleaved over the sequences as 1024-token prefill steps hand them out."""

    w, rb = max(1, _blocks(older_tokens)), ring_tokens // 32
    j, b = np.arange(w)[None, :], np.arange(batch)[:, None]
    older = (j // 32) * (32 * batch) + b * 32 + j % 32
    base = _blocks(w) * 32 * batch
    ring = base + np.arange(rings * batch * rb).reshape(rings, batch, rb)
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a.astype(np.int32))).to(DEV)  # noqa: E731
    return int(base + rings * batch * rb + 1), to(older), to(ring)


def _bthd(x):
    return x.transpose(1, 2)


def _rope_rows(positions):
    """cos / sin [B, n, 128] in bf16 for integer positions [B, n]."""

    inv = 1.0 / (500000.0 ** (torch.arange(0, D, 2, device=DEV, dtype=torch.float32) / D))
    f = positions[..., None].float() * inv
    e = torch.cat((f, f), -1)
    return e.cos().to(BF16), e.sin().to(BF16)


def _attention_inputs(c, seed):
    """Logical inputs of the decode and prefill kinds."""

    L = c.get("tokens", 1)
    n0, n1 = _regions(c, L)
    g = _gen(seed)
    q = _randn(g, c["batch"], L, c["hq"], D)
    ok, ov = _kv(g, c["batch"], c["hkv"], n0)
    lk, lv = _kv(g, c["batch"], c["hkv"], n1)
    vs = _unit(g, c["hkv"]) if c["vscale"] else None
    return q, ok, ov, lk, lv, vs


def _ragged_rows(c):
    rows = [1] * c["decode_rows"] + [c["long_tokens"], c["short_tokens"]]
    cur = c["position"] // c["chunk"] * c["chunk"]
    older = max(0, cur - c["chunk"])
    # decode rows are position - cur tokens into their chunk; the others start it
    local = [cur - older + n + (c["position"] - cur if n == 1 else 0) for n in rows]
    return rows, older, local


def _ragged_inputs(c, seed):
    rows, older, local = _ragged_rows(c)
    g = _gen(seed)
    q = _randn(g, sum(rows), c["hq"], D)
    ok, ov = _kv(g, len(rows), c["hkv"], older)
    lk, lv = _kv(g, len(rows), c["hkv"], max(local))
    return rows, older, local, q, ok, ov, lk, lv, _unit(g, c["hkv"])


def _graph_inputs(c, seed):
    g = _gen(seed)
    B, Ln, p = c["batch"], c["layers"], c["position"]
    n0, n1 = _regions(c)
    qkv = _randn(g, Ln, B, (c["hq"] + 2 * c["hkv"]) * D)
    ok, ov = _kv(g, B, c["hkv"], n0)
    rings = [_kv(g, B, c["hkv"], n1 - 1) for _ in range(Ln)]
    vs = _unit(g, Ln, c["hkv"])
    qw, kw = _unit(g, D).to(BF16), _unit(g, D).to(BF16)
    cos, sin = _rope_rows(torch.full((B, 1), p, device=DEV))
    return qkv, ok, ov, rings, vs, qw, kw, cos, sin, n0, n1


def _epilogue_inputs(c, seed):
    g = _gen(seed)
    B, L, hq, hkv = c["batch"], c["tokens"], c["hq"], c["hkv"]
    qkv = _randn(g, B, L, (hq + 2 * hkv) * D)  # rows of one fused projection
    qw, kw = _unit(g, D).to(BF16), _unit(g, D).to(BF16)
    pos = c["position"] + torch.arange(L, device=DEV)[None, :].expand(B, L)
    cos, sin = _rope_rows(pos)
    mul = (1.0 / _unit(g, hkv)) if c["vllm"] else None
    return qkv, qw, kw, cos, sin, mul


def _commit_inputs(c, seed):
    g = _gen(seed)
    L, B, H, C, p = c["layers"], c["batch"], c["hkv"], c["chunk"], c["position"]
    R = ops.ring_tokens_for_chunk(C)
    # values in the tiled layout (any bits are some K/V)
    rk, rv = _randn(g, L, B, H, R // 32, 4096), _randn(g, L, B, H, R // 32, 4096)
    cap = _blocks(p + C)
    dk, dv = _randn(g, B, H, cap, 4096), _randn(g, B, H, cap, 4096)
    alpha = torch.rand(L * H, generator=g, device=DEV).to(BF16)
    vs = _unit(g, L * H) if c["vscale"] else None
    return rk, rv, dk, dv, alpha.float(), (1 - alpha).to(BF16).float(), vs, R


def _glue_inputs(c, seed):
    g = _gen(seed)
    x, res = _randn(g, c["rows"], c["hidden"]), _randn(g, c["rows"], c["hidden"])
    w = _unit(g, c["hidden"]).to(BF16)
    return x, res, w, _randn(g, c["rows"], 2 * c["width"])  # gate | up: rows of one fused projection


def _video_inputs(c, seed):
    g = _gen(seed)
    H, S = c["heads"], c["block"]
    blocks = [[(_randn(g, 1, S, H, D), _randn(g, 1, S, H, D)) for _ in range(2)] for _ in range(c["index"])]
    gates = torch.randn((2, H), generator=g, device=DEV)
    return blocks, gates, _randn(g, 1, S, H, D), _randn(g, 1, S, H, D), _randn(g, 1, S, H, D)


def _model_config(c):
    return CustomRecurrentMarinAKV254ReuseKVConfig(
        vocab_size=c["vocab"], hidden_size=c["hidden"], intermediate_size=c["width"], num_hidden_layers=c["layers"],
        num_attention_heads=c["hq"], num_key_value_heads=c["hkv"], head_dim=D, rope_theta=500000.0, rms_norm_eps=EPS,
        chunk_size=c["chunk"])


def _model(c, seed):
    with torch.device(DEV):
        model = CustomRecurrentMarinAKV254ReuseKVForCausalLM(_model_config(c)).to(BF16).eval()
    g = _gen(seed)
    with torch.no_grad():
        for p in model.parameters():
            if p.dim() == 2:
                p.normal_(0.0, 0.02, generator=g)
        for layer in model.model.layers:
            att = layer.self_attn
            att.prev_chunk_alphas.normal_(generator=g)
            if att.config.deep_kv_rescale:
                att.deep_v_scale.uniform_(0.5, 1.5, generator=g)
    ids = torch.randint(0, c["vocab"], (c["batch"], c["tokens"]), generator=g, device=DEV)
    return model, ids


# ------------------------------------------------------------------------------------------ prepare
def prepare(case, seed):
    s = {"kind": case["kind"], "case": case}
    s.update(globals()["_prepare_" + case["kind"]](case, seed))
    return s


def _segments_tiled(c, ok, ov, lk, lv, vs):
    n0, n1 = ok.shape[2], lk.shape[2]
    seg = {}
    older = ops.TiledKV.zeros(c["batch"], c["hkv"], max(32, _blocks(n0) * 32), DEV)
    if n0:
        ops.pack_kv(ok, ov, older)
    seg.update(older=older, older_len=n0, vscale=vs)
    if n1:
        R = ops.ring_tokens_for_chunk(c["chunk"])
        seg.update(local=_ring_tiled(lk, lv, n0 % R, R), local_len=n1, local_start=n0 % R)
    return seg


def _fill_pool(c, ok, ov, rings, rows):
    """A page pool with the older segment and one ring per entry of ``rings``, and its tables."""

    n0 = ok.shape[2]
    R = ops.ring_tokens_for_chunk(c["chunk"])
    pages, otab, rtab = _page_tables(rows, n0, len(rings), R)
    pool = ops.PagedKV.zeros(pages, c["hkv"], DEV)
    if n0:
        ops.append_paged(_bthd(ok), _bthd(ov), pool, otab, token0=0)
    for i, (lk, lv) in enumerate(rings):
        if lk.shape[2]:
            ops.append_paged(_bthd(lk), _bthd(lv), pool, rtab[i], token0=n0, wrap_tokens=R)
    return pool, otab, rtab, R


def _prepare_decode(c, seed):
    q, ok, ov, lk, lv, vs = _attention_inputs(c, seed)
    return dict(q=q.view(c["batch"], c["hq"], D), seg=_segments_tiled(c, ok, ov, lk, lv, vs))


def _prepare_prefill(c, seed):
    q, ok, ov, lk, lv, vs = _attention_inputs(c, seed)
    n0, n1 = ok.shape[2], lk.shape[2]
    if c["paged"]:
        pool, otab, rtab, R = _fill_pool(c, ok, ov, [(lk, lv)], c["batch"])
        i32 = lambda x: torch.full((c["batch"],), x, dtype=torch.int32, device=DEV)  # noqa: E731
        seg = dict(older=pool, older_table=otab, older_len=i32(n0), vscale=vs, local=pool, local_table=rtab[0],
                   local_ring_blocks=R // 32, local_len=i32(n1), local_start=i32(n0 % R))
        need = ops.prefill_workspace_bytes(c["batch"], c["hkv"], otab.shape[1] * 32, R, query_rows=c["batch"] * c["tokens"],
                                           num_q_heads=c["hq"])
    else:
        seg = _segments_tiled(c, ok, ov, lk, lv, vs)
        need = ops.prefill_workspace_bytes(c["batch"], c["hkv"], n0, n1, n0 % 32, query_rows=c["batch"] * c["tokens"],
                                           num_q_heads=c["hq"])
    return dict(q=q, seg=seg, ws=torch.empty(need, dtype=torch.uint8, device=DEV))


def _prepare_ragged(c, seed):
    rows, n0, local, q, ok, ov, lk, lv, vs = _ragged_inputs(c, seed)
    B = len(rows)
    pool, otab, rtab, R = _fill_pool(c, ok, ov, [(lk, lv)], B)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    cu = np.concatenate([[0], np.cumsum(rows)]).astype(np.int32)
    seg = dict(older=pool, older_table=otab, older_len=i32([n0] * B), vscale=vs, local=pool, local_table=rtab[0],
               local_ring_blocks=R // 32, local_len=i32(local), local_start=i32([n0 % R] * B))
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    need = max(ops.prefill_workspace_bytes(B, c["hkv"], otab.shape[1] * 32, R, query_rows=sum(rows), num_q_heads=c["hq"]),
               ops.ragged_split_state_bytes(B, c["hq"], c["hkv"], max(rows), 0, cus))
    return dict(q=q, seg=seg, cu=i32(cu.tolist()), cu_host=cu, longest=max(rows),
                ws=torch.empty(need, dtype=torch.uint8, device=DEV))


def _prepare_graph(c, seed):
    qkv, ok, ov, rings, vs, qw, kw, cos, sin, n0, n1 = _graph_inputs(c, seed)
    B, hq, hkv, p = c["batch"], c["hq"], c["hkv"], c["position"]
    pool, otab, rtab, R = _fill_pool(c, ok, ov, rings, B)
    i32 = lambda x: torch.full((B,), x, dtype=torch.int32, device=DEV)  # noqa: E731
    pos, len0, len1, start = i32(p), i32(n0), i32(n1), i32(n0 % R)
    widths = [hq * D, hkv * D, hkv * D]
    mul = [(1.0 / vs[i]).contiguous() if c["vllm"] else None for i in range(c["layers"])]
    splits = ops.default_decode_splits(B, hkv, n0 + n1, torch.cuda.get_device_properties(0).multi_processor_count)
    ws = torch.empty(max(16, ops.decode_workspace_bytes(B, hq, splits)), dtype=torch.uint8, device=DEV)
    q_out = torch.empty((B, 1, hq, D), dtype=BF16, device=DEV)
    out = torch.empty((c["layers"], B, hq, D), dtype=BF16, device=DEV)

    def layers():
        for i in range(c["layers"]):
            q, k, v = qkv[i].view(B, 1, -1).split(widths, dim=-1)
            ops.qkv_epilogue(q, k, v, cos, sin, num_q_heads=hq, num_kv_heads=hkv, q_norm_weight=qw, k_norm_weight=kw,
                             eps=EPS, positions=pos, ring=pool, ring_table=rtab[i], ring_tokens=R, q_out=q_out,
                             rounding="vllm" if c["vllm"] else "torch", ring_v_mul=mul[i])
            ops.decode_attention(q_out.view(B, hq, D), older=pool, older_table=otab, older_len=len0,
                                 vscale=None if c["vllm"] else vs[i], local=pool, local_table=rtab[i],
                                 local_ring_blocks=R // 32, local_len=len1, local_start=start, num_splits=splits,
                                 workspace=ws, out=out[i], out_scale=vs[i] if c["vllm"] else None)

    layers()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        layers()
    keep = (qkv, pool, otab, rtab, vs, qw, kw, cos, sin, pos, len0, len1, start, mul, ws, q_out)
    return dict(graph=graph, out=out, keep=keep)


def _prepare_video(c, seed):
    blocks, gates, q, k, v = _video_inputs(c, seed)
    S = c["block"]
    cache = WanKVCache(num_layers=2, num_heads=c["heads"], block_tokens=S, total_tokens=(c["index"] + 1) * S, device=DEV)
    cache.set_alphas(gates)
    for i, kvs in enumerate(blocks):
        cache.commit(i * S, kvs)
    return dict(cache=cache, q=q, k=k, v=v, start=c["index"] * S)


def _prepare_epilogue(c, seed):
    qkv, qw, kw, cos, sin, mul = _epilogue_inputs(c, seed)
    B, L, p, hkv = c["batch"], c["tokens"], c["position"], c["hkv"]
    R = ops.ring_tokens_for_chunk(c["chunk"])
    q, k, v = qkv.split([c["hq"] * D, hkv * D, hkv * D], dim=-1)
    kw_args = dict(num_q_heads=c["hq"], num_kv_heads=hkv, q_norm_weight=qw, k_norm_weight=kw, eps=EPS,
                   rounding="vllm" if c["vllm"] else "torch", ring_v_mul=mul)
    if c["paged"]:
        pages, otab, rtab = _page_tables(B, p + L, 1, R)
        pool = ops.PagedKV.zeros(pages, hkv, DEV)
        kw_args.update(positions=torch.full((B,), p, dtype=torch.int32, device=DEV), ring=pool, ring_table=rtab[0],
                       ring_tokens=R)
        if c["deep"]:
            kw_args.update(deep=pool, deep_table=otab)
        caches = [pool]
    else:
        ring = ops.TiledKV.zeros(B, hkv, R, DEV)
        caches = [ring]
        kw_args.update(positions=p, ring=ring)
        if c["deep"]:
            caches.append(ops.TiledKV.zeros(B, hkv, _blocks(p + L) * 32, DEV))
            kw_args.update(deep=caches[1])
    return dict(args=(q, k, v, cos, sin), kw=kw_args, caches=caches)


def _prepare_commit(c, seed):
    rk, rv, dk, dv, alpha, om, vs, R = _commit_inputs(c, seed)
    return dict(rk=rk, rv=rv, deep=ops.TiledKV(dk, dv),
                kw=dict(batch=c["batch"], chunk_start=c["position"], chunk_len=c["chunk"], alpha=alpha, one_minus_alpha=om,
                        vscale=vs))


def _prepare_glue(c, seed):
    x, res, w, gate_up = _glue_inputs(c, seed)
    return dict(x=x, res=res, w=w, gate=gate_up[:, :c["width"]], up=gate_up[:, c["width"]:])


def _prepare_model(c, seed):
    model, ids = _model(c, seed)
    return dict(model=model, ids=ids)


# ------------------------------------------------------------------------------------------ run
def run(state):
    return globals()["_run_" + state["kind"]](state)


def _run_decode(s):
    return ops.decode_attention(s["q"], **s["seg"])


def _run_prefill(s):
    return ops.prefill_attention(s["q"], causal=True, workspace=s["ws"], **s["seg"])


def _run_ragged(s):
    return ops.prefill_attention(s["q"], causal=True, workspace=s["ws"], cu_seqlens_q=s["cu"], max_seqlen_q=s["longest"],
                                 cu_seqlens_q_host=s["cu_host"], **s["seg"])


def _run_graph(s):
    s["graph"].replay()
    return s["out"]


def _run_video(s):
    return s["cache"].attention(0, s["q"], s["k"], s["v"], s["start"])


def _run_epilogue(s):
    q = ops.qkv_epilogue(*s["args"], **s["kw"])
    return [q] + [t for cache in s["caches"] for t in (cache.k, cache.v)]


def _run_commit(s):
    ops.blend_chunk(s["rk"], s["rv"], s["deep"], **s["kw"])
    return [s["rk"], s["rv"]]


def _run_glue(s):
    h = ops.rmsnorm(s["x"], s["w"], EPS, residual=s["res"])
    return [h, s["res"], ops.silu_mul(s["gate"], s["up"])]


def _run_model(s):
    with torch.no_grad():
        c = s["case"]
        cache = LastKVCache(c["layers"], c["chunk"], capacity_tokens=c["tokens"])
        return s["model"](input_ids=s["ids"], past_key_values=cache, logits_to_keep=64).logits


# ------------------------------------------------------------------------------------------ work
def _attention_work(batch, hq, hkv, rows, n0, n1, causal):
    """(bytes, flops): q and out, each key and value once, 2 products over the visible pairs."""

    seen = n0 + n1 - (rows - 1) / 2 if causal and n1 else n0 + n1
    return 2 * D * (2 * batch * rows * hq + 2 * batch * hkv * (n0 + n1)), 4 * D * batch * hq * rows * seen


def work(c):
    kind = c["kind"]
    if kind in ("decode", "prefill"):
        L = c.get("tokens", 1)
        b, f = _attention_work(c["batch"], c["hq"], c["hkv"], L, *_regions(c, L), True)
    elif kind == "graph":
        b, f = _attention_work(c["batch"], c["hq"], c["hkv"], 1, *_regions(c), True)
        b, f = c["layers"] * (b + 4 * D * c["batch"] * (c["hq"] + 2 * c["hkv"])), c["layers"] * f
    elif kind == "ragged":
        rows, n0, local = _ragged_rows(c)
        parts = [_attention_work(1, c["hq"], c["hkv"], n, n0, m, True) for n, m in zip(rows, local)]
        b, f = sum(p[0] for p in parts), sum(p[1] for p in parts)
    elif kind == "video":
        S, n = c["block"], c["index"] * c["block"]
        b, f = _attention_work(1, c["heads"], c["heads"], S, n, S, False)
        b += 4 * D * c["heads"] * S  # the block's K / V are also written to the ring
    elif kind == "epilogue":
        rows, hq, hkv = c["batch"] * c["tokens"], c["hq"], c["hkv"]
        b = 2 * D * rows * (2 * hq + 4 * hkv + (2 * hkv if c["deep"] else 0) + 2)
        f = 16 * D * rows * (hq + hkv)
    elif kind == "commit":
        ring = 2 * D * c["layers"] * c["batch"] * c["hkv"] * c["chunk"]  # one of K, V
        b, f = 4 * ring + 2 * ring // c["layers"], 4 * ring
    elif kind == "glue":
        b = 2 * c["rows"] * (4 * c["hidden"] + 3 * c["width"]) + 2 * c["hidden"]
        f = c["rows"] * (6 * c["hidden"] + 6 * c["width"])
    else:
        rows, hid = c["batch"] * c["tokens"], c["hidden"]
        layer = hid * D * (2 * c["hq"] + 2 * c["hkv"]) + 3 * hid * c["width"]
        seen = sum(min(i + 1, c["tokens"]) for i in range(c["tokens"]))
        f = 2 * rows * layer * c["layers"] + 2 * c["batch"] * 64 * hid * c["vocab"] \
            + c["layers"] * 4 * D * c["hq"] * c["batch"] * seen
        b = 2 * (layer * c["layers"] + hid * c["vocab"]) + 2 * rows * hid + 2 * c["batch"] * 64 * c["vocab"]
    return {"bytes": int(b), "flops": int(f)}


# ------------------------------------------------------------------------------------------ tolerance
# Two correct implementations of a bf16 result differ by flips of its last bit, 2^-9 relative at most and
# about 1e-3 in 2-norm (attention outputs are at most 1e-3 from 64 bits, a chain of bf16 roundings as in
# RoPE + norm or the blend 2-3e-3); after two whole decoder layers the flips have travelled.
TOLERANCE = {"decode": 4e-3, "graph": 8e-3, "prefill": 4e-3, "ragged": 4e-3, "video": 4e-3, "epilogue": 4e-3,
             "commit": 4e-3, "glue": 4e-3, "model": 2.5e-2}


def tolerance(c):
    return {"rel": TOLERANCE[c["kind"]]}


# ------------------------------------------------------------------------------------------ exact
def exact(case, seed):
    return globals()["_exact_" + case["kind"]](case, seed)


def _softmax_attention(q, k, v, causal_tail=None):
    """q [L, Hq, 128], k / v [H, n, 128] (64 bits) -> [L, Hq, 128]; with causal_tail query i sees all but
    the last causal_tail - 1 - i keys."""

    L, hq = q.shape[:2]
    H, n = k.shape[:2]
    out = torch.empty((L, hq, D), dtype=torch.float64, device=DEV)
    hide = None
    if causal_tail is not None:
        hide = torch.arange(n, device=DEV)[None, :] > (n - causal_tail + torch.arange(L, device=DEV))[:, None]
    for h in range(hq):
        g = h // (hq // H)
        s = (q[:, h] @ k[g].t().contiguous()) / math.sqrt(D)
        if hide is not None:
            s = s.masked_fill(hide, float("-inf"))
        out[:, h] = torch.softmax(s, -1) @ v[g]
    return out


def _keys(ok, ov, lk, lv, vs, b, n1=None):
    """Sequence b's keys and values in 64 bits, older V scaled."""

    n1 = lk.shape[2] if n1 is None else n1
    o = ov[b].double()
    if vs is not None:
        o = o * vs.double()[:, None, None]
    return torch.cat((ok[b].double(), lk[b, :, :n1].double()), 1), torch.cat((o, lv[b, :, :n1].double()), 1)


def _exact_decode(c, seed):
    q, ok, ov, lk, lv, vs = _attention_inputs(c, seed)
    outs = []
    for b in range(c["batch"]):
        k, v = _keys(ok, ov, lk, lv, vs, b)
        qd = q[b, 0].double().view(c["hkv"], -1, D)
        p = torch.softmax(torch.bmm(qd, k.transpose(1, 2).contiguous()) / math.sqrt(D), -1)
        outs.append(torch.bmm(p, v).reshape(c["hq"], D))
    return torch.stack(outs)


def _exact_prefill(c, seed):
    q, ok, ov, lk, lv, vs = _attention_inputs(c, seed)
    return torch.stack([_softmax_attention(q[b].double(), *_keys(ok, ov, lk, lv, vs, b), causal_tail=c["tokens"])
                        for b in range(c["batch"])])


def _exact_ragged(c, seed):
    rows, n0, local, q, ok, ov, lk, lv, vs = _ragged_inputs(c, seed)
    at, outs = 0, []
    for b, n in enumerate(rows):
        outs.append(_softmax_attention(q[at:at + n].double(), *_keys(ok, ov, lk, lv, vs, b, local[b]), causal_tail=n))
        at += n
    return torch.cat(outs)


def _rope_norm(x, w, cos, sin):
    """RoPE, then RMSNorm with weight w, of x [..., heads, 128]; cos / sin [..., 1, 128] (all 64 bits)."""

    half = torch.cat((-x[..., 64:], x[..., :64]), -1)
    r = x * cos + half * sin
    return r * torch.rsqrt(r.square().mean(-1, keepdim=True) + EPS) * w


def _exact_graph(c, seed):
    qkv, ok, ov, rings, vs, qw, kw, cos, sin, n0, n1 = _graph_inputs(c, seed)
    B, hq, hkv = c["batch"], c["hq"], c["hkv"]
    cd, sd = cos.double(), sin.double()
    out = torch.empty((c["layers"], B, hq, D), dtype=torch.float64, device=DEV)
    for i in range(c["layers"]):
        q, k, v = (t.reshape(B, -1, D) for t in qkv[i].double().split([hq * D, hkv * D, hkv * D], dim=-1))
        q, k = _rope_norm(q, qw.double(), cd, sd), _rope_norm(k, kw.double(), cd, sd)
        lk, lv = rings[i]
        for b in range(B):
            s = vs[i].double()[:, None, None]
            # the vLLM contract's rings hold V / s, the output is scaled by s; its new token's V enters as V
            old_v = ov[b].double() * s
            ring_v = lv[b].double() * (s if c["vllm"] else 1.0)
            kk = torch.cat((ok[b].double(), lk[b].double(), k[b][:, None]), 1)
            vv = torch.cat((old_v, ring_v, v[b][:, None]), 1)
            qd = q[b].view(hkv, -1, D)
            p = torch.softmax(torch.bmm(qd, kk.transpose(1, 2).contiguous()) / math.sqrt(D), -1)
            out[i, b] = torch.bmm(p, vv).reshape(hq, D)
    return out


def _exact_video(c, seed):
    blocks, gates, q, k, v = _video_inputs(c, seed)
    S = c["block"]
    alpha = gates.sigmoid().to(BF16).double()[0][None, :, None]
    keys = []
    for x in (0, 1):
        hist = [blocks[0][0][x][0].double()]  # the retained first block: layer 0's own
        hist += [blocks[i][1][x][0].double() for i in range(1, c["index"])]  # the final layer's, shared
        if c["index"] > 1:  # the previous block: blended
            last = c["index"] - 1
            hist[-1] = alpha * blocks[last][1][x][0].double() + (1 - alpha) * blocks[last][0][x][0].double()
        hist.append((k, v)[x][0].double())
        keys.append(torch.cat(hist, 0).transpose(0, 1).contiguous())
    return _softmax_attention(q[0].double(), *keys)[None]


def _k_order():
    """Element (token w, dim d) of a K block by its place in the block, as w * 128 + d."""

    w, d = np.meshgrid(np.arange(32), np.arange(D), indexing="ij")
    place = ((((w >> 2) & 1) * 4 + (d >> 5)) * 16 + (((w >> 3) << 2) | (w & 3))) * 32 + (d & 31)
    order = np.empty(4096, dtype=np.int64)
    order[place.reshape(-1)] = (w * D + d).reshape(-1)
    return torch.from_numpy(order).to(DEV)


def _tiles(x, is_v):
    """[..., T, 128] (T a multiple of 32) -> [..., T / 32, 4096] in the cache's tile order."""

    x = x.reshape(*x.shape[:-2], x.shape[-2] // 32, 32, D)
    if is_v:
        return x.transpose(-1, -2).reshape(*x.shape[:-2], 4096)
    return x.reshape(*x.shape[:-2], 4096)[..., _k_order()]


def _exact_epilogue(c, seed):
    qkv, qw, kw, cos, sin, mul = _epilogue_inputs(c, seed)
    B, L, p, hq, hkv = c["batch"], c["tokens"], c["position"], c["hq"], c["hkv"]
    R = ops.ring_tokens_for_chunk(c["chunk"])
    cd, sd = cos.double()[:, :, None], sin.double()[:, :, None]
    q = torch.empty((B, L, hq, D), dtype=torch.float64, device=DEV)
    k = torch.empty((B, hkv, L, D), dtype=torch.float64, device=DEV)
    v = torch.empty_like(k)
    for b in range(B):
        x, y, z = (t.reshape(L, -1, D) for t in qkv[b].double().split([hq * D, hkv * D, hkv * D], dim=-1))
        q[b] = _rope_norm(x, qw.double(), cd[b], sd[b])
        k[b] = _rope_norm(y, kw.double(), cd[b], sd[b]).transpose(0, 1)
        v[b] = z.transpose(0, 1)
    at = p + torch.arange(L, device=DEV)
    rv = v if mul is None else v * mul.double()[None, :, None, None]
    caches = []
    if c["paged"]:
        pages, otab, rtab = _page_tables(B, p + L, 1, R)
        for x, rx, is_v in ((k, k, False), (v, rv, True)):
            pool = torch.zeros((hkv, pages, 4096), dtype=torch.float64, device=DEV)
            parts = [(rx, R, rtab[0], at % R)]
            if c["deep"]:
                parts.append((x, _blocks(p + L) * 32, otab, at))
            for y, size, table, index in parts:
                logical = torch.zeros((B, hkv, size, D), dtype=torch.float64, device=DEV)
                logical[:, :, index] = y
                pool[:, table.long().reshape(-1)] = _tiles(logical, is_v).transpose(0, 1).reshape(hkv, -1, 4096)
            caches.append(pool)
        return [q] + caches
    for size, index, vx in [(R, at % R, rv)] + ([(_blocks(p + L) * 32, at, v)] if c["deep"] else []):
        for y, is_v in ((k, False), (vx, True)):
            logical = torch.zeros((B, hkv, size, D), dtype=torch.float64, device=DEV)
            logical[:, :, index] = y
            caches.append(_tiles(logical, is_v))
    return [q] + caches


def _exact_commit(c, seed):
    rk, rv, dk, dv, alpha, om, vs, R = _commit_inputs(c, seed)
    L, B, H, C, p = c["layers"], c["batch"], c["hkv"], c["chunk"], c["position"]
    blocks = torch.arange(p // 32, _blocks(p + C), device=DEV)
    ring_blocks = blocks % (R // 32)
    inside = torch.zeros((len(blocks) * 32, D), dtype=torch.bool, device=DEV)
    inside[p % 32:p % 32 + C] = True
    outs = []
    for ring, deep, is_v in ((rk, dk, False), (rv, dv, True)):
        mask = _tiles(inside.double()[None], is_v)[0] > 0
        out = ring.double()
        for l in range(L):
            a, o = (t[l * H:(l + 1) * H].double()[None, :, None, None] for t in (alpha, om))
            s = vs[l * H:(l + 1) * H].double()[None, :, None, None] if is_v and vs is not None else 1.0
            own = out[l][:, :, ring_blocks]
            out[l][:, :, ring_blocks] = torch.where(mask, a * deep[:, :, blocks].double() * s + o * own, own)
        outs.append(out)
    return outs


def _exact_glue(c, seed):
    x, res, w, gate_up = _glue_inputs(c, seed)
    r = x.double() + res.double()
    h = r * torch.rsqrt(r.square().mean(-1, keepdim=True) + EPS) * w.double()
    gate, up = gate_up[:, :c["width"]].double(), gate_up[:, c["width"]:].double()
    return [h, r, F.silu(gate) * up]


def _exact_model(c, seed):
    model, ids = _model(c, seed)
    cfg, B, T, C = model.config, c["batch"], c["tokens"], c["chunk"]
    hq, hkv = c["hq"], c["hkv"]
    wt = {n: p.detach() for n, p in model.named_parameters()}
    norm = lambda x, w: x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()  # noqa: E731
    lin = lambda x, n: x @ wt[n + ".weight"].double().t().contiguous()  # noqa: E731
    inv = model.model.inv_freq.to(DEV).double()
    hidden = wt["model.embed_tokens.weight"][ids].double()
    deep, previous, outs = None, [None] * c["layers"], []
    for start in range(0, T, C):
        x = hidden[:, start:start + C]
        n = x.shape[1]
        f = torch.arange(start, start + n, device=DEV).double()[:, None] * inv
        cos, sin = (torch.cat((t, t), -1)[:, None] for t in (f.cos(), f.sin()))
        current = []
        for l in range(c["layers"]):
            base = "model.layers.%d." % l
            att = base + "self_attn."
            h = norm(x, wt[base + "input_layernorm.weight"])
            q, k, v = (lin(h, att + m).view(B, n, -1, D) for m in ("q_proj", "k_proj", "v_proj"))
            rot = lambda y: y * cos + torch.cat((-y[..., 64:], y[..., :64]), -1) * sin  # noqa: E731
            q, k = rot(q), rot(k)
            if cfg.use_qk_norm:
                q, k = norm(q, wt[att + "q_norm.weight"]), norm(k, wt[att + "k_norm.weight"])
            k, v = k.transpose(1, 2), v.transpose(1, 2)
            current.append((k, v))
            kk, vv = [k], [v]
            if previous[l] is not None:
                kk.insert(0, previous[l][0])
                vv.insert(0, previous[l][1])
                s = wt[att + "deep_v_scale"].double()[None, :, None, None] if cfg.deep_kv_rescale else 1.0
                kk.insert(0, deep[0][:, :, :start - C])
                vv.insert(0, deep[1][:, :, :start - C] * s)
            kk, vv = torch.cat(kk, 2), torch.cat(vv, 2)
            o = torch.stack([_softmax_attention(q[b], kk[b], vv[b], causal_tail=n) for b in range(B)])
            x = x + lin(o.reshape(B, n, hq * D), att + "o_proj")
            h = norm(x, wt[base + "post_attention_layernorm.weight"])
            x = x + lin(F.silu(lin(h, base + "mlp.gate_proj")) * lin(h, base + "mlp.up_proj"), base + "mlp.down_proj")
        outs.append(x)
        last = current[-1]
        deep = last if deep is None else tuple(torch.cat((a, b), 2) for a, b in zip(deep, last))
        for l, (k, v) in enumerate(current):
            att = "model.layers.%d.self_attn." % l
            a = wt[att + "prev_chunk_alphas"].sigmoid().to(BF16).double()[None, :, None, None]
            s = wt[att + "deep_v_scale"].double()[None, :, None, None] if cfg.deep_kv_rescale else 1.0
            previous[l] = (a * last[0] + (1 - a) * k, a * last[1] * s + (1 - a) * v)
    x = norm(torch.cat(outs, 1)[:, -64:], wt["model.norm.weight"])
    return x @ wt["lm_head.weight"].double().t().contiguous()
