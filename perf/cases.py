"""The calls whose speed this framework is measured by.

A serving program spends its time in these: the attention of a decode step
over compact FP8 pages (few and many sequences), the attention of a prefill
batch (long ragged prompts, short ones, a chunk over a retained prefix), a
whole prefill attention layer with the DMS decisions and the pack, the decode
MLPs in bf16 / FP8 / INT4 weights, the FP8 prefill linear into a caller's
buffer, the prefill norm and activation, and the decode forward of a model.
Model widths are those of the presets in fastdms_amd/models/synthetic.py.

Decode calls are captured once in a HIP graph and replayed, as the engine
does; prefill calls are made eagerly, as the engine does.
"""
from __future__ import annotations

import math
from dataclasses import replace

import torch

from fastdms_amd.engine.paged_kv import PAGE_SIZE, PagedCompactKVManager
from fastdms_amd.engine.sequence import Sequence
from fastdms_amd.layers.activation import silu_and_mul
from fastdms_amd.layers.attention import prefill_attention
from fastdms_amd.layers.compact_attention import (DecodePlan, decode_plan_enabled,
                                                  fused_dms_rope_store_compact_decode_attention)
from fastdms_amd.layers.layernorm import rms_norm
from fastdms_amd.layers.linear import (EPI_SILU_MUL, QX_DIVIDE, fp8_gemm, linear_int4_partials, linear_int4_small_m,
                                       linear_partials, linear_small_m)
from fastdms_amd.models.llama import LlamaAttention, LlamaForCausalLM
from fastdms_amd.models.synthetic import dms_decision_rows, model_config
from fastdms_amd.sampling_params import SamplingParams
from fastdms_amd.utils.context import get_context, reset_context, set_context

DEV = "cuda"
WINDOW = 256             # the DMS window, decision scale and offset of the benchmark
ALPHA_SCALE, ALPHA_OFFSET = 10.0, 5.0
EPS = 1e-5
KV_HEADS = 8
BF16, F32, F64, FP8 = torch.bfloat16, torch.float32, torch.float64, torch.float8_e4m3fn

# hidden, ffn of the two presets
WIDTHS = {"llama-3.2-1b": (2048, 8192), "qwen3-8b": (4096, 12288)}


def listed():
    return [
        # one user's decode step: the attention launches of a 16-layer model, ~1 250 live rows per head
        dict(name="decode-attn-1seq", kind="decode_attn", batch=1, prompt=8000, head_dim=64, group=4, layers=16),
        # a loaded server: 128 sequences with prompts of 4-8k tokens (four layers' worth)
        dict(name="decode-attn-128seq", kind="decode_attn", batch=128, prompt=6000, head_dim=64, group=4, layers=4),
        # the benchmark's prefill batch: 8 ragged prompts of 4-8k tokens, head_dim 64
        dict(name="prefill-attn-ragged", kind="prefill_attn", seqs=8, tokens=6144, prefix=0, head_dim=64, group=4),
        # many short prompts in one batch (chat turns)
        dict(name="prefill-attn-short", kind="prefill_attn", seqs=24, tokens=400, prefix=0, head_dim=64, group=4),
        # a chunk of a long prompt over its retained prefix, head_dim 128
        dict(name="prefill-attn-chunk", kind="prefill_attn", seqs=1, tokens=4096, prefix=12300, head_dim=128,
             group=4),
        # a prefill attention layer as the engine runs it: qkv, QK-norm, decisions, RoPE, pack, attention, o
        dict(name="prefill-attn-layer", kind="attn_layer", shape="qwen3-8b", seqs=4, tokens=3000),
        # decode MLPs at 8 sequences: bf16, and the INT4 weights of the 8B shape at 4
        dict(name="decode-mlp-bf16", kind="decode_mlp", shape="llama-3.2-1b", rows=8, weights="bf16", layers=4),
        dict(name="decode-mlp-int4", kind="decode_mlp", shape="qwen3-8b", rows=4, weights="int4", layers=6),
        # an FP8 prefill linear (gate_up of the 1B shape) into the caller's buffer
        dict(name="fp8-linear-prefill", kind="fp8_linear", rows=12000, n=16384, k=2048),
        # a prefill layer's residual norm and MLP activation
        dict(name="prefill-norm-act", kind="norm_act", shape="llama-3.2-1b", rows=16384),
        # the whole decode forward at 8 sequences: logits of a three-layer model of the 8B shape
        dict(name="decode-forward-8b", kind="decode_forward", shape="qwen3-8b", batch=8, prompt=6000, layers=3),
        # and of a four-layer model of the 1B shape at one sequence
        dict(name="decode-forward-1b", kind="decode_forward", shape="llama-3.2-1b", batch=1, prompt=3000, layers=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode_attn", "prefill_attn", "attn_layer", "decode_mlp", "fp8_linear", "norm_act",
                       "decode_forward"])
    if kind == "decode_attn":
        batch, prompt, d = _log(rng, 1, 128), _log(rng, 300, 12000), rng.choice([64, 128])
        rows = batch * KV_HEADS * (WINDOW + prompt // 8)
        layers = max(1, min(16, 600_000_000 // (rows * d * 2)))
        return dict(kind=kind, batch=batch, prompt=prompt, head_dim=d, group=rng.choice([4, 4, 2, 1]), layers=layers)
    if kind == "prefill_attn":
        d, prefix = rng.choice([64, 128]), rng.choice([0, 0, _log(rng, 100, 16000)])
        seqs = 1 if prefix else _log(rng, 1, 32)
        tokens = _log(rng, 20, 8192)
        while 4 * d * 32 * seqs * tokens * (prefix + tokens / 2) > 1.2e12:
            seqs, tokens = max(1, seqs // 2), max(20, tokens * 3 // 4)
        return dict(kind=kind, seqs=seqs, tokens=tokens, prefix=prefix, head_dim=d, group=rng.choice([4, 4, 2, 1]))
    if kind == "attn_layer":
        seqs = _log(rng, 1, 8)
        return dict(kind=kind, shape=rng.choice(sorted(WIDTHS)), seqs=seqs,
                    tokens=_log(rng, 64, min(6000, 14000 // seqs)))
    if kind == "decode_mlp":
        weights = rng.choice(["bf16", "fp8", "int4"])
        shape = "llama-3.2-1b" if weights == "bf16" else rng.choice(sorted(WIDTHS))
        return dict(kind=kind, shape=shape, rows=rng.randint(1, 16), weights=weights,
                    layers=rng.randint(1, 2) if weights == "fp8" else rng.randint(3, 5))
    if kind == "fp8_linear":
        return dict(kind=kind, rows=_log(rng, 17, 12000), n=rng.choice([2048, 3072, 4096, 6144, 16384, _log(rng, 1000, 16000)]),
                    k=rng.choice([2048, 4096, 8192, 16 * _log(rng, 32, 500)]))
    if kind == "norm_act":
        return dict(kind=kind, shape=rng.choice(sorted(WIDTHS)), rows=_log(rng, 20, 10000))
    return dict(kind=kind, shape=rng.choice(sorted(WIDTHS)), batch=rng.randint(1, 16), prompt=_log(rng, 300, 8000),
                layers=rng.randint(2, 3))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 13)


def _randn(gen, shape, std=1.0, dtype=BF16):
    return (torch.randn(shape, generator=gen, device=DEV) * std).to(dtype)


def _prompt_lengths(seqs, mean):
    """Ragged lengths spread between two thirds and four thirds of the mean
    (multiples of the golden ratio's fraction, so every batch size is spread)."""
    return [max(1, int(mean * (2 + 2 * ((0.5 + 0.6180339887 * i) % 1.0)) / 3)) for i in range(seqs)]


def _rope_table(head_dim, positions, theta=500000.0):
    inv = 1.0 / (theta ** (torch.arange(0, head_dim, 2, dtype=F32) / head_dim))
    f = torch.arange(positions, dtype=F32)[:, None] * inv[None, :]
    return torch.cat((f.cos(), f.sin()), dim=-1).unsqueeze(1).to(DEV)


def _pages(gen, layers, batch, prompt, head_dim):
    """Compact FP8 pages of ``layers`` layers as a decode step finds them: per
    (layer, sequence, kv head) the window's tokens plus about an eighth of the
    older ones (heads differ by a factor of two either way), in randomly placed
    16-row pages.  The appended token's row (rank live - 1) is still empty.
    Lengths and live counts go by the sizes alone, page places and contents by
    the seed."""
    lens = torch.tensor(_prompt_lengths(batch, prompt), device=DEV)
    spread = torch.randn((layers, batch, KV_HEADS), generator=_gen(batch * 100003 + prompt), device=DEV)
    frac = 0.125 * torch.exp(0.45 * spread)
    old = (lens - WINDOW).clamp_min(0)[None, :, None]
    live = (lens.clamp_max(WINDOW)[None, :, None] + (old * frac.clamp_max(1.0))).to(torch.int32) + 1
    held = (live + PAGE_SIZE - 1) // PAGE_SIZE
    width = int(held.max()) + 1
    per_layer = int(held.sum(dim=(1, 2)).max())
    tables = torch.full((layers, batch, KV_HEADS, width), -1, device=DEV, dtype=torch.int32)
    for li in range(layers):
        ids = torch.randperm(per_layer, generator=gen, device=DEV).to(torch.int32)
        mask = torch.arange(width, device=DEV)[None, None, :] < held[li][:, :, None]
        tables[li][mask] = ids[: int(mask.sum())]
    rank = (live - 1).long()
    slot = (torch.gather(tables, 3, (rank // PAGE_SIZE)[..., None])[..., 0] * PAGE_SIZE
            + (rank % PAGE_SIZE).to(torch.int32)).to(torch.int32)
    arena = torch.empty((2, layers, per_layer * PAGE_SIZE, head_dim), device=DEV, dtype=FP8)
    for t in range(2):
        for li in range(layers):
            arena[t, li] = torch.randn(arena.shape[2:], generator=gen, device=DEV).to(FP8)
    positions = lens.to(torch.int64)
    return dict(live=live, tables=tables, slot=slot, arena=arena, positions=positions)


def _captured(fn):
    """fn() once, then captured; the graph."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def _live_bound(prompt):
    """The engine's static bound of a span's rows: its model length, in 256s."""
    return (2 * prompt // 256 + 2) * 256


# -- decode attention --------------------------------------------------------
def _decode_attn_inputs(case, seed):
    gen = _gen(seed)
    b, d, layers, hq = case["batch"], case["head_dim"], case["layers"], KV_HEADS * case["group"]
    s = _pages(gen, layers, b, case["prompt"], d)
    s["qkv"] = _randn(gen, (layers, b, (hq + 2 * KV_HEADS) * d))
    s["scales"] = torch.rand((layers, 2, KV_HEADS), generator=gen, device=DEV) * 0.5 + 0.75
    s["rope"] = _rope_table(d, 2 * case["prompt"] + 64)
    return s


def _split_qkv(qkv, hq, d):
    b = qkv.shape[0]
    return (qkv[:, :hq * d].view(b, hq, d), qkv[:, hq * d:(hq + KV_HEADS) * d].view(b, KV_HEADS, d),
            qkv[:, (hq + KV_HEADS) * d:].view(b, KV_HEADS, d))


def _prepare_decode_attn(case, seed):
    s = _decode_attn_inputs(case, seed)
    b, d, layers, hq = case["batch"], case["head_dim"], case["layers"], KV_HEADS * case["group"]
    s["out"] = torch.empty((layers, b, hq, d), device=DEV, dtype=BF16)
    s["evict"] = torch.zeros((layers, b, KV_HEADS), device=DEV, dtype=torch.bool)

    def step():
        for li in range(layers):
            q, k, v = _split_qkv(s["qkv"][li], hq, d)
            fused_dms_rope_store_compact_decode_attention(
                q, k, v, s["rope"], s["arena"][0, li], s["arena"][1, li], s["slot"][li], s["evict"][li],
                s["positions"], None, s["live"][li], num_kv_heads=KV_HEADS, alpha_scale=ALPHA_SCALE,
                alpha_offset=ALPHA_OFFSET, max_live_count=_live_bound(case["prompt"]), out=s["out"][li],
                k_scale=s["scales"][li, 0], v_scale=s["scales"][li, 1], block_tables=s["tables"][li],
                page_size=PAGE_SIZE)

    s["graph"], _ = _captured(step)
    return s


def _run_decode_attn(s):
    s["graph"].replay()
    return s["out"], s["evict"], s["arena"].view(torch.uint8)


def _rope64(x, positions, table):
    """x [T, H, D] rotated in 64 bits."""
    h = x.shape[-1] // 2
    cs = table[positions].to(F64)
    c, sn = cs[..., :h], cs[..., h:]
    x1, x2 = x[..., :h], x[..., h:]
    return torch.cat((x1 * c - x2 * sn, x2 * c + x1 * sn), dim=-1)


def _to_fp8(x):
    return x.to(F32).clamp(-448.0, 448.0).to(FP8)


def _compact_decode64(q, k, v, s, li, table, k_scale, v_scale):
    """One layer's decode attention in 64 bits on raw q, k, v [B, H, D] (fp64):
    decision, RoPE, append, attention; returns (out, evict)."""
    b, hq, d = q.shape
    group = hq // KV_HEADS
    pos = s["positions"]
    dec = q[:, ::group, d - 1]
    evict = dec * ALPHA_SCALE - ALPHA_OFFSET > 0
    q = q.clone()
    q[:, ::group, d - 1] = 0
    q, k = _rope64(q, pos, table), _rope64(k, pos, table)
    live, tables = s["live"][li].long(), s["tables"][li].long()
    n = int(live.max())
    r = torch.arange(n, device=DEV)
    rows = tables[:, :, r // PAGE_SIZE].clamp_min(0) * PAGE_SIZE + r % PAGE_SIZE
    ks = torch.ones(KV_HEADS, device=DEV) if k_scale is None else k_scale
    vs = torch.ones(KV_HEADS, device=DEV) if v_scale is None else v_scale
    ks, vs = ks.to(F64)[:, None], vs.to(F64)[:, None]
    out = torch.empty((b, hq, d), device=DEV, dtype=F64)
    knew, vnew = _to_fp8(k / ks).to(F64), _to_fp8(v / vs).to(F64)
    for i in range(b):
        kk = s["arena"][0, li].view(torch.uint8)[rows[i]].view(FP8).to(F64)  # [H, n, D]
        vv = s["arena"][1, li].view(torch.uint8)[rows[i]].view(FP8).to(F64)
        last = (live[i] - 1)[:, None, None].expand(-1, 1, d)
        kk = kk.scatter(1, last, knew[i][:, None]) * ks[:, None]
        vv = vv.scatter(1, last, vnew[i][:, None]) * vs[:, None]
        sc = torch.matmul(q[i].view(KV_HEADS, group, d), kk.transpose(1, 2).contiguous()) * d ** -0.5
        sc = sc.masked_fill(r[None, None, :] >= live[i][:, None, None], -math.inf)
        out[i] = torch.matmul(torch.softmax(sc, dim=-1), vv).view(hq, d)
    return out, evict


def _exact_decode_attn(case, seed):
    s = _decode_attn_inputs(case, seed)
    d, hq = case["head_dim"], KV_HEADS * case["group"]
    out, ev = [], []
    for li in range(case["layers"]):
        q, k, v = (x.to(F64) for x in _split_qkv(s["qkv"][li], hq, d))
        o, e = _compact_decode64(q, k, v, s, li, s["rope"], s["scales"][li, 0], s["scales"][li, 1])
        out.append(o)
        ev.append(e)
    return torch.stack(out), torch.stack(ev), None


def _mean_live(prompt):
    return min(prompt, WINDOW) + max(0, prompt - WINDOW) * 0.125 * math.exp(0.5 * 0.45 ** 2) + 1


def _work_decode_attn(case):
    hq = KV_HEADS * case["group"]
    pairs, live, d = case["batch"] * KV_HEADS, _mean_live(case["prompt"]), case["head_dim"]
    row = case["batch"] * d * 2 * (2 * hq + 2 * KV_HEADS)
    return dict(bytes=case["layers"] * (pairs * live * (2 * d + 0.25) + row + pairs * 2 * d),
                flops=case["layers"] * 4.0 * case["batch"] * hq * live * d)


# -- prefill attention -------------------------------------------------------
def _prefill_attn_inputs(case, seed):
    gen = _gen(seed)
    hq, d = KV_HEADS * case["group"], case["head_dim"]
    lens = _prompt_lengths(case["seqs"], case["tokens"])
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    s = dict(lens=lens, cu_host=cu, cu=torch.tensor(cu, device=DEV, dtype=torch.int32), cu_k=None, group=case["group"])
    qkv = _randn(gen, (cu[-1], (hq + 2 * KV_HEADS) * d))
    q, k, v = _split_qkv(qkv, hq, d)
    if case["prefix"]:  # a dense stage of earlier tokens plus this chunk's
        total = case["prefix"] + cu[-1]
        k, v = (_randn(gen, (total, KV_HEADS, d)) for _ in range(2))
        s["cu_k"] = torch.tensor([0, total], device=DEV, dtype=torch.int32)
    s.update(q=q, k=k, v=v)
    return s


def _run_prefill_attn(s):
    return prefill_attention(s["q"], s["k"], s["v"], s["cu"], max(s["lens"]), s["q"].shape[2] ** -0.5,
                             cu_seqlens_k=s["cu_k"])


def _causal64(q, k, v, group):
    """q [n, Hq, D], k / v [m, Hkv, D] in 64 bits, queries the last of the keys."""
    n, hq, d = q.shape
    m = k.shape[0]
    out = torch.empty((n, hq, d), device=DEV, dtype=F64)
    key = torch.arange(m, device=DEV)
    for h in range(hq):
        kt, vv = k[:, h // group].to(F64).t().contiguous(), v[:, h // group].to(F64)
        for a in range(0, n, 2048):
            e = min(n, a + 2048)
            sc = (q[a:e, h].to(F64) @ kt) * d ** -0.5
            lim = torch.arange(a, e, device=DEV) + (m - n)
            sc.masked_fill_(key[None, :] > lim[:, None], -math.inf)
            out[a:e, h] = torch.softmax(sc, dim=-1) @ vv
    return out


def _exact_prefill_attn(case, seed):
    s = _prefill_attn_inputs(case, seed)
    if s["cu_k"] is not None:
        return _causal64(s["q"], s["k"], s["v"], s["group"])
    cu = s["cu_host"]
    return torch.cat([_causal64(s["q"][cu[i]:cu[i + 1]], s["k"][cu[i]:cu[i + 1]], s["v"][cu[i]:cu[i + 1]], s["group"])
                      for i in range(len(cu) - 1)])


def _work_prefill_attn(case):
    hq, d, n = KV_HEADS * case["group"], case["head_dim"], case["tokens"]
    # mean of n^2 over lengths uniform in [2n/3, 4n/3]
    pairs = case["seqs"] * (n * case["prefix"] + 0.5 * n * n * 28 / 27)
    return dict(flops=4.0 * hq * d * pairs,
                bytes=2.0 * d * case["seqs"] * (2 * hq * n + 2 * KV_HEADS * (n + case["prefix"])))


# -- a prefill attention layer ------------------------------------------------
def _layer_config(shape, layers, positions):
    return replace(model_config(shape), num_hidden_layers=layers, max_position_embeddings=positions,
                   rope_scaling=None, attention_bias=True, rms_norm_eps=EPS)


def _draw_parameters(module, config, gen):
    """Weights N(0, 0.02), norm weights near 1, the DMS decision rows as the
    synthetic presets draw them (about 1/8 of the older tokens survive)."""
    rows = dms_decision_rows(config)
    for name, p in sorted(module.named_parameters(), key=lambda kv: kv[0]):
        if name.endswith("norm.weight"):
            p.data = (1.0 + 0.1 * torch.randn(p.shape, generator=gen, device=DEV)).to(BF16)
        elif name.endswith("bias"):
            b = torch.zeros(p.shape, device=DEV)
            b[rows] = 1.65
            p.data = b.to(BF16)
        else:
            p.data = _randn(gen, p.shape, 0.02)
            if name.endswith("qkv_proj.weight"):
                p.data[rows] = _randn(gen, (len(rows), p.shape[1]), p.shape[1] ** -0.5)


def _attn_layer_inputs(case, seed):
    gen = _gen(seed)
    lens = _prompt_lengths(case["seqs"], case["tokens"])
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    config = _layer_config(case["shape"], 1, 16384)
    attn = LlamaAttention(config)
    _draw_parameters(attn, config, gen)
    table = _rope_table(config.head_dim, max(lens))
    attn.rotary_emb.cos_sin_cache = table
    return dict(config=config, attn=attn, lens=lens, cu_host=cu, table=table,
                cu=torch.tensor(cu, device=DEV, dtype=torch.int32),
                positions=torch.cat([torch.arange(n, device=DEV) for n in lens]),
                hidden=_randn(gen, (cu[-1], config.hidden_size)))


def _prepare_attn_layer(case, seed):
    s = _attn_layer_inputs(case, seed)
    c, lens = s["config"], s["lens"]
    s["attn"].attn.layer_id = 0
    s["manager"] = PagedCompactKVManager(
        num_layers=1, num_kv_heads=KV_HEADS, capacity_tokens=KV_HEADS * (s["cu_host"][-1] + 64 * len(lens)),
        max_model_len=max(lens) + 32, device=DEV, head_dim=c.head_dim, compact_dtype=FP8, max_active_seqs=len(lens))
    s["manager"].attach_attention_modules([s["attn"].attn])
    s["requests"] = [Sequence([0] * n, SamplingParams(max_tokens=16)) for n in lens]
    return s


@torch.inference_mode()
def _run_attn_layer(s):
    m, requests = s["manager"], s["requests"]
    for r in requests:  # the last pass's prompts give their pages back, this pass's come in
        m.free(r.seq_id)
    for r in requests:
        m.allocate(r)
    m.begin_prefill()
    longest = max(s["lens"])
    set_context(True, s["cu"], s["cu"], longest, longest, dms_capture_enabled=True, dms_alpha_scale=ALPHA_SCALE,
                dms_alpha_offset=ALPHA_OFFSET, dms_layer_evictions={}, streaming_pack_manager=m,
                streaming_pack_seq_ids=[r.seq_id for r in requests], streaming_pack_window_size=WINDOW,
                cu_seqlens_q_host=s["cu_host"])
    try:
        out = s["attn"](s["positions"], s["hidden"])
        evict = get_context().dms_layer_evictions[0]
    finally:
        reset_context()
    return out, evict, m.layer_major_live_counts, m.layer_major_token_positions, m.layer_major_evict_mask


def _norm64(x, w):
    return x * torch.rsqrt(x.pow(2).mean(dim=-1, keepdim=True) + EPS) * w.to(F64)


def _exact_attn_layer(case, seed):
    s = _attn_layer_inputs(case, seed)
    a, c, cu = s["attn"], s["config"], s["cu_host"]
    d, hq = c.head_dim, c.num_attention_heads
    group = hq // KV_HEADS
    qkv = s["hidden"].to(F64) @ a.qkv_proj.weight.to(F64).t() + a.qkv_proj.bias.to(F64)
    q, k, v = _split_qkv(qkv, hq, d)
    if c.qk_norm:
        q, k = _norm64(q, a.q_norm.weight), _norm64(k, a.k_norm.weight)
    q = q.clone()
    evict = q[:, ::group, d - 1] * ALPHA_SCALE - ALPHA_OFFSET > 0
    q[:, ::group, d - 1] = 0
    q, k = _rope64(q, s["positions"], s["table"]), _rope64(k, s["positions"], s["table"])
    o = torch.cat([_causal64(q[cu[i]:cu[i + 1]], k[cu[i]:cu[i + 1]], v[cu[i]:cu[i + 1]], group)
                   for i in range(len(cu) - 1)])
    return o.reshape(o.shape[0], hq * d) @ a.o_proj.weight.to(F64).t(), evict, None, None, None


def _work_attn_layer(case):
    hidden = WIDTHS[case["shape"]][0]
    d = 64 if hidden == 2048 else 128
    t, qkv = case["seqs"] * case["tokens"], (32 + 2 * KV_HEADS) * d
    att = _work_prefill_attn(dict(seqs=case["seqs"], tokens=case["tokens"], prefix=0, head_dim=d, group=4))
    live = case["seqs"] * KV_HEADS * _mean_live(case["tokens"])
    return dict(flops=att["flops"] + 2.0 * t * hidden * (qkv + 32 * d),
                bytes=2.0 * hidden * (qkv + 32 * d) + 4.0 * t * hidden + t * KV_HEADS + live * (2 * d + 5))


# -- decode MLPs ---------------------------------------------------------------
def _decode_mlp_inputs(case, seed):
    gen = _gen(seed)
    hidden, ffn = WIDTHS[case["shape"]]
    rows, kind = case["rows"], case["weights"]
    s = dict(kind=kind, x=_randn(gen, (rows, hidden)), res=_randn(gen, (rows, hidden)), layers=[],
             norm=(1.0 + 0.1 * torch.randn(hidden, generator=gen, device=DEV)).to(BF16))
    for _ in range(case["layers"]):
        layer = dict(norm=(1.0 + 0.1 * torch.randn(hidden, generator=gen, device=DEV)).to(BF16))
        for name, n, k in (("gate_up", 2 * ffn, hidden), ("down", hidden, ffn)):
            if kind == "bf16":
                layer[name] = (_randn(gen, (n, k), 0.02),)
            elif kind == "fp8":  # e4m3 rows and their inverse scales
                w = torch.randn((n, k), generator=gen, device=DEV).mul_(100.0).clamp_(-448, 448).to(FP8)
                layer[name] = (w, 0.0002 * (0.5 + torch.rand(n, generator=gen, device=DEV)))
            else:  # two codes a byte, bf16 (scale, zero) per 128-column group
                w = torch.randint(0, 256, (n, k // 2), generator=gen, device=DEV, dtype=torch.uint8)
                sz = torch.zeros((k // 128, n, 2), device=DEV, dtype=BF16)
                sz[..., 0] = (0.004 * (0.5 + torch.rand(sz.shape[:2], generator=gen, device=DEV))).to(BF16)
                layer[name] = (w, sz)
        s["layers"].append(layer)
    return s


def _prepare_decode_mlp(case, seed):
    s = _decode_mlp_inputs(case, seed)
    hidden, ffn = WIDTHS[case["shape"]]
    rows = case["rows"]

    def step():
        x, res = s["x"], s["res"]
        for layer in s["layers"]:
            gu, down = layer["gate_up"], layer["down"]
            if s["kind"] == "fp8":  # the norm hands over e4m3 codes, gate_up its strips' maxima
                am = torch.empty((rows, 1), device=DEV, dtype=F32)
                codes = torch.empty((rows, hidden), device=DEV, dtype=FP8)
                strips = torch.empty((rows, ffn // 16), device=DEV, dtype=F32)
                _, res = rms_norm(x, layer["norm"], EPS, res, amax_out=am, q_out=codes, q_mode=QX_DIVIDE,
                                  bf16_out=False)
                act = linear_small_m(codes, gu[0], weight_scale_inv=gu[1], quantize_x=QX_DIVIDE,
                                     epilogue=EPI_SILU_MUL, x_amax=am, amax_out=strips)
                x = linear_partials(act, down[0], weight_scale_inv=down[1], quantize_x=QX_DIVIDE, x_amax=strips)
                continue
            h, res = rms_norm(x, layer["norm"], EPS, res)
            if s["kind"] == "bf16":
                x = linear_partials(linear_small_m(h, gu[0], epilogue=EPI_SILU_MUL), down[0])
            else:
                act = linear_int4_small_m(h, gu[0], gu[1], 128, epilogue=EPI_SILU_MUL)
                x = linear_int4_partials(act, down[0], down[1], 128)
        return rms_norm(x, s["norm"], EPS, res)

    s["graph"], s["out"] = _captured(step)
    return s


def _run_graph(s):
    s["graph"].replay()
    return s["out"]


def _quantised64(x):
    """x as the e4m3 codes times their inverse scale that a row-quantised FP8 linear multiplies."""
    scale = 448.0 / x.abs().amax(dim=1, keepdim=True)
    return _to_fp8(x * scale).to(F64) / scale


def _weight64(kind, w):
    if kind == "bf16":
        return w[0].to(F64)
    if kind == "fp8":
        return w[0].to(F64) * w[1].to(F64)[:, None]
    codes = torch.stack((w[0] & 15, w[0] >> 4), dim=-1).view(w[0].shape[0], -1).to(F64) - 8.0
    sz = w[1].to(F64).permute(1, 0, 2).repeat_interleave(128, dim=1)
    return codes * sz[..., 0] + sz[..., 1]


def _exact_decode_mlp(case, seed):
    s = _decode_mlp_inputs(case, seed)
    x, res = s["x"].to(F64), s["res"].to(F64)
    q = _quantised64 if s["kind"] == "fp8" else (lambda t: t)
    for layer in s["layers"]:
        res = x + res
        g, u = (q(_norm64(res, layer["norm"])) @ _weight64(s["kind"], layer["gate_up"]).t()).chunk(2, dim=1)
        x = q(torch.nn.functional.silu(g) * u) @ _weight64(s["kind"], layer["down"]).t()
    res = x + res
    return _norm64(res, s["norm"]), res


def _work_decode_mlp(case):
    hidden, ffn = WIDTHS[case["shape"]]
    weights = 3.0 * hidden * ffn * case["layers"]
    per = {"bf16": 2.0, "fp8": 1.0, "int4": 0.5 + 4.0 / 128}[case["weights"]]
    return dict(bytes=weights * per + 8.0 * case["rows"] * hidden, flops=2.0 * case["rows"] * weights)


# -- FP8 prefill linear ----------------------------------------------------------
def _fp8_linear_inputs(case, seed):
    gen = _gen(seed)
    return dict(x=_randn(gen, (case["rows"], case["k"])),
                w=torch.randn((case["n"], case["k"]), generator=gen, device=DEV).mul_(100.0).clamp_(-448, 448).to(FP8),
                sinv=0.0002 * (0.5 + torch.rand(case["n"], generator=gen, device=DEV)))


def _prepare_fp8_linear(case, seed):
    s = _fp8_linear_inputs(case, seed)
    s["out"] = torch.empty((case["rows"], case["n"]), device=DEV, dtype=BF16)
    return s


def _run_fp8_linear(s):
    return fp8_gemm(s["x"], s["w"], s["sinv"], out=s["out"])


def _exact_fp8_linear(case, seed):
    s = _fp8_linear_inputs(case, seed)
    x = s["x"].to(F32)
    scale = x.abs().amax(dim=1, keepdim=True).reciprocal() * 448.0
    xq = _to_fp8(x * scale).to(F64) * scale.reciprocal().to(F64)
    return (xq @ s["w"].to(F64).t()) * s["sinv"].to(F64)[None, :]


def _work_fp8_linear(case):
    m, n, k = case["rows"], case["n"], case["k"]
    return dict(flops=2.0 * m * n * k, bytes=2.0 * m * k + 1.0 * n * k + 4.0 * n + 2.0 * m * n)


# -- prefill norm and activation ---------------------------------------------------
def _prepare_norm_act(case, seed):
    gen = _gen(seed)
    hidden, ffn = WIDTHS[case["shape"]]
    return dict(x=_randn(gen, (case["rows"], hidden)), res=_randn(gen, (case["rows"], hidden)),
                w=(1.0 + 0.1 * torch.randn(hidden, generator=gen, device=DEV)).to(BF16),
                gate_up=_randn(gen, (case["rows"], 2 * ffn)))


def _run_norm_act(s):
    h, res = rms_norm(s["x"], s["w"], EPS, s["res"])
    return h, res, silu_and_mul(s["gate_up"])


def _exact_norm_act(case, seed):
    s = _prepare_norm_act(case, seed)
    res = s["x"].to(F64) + s["res"].to(F64)
    g, u = s["gate_up"].to(F64).chunk(2, dim=1)
    return _norm64(res, s["w"]), res, torch.nn.functional.silu(g) * u


def _work_norm_act(case):
    hidden, ffn = WIDTHS[case["shape"]]
    return dict(bytes=case["rows"] * (8.0 * hidden + 6.0 * ffn), flops=case["rows"] * (4.0 * hidden + 4.0 * ffn))


# -- the decode forward of a model ----------------------------------------------------
def _decode_forward_inputs(case, seed):
    gen = _gen(seed)
    config = _layer_config(case["shape"], case["layers"], 16384)
    model = LlamaForCausalLM(config)
    _draw_parameters(model, config, gen)
    if config.tie_word_embeddings:
        model.lm_head.weight = model.model.embed_tokens.weight
    model.eval()
    table = _rope_table(config.head_dim, 2 * case["prompt"] + 64)
    for layer in model.model.layers:
        layer.self_attn.rotary_emb.cos_sin_cache = table
    s = _pages(gen, case["layers"], case["batch"], case["prompt"], config.head_dim)
    s["ids"] = torch.randint(0, config.vocab_size, (case["batch"],), generator=gen, device=DEV)
    s.update(model=model, config=config, table=table)
    return s


def _prepare_decode_forward(case, seed):
    s = _decode_forward_inputs(case, seed)
    layers, b, c = case["layers"], case["batch"], s["config"]
    s["evict"] = torch.zeros((layers, b, KV_HEADS), device=DEV, dtype=torch.bool)
    for li, layer in enumerate(s["model"].model.layers):
        layer.self_attn.attn.layer_id = li
        layer.self_attn.attn.compact_k_cache, layer.self_attn.attn.compact_v_cache = s["arena"][0, li], s["arena"][1, li]
    bound = _live_bound(case["prompt"])
    plan = None
    tables = s["tables"]
    if decode_plan_enabled(c.head_dim):
        # the manager that assigns the step's append rows writes the step's work plan
        m = PagedCompactKVManager(num_layers=layers, num_kv_heads=KV_HEADS, capacity_tokens=s["arena"].shape[2],
                                  max_model_len=bound, device=DEV, head_dim=c.head_dim, compact_dtype=FP8,
                                  max_active_seqs=b)
        m.block_tables[..., :tables.shape[3]].copy_(tables)
        m.pages_held.copy_((s["live"] + PAGE_SIZE - 1) // PAGE_SIZE)
        m.layer_major_live_counts.copy_(s["live"] - 1)  # the step's own append makes it s["live"]
        plan = DecodePlan(DEV, layers, b * KV_HEADS, bound + 1, c.head_dim)
        tables, _ = m.paged_prepare_decode(0, b, torch.empty_like(s["slot"]), plan=plan, positions=s["positions"])
        s["manager"], s["plan"] = m, plan

    @torch.inference_mode()
    def step():
        set_context(False, block_tables=tables, compact_kv_enabled=True, compact_live_counts=s["live"],
                    compact_slot_mapping=s["slot"], compact_max_live_count=bound, dms_capture_enabled=True,
                    dms_alpha_scale=ALPHA_SCALE, dms_alpha_offset=ALPHA_OFFSET, dms_layer_evictions_buffer=s["evict"],
                    compact_plan=plan)
        try:
            return s["model"].forward_decode_fused(s["ids"], s["positions"])
        finally:
            reset_context()

    s["graph"], s["logits"] = _captured(step)
    return s


def _run_decode_forward(s):
    s["graph"].replay()
    return s["logits"], s["evict"]


def _exact_decode_forward(case, seed):
    s = _decode_forward_inputs(case, seed)
    c, model = s["config"], s["model"].model
    d, hq = c.head_dim, c.num_attention_heads
    res, x, ev = None, model.embed_tokens.weight[s["ids"]].to(F64), []
    for li, layer in enumerate(model.layers):
        a, mlp = layer.self_attn, layer.mlp
        res = x if res is None else x + res
        h = _norm64(res, layer.input_layernorm.weight)
        q, k, v = _split_qkv(h @ a.qkv_proj.weight.to(F64).t() + a.qkv_proj.bias.to(F64), hq, d)
        if c.qk_norm:
            q, k = _norm64(q, a.q_norm.weight), _norm64(k, a.k_norm.weight)
        o, e = _compact_decode64(q, k, v, s, li, s["table"], None, None)
        ev.append(e)
        res = res + o.reshape(o.shape[0], -1) @ a.o_proj.weight.to(F64).t()
        h = _norm64(res, layer.post_attention_layernorm.weight)
        g, u = (h @ mlp.gate_up_proj.weight.to(F64).t()).chunk(2, dim=1)
        x = (torch.nn.functional.silu(g) * u) @ mlp.down_proj.weight.to(F64).t()
    h = _norm64(x + res, model.norm.weight)
    head = s["model"].lm_head.weight
    return torch.cat([h @ head[i:i + 16384].to(F64).t() for i in range(0, head.shape[0], 16384)], dim=1), torch.stack(ev)


def _work_decode_forward(case):
    hidden, ffn = WIDTHS[case["shape"]]
    d, vocab = (64, 128256) if hidden == 2048 else (128, 151936)
    weights = case["layers"] * hidden * ((64 + 2 * KV_HEADS) * d + 3.0 * ffn) + vocab * hidden
    att = _work_decode_attn(dict(batch=case["batch"], prompt=case["prompt"], head_dim=d, group=4,
                                 layers=case["layers"]))
    return dict(bytes=2.0 * weights + att["bytes"] + 2.0 * case["batch"] * vocab,
                flops=2.0 * case["batch"] * weights + att["flops"])


# ---------------------------------------------------------------------------
_KINDS = {
    "decode_attn": (_prepare_decode_attn, _run_decode_attn, _exact_decode_attn, _work_decode_attn),
    "prefill_attn": (_prefill_attn_inputs, _run_prefill_attn, _exact_prefill_attn, _work_prefill_attn),
    "attn_layer": (_prepare_attn_layer, _run_attn_layer, _exact_attn_layer, _work_attn_layer),
    "decode_mlp": (_prepare_decode_mlp, _run_graph, _exact_decode_mlp, _work_decode_mlp),
    "fp8_linear": (_prepare_fp8_linear, _run_fp8_linear, _exact_fp8_linear, _work_fp8_linear),
    "norm_act": (_prepare_norm_act, _run_norm_act, _exact_norm_act, _work_norm_act),
    "decode_forward": (_prepare_decode_forward, _run_decode_forward, _exact_decode_forward, _work_decode_forward),
}


def prepare(case, seed):
    s = _KINDS[case["kind"]][0](case, seed)
    s["case_kind"] = case["kind"]
    return s


def run(state):
    return _KINDS[state["case_kind"]][1](state)


@torch.no_grad()
def exact(case, seed):
    return _KINDS[case["kind"]][2](case, seed)


def work(case):
    return _KINDS[case["kind"]][3](case)


def tolerance(case):
    kind = case["kind"]
    # bf16 results of 32-bit sums; whole values: decisions, appended / packed e4m3 bytes on a rounding boundary
    if kind in ("decode_attn", "prefill_attn"):
        return {"rel": 0.01, "max": 0.25, "differ": 0.001}
    if kind == "attn_layer":  # the projections and the attention round in turn
        return {"rel": 0.016, "max": 0.25, "differ": 0.002}
    if kind == "decode_mlp":  # activations that cross an e4m3 step move by a sixteenth
        return {"rel": 0.03, "max": 0.5} if case["weights"] == "fp8" else {"rel": 0.02, "max": 0.2}
    if kind == "decode_forward":
        return {"rel": 0.03, "max": 0.5, "differ": 0.01}
    return {"rel": 0.008, "max": 0.05}
