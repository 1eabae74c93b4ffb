"""The work that users of shadowkv_amd have it do, as cases that can be timed and compared.

Six kinds, each through public entry points and over the range of sizes that the workloads of
bench.py, the tests and decode_model's model shapes span:

  layer    ShadowAttention.decode: one new token through one layer's sparse attention, eager, with
           the value store in pinned host memory (the default) or in device memory. Successive
           passes take successive queries of a slowly drifting sequence, so that about half of the
           selected chunks are hits, as in a real decode.
  step     whole decode steps captured in a HIP graph, as a serving loop runs them: embedding, per
           layer RMSNorm, QKV projection + RoPE + KV append, sparse attention, output projection,
           residual RMSNorm, SiLU MLP, then the lm head; logits come back.
  attend   a decode layer's second half on a given selection: the missed chunks' keys rebuilt and
           rotated into the buffer, then the sparse attention over buffer and value store.
  mlp      the dense half of a few layers at decode batch sizes: RMSNorm, gate/up projection with
           SiLU-and-mul, down projection, residual.
  prefill  ShadowAttention.prefill: one layer's prompt (low-rank factors, causal attention, the
           decode state).
  encode   the same prompt state without the attention (get_svd + prefill_kv_cache), for callers
           whose model ran its own prefill attention.

A case is a dict of plain values; model names are decode_model's shapes.
"""
import math
import types

import torch
import torch.nn.functional as F

from shadowkv_amd.decode_model import GLM4_9B, LLAMA31_8B, LLAMA3_8B_1M, synthesize_state
from shadowkv_amd.kernels import shadowkv
from shadowkv_amd.models.attention import ShadowAttention
from shadowkv_amd.models.kvcache import ShadowKVCache_CPU
from shadowkv_amd.models.tensor_op import (apply_rotary_pos_emb_cuda, apply_rotary_pos_emb_glm_single,
                                           build_cos_sin_cache, build_glm_cos_sin_cache)
from shadowkv_amd.streams import capture_graph

DEV = "cuda:0"
BF16 = torch.bfloat16
D = 128
RANK = 160
MODELS = {"llama31-8b": LLAMA31_8B, "llama3-8b-1m": LLAMA3_8B_1M, "glm4-9b": GLM4_9B}
QUERIES = 8   # queries of a layer case's drifting sequence
DRIFT = 0.9   # correlation of any two of them


def listed():
    return [
        # The smallest decode call: one sequence, a short prompt (the single-layer workload of the
        # benchmark), values in pinned host memory. Latency and launches.
        dict(name="layer_b1_8k", kind="layer", model="llama31-8b", batch=1, ctx=8192, budget=2048, chunk=8,
             store="host"),
        # A decode lane of the benchmark's default workload (batch 8 runs as two lanes of 4): the host
        # link carries the missed value chunks.
        dict(name="layer_b4_122k_host", kind="layer", model="llama31-8b", batch=4, ctx=122880, budget=2048, chunk=8,
             store="host"),
        # The step of the benchmark's device-store variant, batch 8 at 122880 tokens.
        dict(name="step_b8_122k", kind="step", model="llama31-8b", batch=8, ctx=122880, budget=2048, layers=3,
             steps=2),
        # Batch 16, a shorter and ragged prompt: 9 to 16 token rows in every projection.
        dict(name="step_b16_30k", kind="step", model="llama31-8b", batch=16, ctx=30011, budget=2048, layers=3,
             steps=2),
        # GLM-4-9B's layout: 2 kv heads of 16 query heads, QKV bias, interleaved rotary table.
        dict(name="step_glm_b4_262k", kind="step", model="glm4-9b", batch=4, ctx=262144, budget=2048, layers=3,
             steps=2),
        # One sequence of a million tokens with a budget of 16384.
        dict(name="step_1m_b1", kind="step", model="llama3-8b-1m", batch=1, ctx=1048576, budget=16384, layers=2,
             steps=2),
        # The published 122K setting's batch, on a given selection with 60% hits.
        dict(name="attend_b24_122k", kind="attend", model="llama31-8b", batch=24, ctx=122880, budget=2048, hits=154),
        # The dense half at the smallest batch and at an odd one.
        dict(name="mlp_1", kind="mlp", model="llama31-8b", rows=1, layers=4),
        dict(name="mlp_11", kind="mlp", model="glm4-9b", rows=11, layers=4),
        # Prompts of one sequence through a layer: 8192 tokens, and a longer ragged one on 2 kv heads.
        dict(name="prefill_8k", kind="prefill", model="llama31-8b", batch=1, ctx=8192, budget=2048),
        dict(name="prefill_glm_19k", kind="prefill", model="glm4-9b", batch=1, ctx=19333, budget=2048),
        # The prompt state alone at the benchmark's context.
        dict(name="encode_122k", kind="encode", model="llama31-8b", batch=1, ctx=122880, budget=2048),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "step", "attend", "mlp", "prefill", "encode"])
    model = rng.choice(["llama31-8b", "glm4-9b"])
    if kind == "layer":
        return dict(kind=kind, model="llama31-8b", batch=rng.randint(1, 4), ctx=_log(rng, 6000, 122880),
                    budget=rng.choice([1024, 2048, 4096]), chunk=rng.choice([4, 8, 8, 16]),
                    store=rng.choice(["host", "device"]))
    if kind == "step":
        return dict(kind=kind, model=model, batch=rng.randint(1, 16), ctx=_log(rng, 8192, 60000),
                    budget=rng.choice([1024, 2048, 4096]), layers=2, steps=2)
    if kind == "attend":
        budget = rng.choice([1024, 2048, 4096])
        return dict(kind=kind, model=model, batch=rng.randint(1, 16), ctx=_log(rng, 8192, 122880), budget=budget,
                    hits=rng.randint(0, budget // 8))
    if kind == "mlp":
        return dict(kind=kind, model=model, rows=rng.randint(1, 16), layers=4)
    if kind == "prefill":
        return dict(kind=kind, model=model, batch=rng.choice([1, 1, 2]), ctx=_log(rng, 3000, 12000),
                    budget=rng.choice([1024, 2048]))
    return dict(kind=kind, model=model, batch=1, ctx=_log(rng, 3000, 122880), budget=rng.choice([1024, 2048]))


# ------------------------------------------------------------------------------------ shared parts

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *size, scale=1.0):
    return torch.randn(*size, generator=g, device=DEV).mul_(scale).to(BF16)


def _config(shape, layers):
    return types.SimpleNamespace(num_attention_heads=shape.heads, num_key_value_heads=shape.kv_heads,
                                 hidden_size=shape.heads * D, num_hidden_layers=layers)


def _table(shape, length):
    if shape.rope == "glm":
        return build_glm_cos_sin_cache(length, shape.rope_theta, device=DEV)
    return build_cos_sin_cache(length, shape.rope_theta, D, device=DEV)


def _geometry(case):
    """(landmarks, outlier chunks, first row of the selected region) of a prompt of ctx tokens."""
    c = case.get("chunk", 8)
    chunks = case["ctx"] // c - 4
    chunks -= chunks % 8
    outliers = case["budget"] // 1024 * 24
    return chunks - outliers, outliers, case["ctx"] - chunks * c + outliers * c


def _rotate_bf16(x, table, pos):
    """RoPE in bf16 torch operations, each rounded (half-split for a 128-wide table, else GLM's
    interleaved pairs on the first 64 dims); x [b, h, s, 128], pos [s]."""
    cs = table[pos]
    if table.shape[-1] == D:
        c, s = cs[:, :64], cs[:, 64:]
        a, b = x[..., :64], x[..., 64:]
        return torch.cat((a * c - b * s, b * c + a * s), dim=-1)
    return apply_rotary_pos_emb_glm_single(x, table, pos)


# ------------------------------------------------------------------------------------------- layer

def _prepare_layer(case, seed):
    shape, B, ctx = MODELS[case["model"]], case["batch"], case["ctx"]
    Hq, H = shape.heads, shape.kv_heads
    g = _gen(seed)
    table = _table(shape, ctx + 64)
    cache = ShadowKVCache_CPU(_config(shape, 1), batch_size=B, max_length=ctx, device=DEV,
                              sparse_budget=case["budget"], chunk_size=case["chunk"], rank=RANK, max_decode_len=64,
                              zero_host_store=False, value_store=case["store"])
    synthesize_state(cache, ctx, seed=seed + 1, cos_sin=table)

    def rope(q, k, pos):
        return (apply_rotary_pos_emb_cuda(q, table, pos.expand(B, Hq, 1)),
                apply_rotary_pos_emb_cuda(k, table, pos.expand(B, H, 1)))

    attn = ShadowAttention(cache, Hq // H, D, shape.hidden, rope, None, table)
    base = torch.randn(1, B, Hq, 1, D, generator=g, device=DEV)
    noise = torch.randn(QUERIES, B, Hq, 1, D, generator=g, device=DEV)
    q = (math.sqrt(DRIFT) * base + math.sqrt(1 - DRIFT) * noise).to(BF16)
    return dict(cache=cache, attn=attn, q=q, k=_randn(g, QUERIES, B, H, 1, D), v=_randn(g, QUERIES, B, H, 1, D),
                pos=torch.full((1, 1, 1), ctx, dtype=torch.int64, device=DEV), ctx=ctx, turn=0)


def _run_layer(st):
    i = st["turn"]
    st["turn"] = (i + 1) % QUERIES
    cache = st["cache"]
    cache.gen_offset, cache.kv_offset = 0, st["ctx"]  # every pass decodes the token after the prompt
    out = st["attn"].decode(st["q"][i], st["k"][i], st["v"][i], st["pos"], 0)
    return {"out": out, "scores": cache.chunk_attn}


def _exact_layer(case, seed):
    """The GQA-max landmark probabilities of the first query; the attention output depends on how
    the selection breaks its ties, so it has no 64-bit value."""
    st = _prepare_layer(case, seed)
    cache, shape = st["cache"], MODELS[case["model"]]
    B, H, G = case["batch"], shape.kv_heads, shape.heads // shape.kv_heads
    q = _rotate_bf16(st["q"][0], st["attn"].cos_sin_cache, torch.tensor([case["ctx"]], device=DEV))
    logits = torch.matmul(q.view(B * H, G, D).double(),
                          cache.k_landmark[0].view(B * H, -1, D).double().transpose(1, 2).contiguous()) / math.sqrt(D)
    return {"out": None, "scores": torch.softmax(logits, dim=-1).amax(1).view(B, H, -1)}


# -------------------------------------------------------------------------------------------- step

def _prepare_step(case, seed):
    shape, B, ctx = MODELS[case["model"]], case["batch"], case["ctx"]
    layers, steps = case["layers"], case["steps"]
    g = _gen(seed)
    Hq, H, hid = shape.heads, shape.kv_heads, shape.hidden
    table = _table(shape, ctx + 64)
    cache = ShadowKVCache_CPU(_config(shape, layers), batch_size=B, max_length=ctx, device=DEV,
                              sparse_budget=case["budget"], chunk_size=8, rank=RANK, max_decode_len=64,
                              value_store="device", zero_host_store=False)
    synthesize_state(cache, ctx, seed=seed + 1, cos_sin=table)
    attn = ShadowAttention(cache, Hq // H, D, hid, None, None, table)
    cache.use_device_lengths()
    cache.fold_hit_moves = cache.one_stream_fetch = True
    first_row, first_len = int(cache.append_row_dev), int(cache.kv_len_dev)
    glm, fused_rope = shape.rope == "glm", B <= shadowkv.QKV_ROPE_MAX_ROWS
    ws = []
    for _ in range(layers):
        wqkv = _randn(g, (Hq + 2 * H) * D, hid, scale=0.02)
        bqkv = _randn(g, (Hq + 2 * H) * D, scale=0.1) if shape.qkv_bias else None
        if fused_rope:
            wqkv = shadowkv.qkv_rope_weight(wqkv, Hq, H, glm)
            bqkv = None if bqkv is None else shadowkv.qkv_rope_weight(bqkv, Hq, H, glm)
        ws.append(types.SimpleNamespace(
            wqkv=wqkv, bqkv=bqkv, wo=_randn(g, hid, Hq * D, scale=0.02),
            gate_up=shadowkv.interleave_gate_up(_randn(g, 2 * shape.ffn, hid, scale=0.02)),
            down=_randn(g, hid, shape.ffn, scale=0.02),
            in_norm=1 + _randn(g, hid, scale=0.1), post_norm=1 + _randn(g, hid, scale=0.1)))
    norm, head = 1 + _randn(g, hid, scale=0.1), _randn(g, shape.vocab, hid, scale=0.02)
    embed = _randn(g, shape.vocab, hid)
    tokens = torch.randint(0, shape.vocab, (steps, B), generator=g, device=DEV)
    pos = torch.full((B,), ctx, dtype=torch.int64, device=DEV)
    logits = torch.empty(steps, B, shape.vocab, dtype=BF16, device=DEV)

    def linear(x, w, bias=None):
        y = torch.empty(B, w.shape[0], dtype=BF16, device=DEV)
        shadowkv.linear(x, w, y, bias=bias)
        return y

    def program():
        cache.append_row_dev.fill_(first_row)  # the first tokens after the prompt
        cache.kv_len_dev.fill_(first_len)
        pos.fill_(ctx)
        for t in range(steps):
            h = F.embedding(tokens[t], embed)
            x = torch.empty_like(h)
            shadowkv.rmsnorm(h, ws[0].in_norm, shape.eps, x)
            for i, w in enumerate(ws):
                q_out = torch.empty(B, Hq, D, dtype=BF16, device=DEV)
                if fused_rope:
                    q = cache.qkv_rope_and_append(x, w.wqkv, pos, table, i, q_out, bias_rope=w.bqkv)
                else:
                    q = cache.rope_and_append(linear(x, w.wqkv, w.bqkv), pos, table, i, q_out)
                a = attn.decode_end(attn.decode_begin_appended(q, i))
                o = linear(a.view(B, Hq * D), w.wo)
                h2, x2 = torch.empty_like(h), torch.empty_like(h)
                shadowkv.rmsnorm(o, w.post_norm, shape.eps, x2, residual=h, residual_out=h2)
                act = torch.empty(B, shape.ffn, dtype=BF16, device=DEV)
                shadowkv.linear_gate_up_silu(x2, w.gate_up, act)
                h, x = torch.empty_like(h), torch.empty_like(h)
                shadowkv.rmsnorm(linear(act, w.down), ws[i + 1].in_norm if i + 1 < layers else norm, shape.eps, x,
                                 residual=h2, residual_out=h)
            shadowkv.linear(x, head, logits[t])
            pos.add_(1)

    def rewind():
        cache.gen_offset, cache.kv_offset = 0, ctx

    with torch.inference_mode():
        program()
        torch.cuda.synchronize()
        rewind()
        graph = torch.cuda.CUDAGraph()
        with capture_graph(graph, DEV):
            program()
        rewind()
    return dict(graph=graph, logits=logits, keep=(cache, attn, ws, norm, head, embed, tokens, pos, table))


def _run_step(st):
    st["graph"].replay()
    return st["logits"]


# ------------------------------------------------------------------------------------------ attend

def _prepare_attend(case, seed):
    shape, B, ctx, S = MODELS[case["model"]], case["batch"], case["ctx"], case["budget"] // 8
    Hq, H = shape.heads, shape.kv_heads
    n, outliers, start = _geometry(case)
    g = _gen(seed)
    rows = start + case["budget"] + 40  # 33 generated tokens, the last rows of the tail unused
    ids = torch.rand(B * H, ctx // 8 - 16, generator=g, device=DEV).argsort(dim=-1)[:, :S].view(B, H, S).contiguous()
    return dict(
        u=_randn(g, B, ctx, RANK, scale=1 / math.sqrt(RANK)), sv=_randn(g, B, H, D, RANK), ids=ids,
        cnts=torch.full((B * H,), case["hits"], dtype=torch.int32, device=DEV), table=_table(shape, ctx + 64),
        k=_randn(g, B, H, rows, D), v=_randn(g, B, H, rows, D), store=_randn(g, B, H, ctx // 8, 8 * D),
        q=_randn(g, B, Hq, D, scale=1.5), out=torch.empty(B, Hq, D, dtype=BF16, device=DEV),
        ws=shadowkv.sparse_attn_workspace(B, Hq, rows, DEV), start=start, S=S, length=start + case["budget"] + 33)


def _run_attend(st):
    shadowkv.rebuild_k_rope(st["u"], st["sv"], st["ids"], st["cnts"], st["table"], st["k"], st["start"], 8)
    shadowkv.sparse_attn_decode(st["q"], st["k"], st["v"], st["length"], st["out"], st["ws"],
                                vstore=(st["store"], st["ids"], st["start"], st["S"], 8))
    return {"out": st["out"], "k": st["k"]}


def _exact_attend(case, seed):
    st = _prepare_attend(case, seed)
    B, H, S = st["ids"].shape
    G, start, L = st["q"].shape[1] // H, st["start"], st["length"]
    rows = (st["ids"].unsqueeze(-1) * 8 + torch.arange(8, device=DEV)).view(B, H, S * 8)
    k = st["k"].double()
    out = torch.empty(B, H * G, D, dtype=torch.float64, device=DEV)
    for b in range(B):
        for h in range(H):
            r = rows[b, h]
            x = st["u"][b].index_select(0, r).double() @ st["sv"][b, h].double().t().contiguous()
            cs = st["table"][r].double()
            if cs.shape[-1] == D:
                c, s, a, e = cs[:, :64], cs[:, 64:], x[:, :64], x[:, 64:]
                x = torch.cat((a * c - e * s, e * c + a * s), dim=-1)
            else:
                c, s, a, e = cs[:, :32], cs[:, 32:], x[:, 0:64:2], x[:, 1:64:2]
                x = torch.cat((torch.stack((a * c - e * s, e * c + a * s), -1).flatten(1), x[:, 64:]), dim=-1)
            miss = case["hits"] * 8
            k[b, h, start + miss:start + S * 8] = x[miss:]
            v = st["v"][b, h, :L].double()
            v[start:start + S * 8] = st["store"][b, h].index_select(0, st["ids"][b, h]).view(S * 8, D).double()
            p = torch.softmax(st["q"][b, h * G:(h + 1) * G].double() @ k[b, h, :L].t().contiguous() / math.sqrt(D), -1)
            out[b, h * G:(h + 1) * G] = p @ v
    return {"out": out, "k": k}


# --------------------------------------------------------------------------------------------- mlp

def _prepare_mlp(case, seed):
    shape, M = MODELS[case["model"]], case["rows"]
    g = _gen(seed)
    hid = shape.hidden
    ws = [types.SimpleNamespace(norm=1 + _randn(g, hid, scale=0.1),
                                gate_up=_randn(g, 2 * shape.ffn, hid, scale=0.02),  # rows alternate gate, up
                                down=_randn(g, hid, shape.ffn, scale=0.02)) for _ in range(case["layers"])]
    return dict(ws=ws, x=_randn(g, M, hid), ffn=shape.ffn, eps=shape.eps)


def _run_mlp(st):
    x = st["x"]
    h, n = x, torch.empty_like(x)
    shadowkv.rmsnorm(x, st["ws"][0].norm, st["eps"], n)
    for i, w in enumerate(st["ws"]):
        act = torch.empty(x.shape[0], st["ffn"], dtype=BF16, device=DEV)
        shadowkv.linear_gate_up_silu(n, w.gate_up, act)
        y, h2, n = torch.empty_like(x), torch.empty_like(x), torch.empty_like(x)
        shadowkv.linear(act, w.down, y)
        shadowkv.rmsnorm(y, st["ws"][(i + 1) % len(st["ws"])].norm, st["eps"], n, residual=h, residual_out=h2)
        h = h2
    return h


def _exact_mlp(case, seed):
    st = _prepare_mlp(case, seed)
    h = st["x"].double()
    for w in st["ws"]:
        n = h * torch.rsqrt(h.square().mean(-1, keepdim=True) + st["eps"]) * w.norm.double()
        gu = n @ w.gate_up.double().t().contiguous()
        h = h + (F.silu(gu[:, 0::2]) * gu[:, 1::2]) @ w.down.double().t().contiguous()
    return h


# -------------------------------------------------------------------------------- prefill and encode

def _prepare_prompt(case, seed):
    shape, B, ctx = MODELS[case["model"]], case["batch"], case["ctx"]
    Hq, H = shape.heads, shape.kv_heads
    g = _gen(seed)
    table = _table(shape, ctx + 64)
    cache = ShadowKVCache_CPU(_config(shape, 1), batch_size=B, max_length=ctx, device=DEV,
                              sparse_budget=case["budget"], chunk_size=8, rank=RANK, max_decode_len=64)
    # Pre-RoPE keys of a decaying spectrum (a rank-160 part and noise), values and queries ~ N(0, 1).
    cols = H * D
    spread = torch.logspace(0.5, -0.5, RANK, device=DEV)
    a = torch.randn(B, ctx, RANK, generator=g, device=DEV) * spread
    b = torch.randn(B, RANK, cols, generator=g, device=DEV) / math.sqrt(RANK)
    k = (torch.matmul(a, b) + 0.05 * torch.randn(B, ctx, cols, generator=g, device=DEV)).to(BF16)
    k = k.view(B, ctx, H, D).transpose(1, 2).contiguous()
    v = _randn(g, B, H, ctx, D)
    pos = torch.arange(ctx, device=DEV)

    def rotate(x):
        if shape.rope == "glm":
            return apply_rotary_pos_emb_glm_single(x, table, pos)
        return apply_rotary_pos_emb_cuda(x, table, pos.view(1, 1, -1).expand(x.shape[0], x.shape[1], -1))

    ids = torch.rand(B * H, ctx // 8, generator=g, device=DEV).argsort(dim=-1)[:, :case["budget"] // 8]
    st = dict(cache=cache, table=table, pos=pos, k=k, v=v, ids=ids.to(torch.int32).contiguous(),
              offsets=torch.zeros(B * H * (case["budget"] // 8), dtype=torch.int32, device=DEV),
              keys=torch.empty(B, H, case["budget"], D, dtype=BF16, device=DEV))
    if case["kind"] == "prefill":
        st["q"] = _randn(g, B, Hq, ctx, D)
        st["attn"] = ShadowAttention(cache, Hq // H, D, shape.hidden, lambda q, k, p: (rotate(q), rotate(k)), None, table)
    else:
        st["k_rot"] = rotate(k)
        st["q"] = _randn(g, B, Hq, 1, D)
    return st


def _prompt_state(st):
    """The layer's decode state, and the keys that its factors give back for a random set of chunks
    (U and SV themselves are determined up to the sign of each column)."""
    cache = st["cache"]
    B, H, ctx = cache.batch_size, cache.num_key_value_heads, cache.U.shape[2]
    shadowkv.batch_gather_gemm(cache.U[0], cache.SV[0], None, None, st["ids"], st["keys"], B, H, ctx, D, RANK,
                               cache.sparse_budget, ctx, 8, st["offsets"])
    return {"keys": st["keys"], "landmarks": cache.k_landmark, "landmark_idx": cache.k_landmark_idx,
            "selected": cache.position_ids, "k_buffer": cache.k_cache_buffer, "v_buffer": cache.v_cache_buffer,
            "v_store": cache.v_cache_cpu[0]}


def _run_prefill(st):
    st["cache"].clear()  # a new prompt
    out = st["attn"].prefill(st["q"], st["k"], st["v"], st["pos"], 0)
    return {"out": out, **_prompt_state(st)}


def _run_encode(st):
    cache = st["cache"]
    cache.clear()  # a new prompt
    cache.get_svd(st["k"], 0)
    cache.prefill_kv_cache(st["v"], 0, st["k_rot"], st["q"])
    return _prompt_state(st)


def _exact_prompt(case, seed):
    st = _prepare_prompt(case, seed)
    B, H, ctx, _ = st["k"].shape
    keys = torch.empty(B, H, case["budget"], D, dtype=torch.float64, device=DEV)
    rows = (st["ids"].view(B, H, -1, 1).long() * 8 + torch.arange(8, device=DEV)).view(B, H, -1)
    for b in range(B):
        k = st["k"][b].transpose(0, 1).reshape(ctx, H * D).double()
        v = torch.linalg.eigh(k.t().contiguous() @ k)[1][:, -RANK:]
        low = (k @ v) @ v.t().contiguous()
        for h in range(H):
            keys[b, h] = low[rows[b, h], h * D:(h + 1) * D]
    res = {"keys": keys, "landmarks": None, "landmark_idx": None, "selected": None, "k_buffer": None,
           "v_buffer": None, "v_store": None}
    if case["kind"] == "prefill":
        q, k = (_rotate_bf16(x, st["table"], st["pos"]) for x in (st["q"], st["k"]))
        Hq = q.shape[1]
        out = torch.empty(B, ctx, Hq, D, dtype=torch.float64, device=DEV)
        for b in range(B):
            for hq in range(Hq):
                kh, vh = k[b, hq * H // Hq].double(), st["v"][b, hq * H // Hq].double()
                for s in range(0, ctx, 4096):
                    e = min(ctx, s + 4096)
                    x = q[b, hq, s:e].double() @ kh[:e].t().contiguous() / math.sqrt(D)
                    x.masked_fill_(torch.arange(e, device=DEV)[None] > torch.arange(s, e, device=DEV)[:, None],
                                   float("-inf"))
                    out[b, s:e, hq] = torch.softmax(x, -1) @ vh[:e]
        res["out"] = out
    return res


# ------------------------------------------------------------------------------------- entry points

_KINDS = {"layer": (_prepare_layer, _run_layer, _exact_layer), "step": (_prepare_step, _run_step, None),
          "attend": (_prepare_attend, _run_attend, _exact_attend), "mlp": (_prepare_mlp, _run_mlp, _exact_mlp),
          "prefill": (_prepare_prompt, _run_prefill, _exact_prompt),
          "encode": (_prepare_prompt, _run_encode, _exact_prompt)}


def prepare(case, seed):
    st = _KINDS[case["kind"]][0](case, seed)
    st["run"] = _KINDS[case["kind"]][1]
    return st


def run(state):
    return state["run"](state)


def exact(case, seed):
    f = _KINDS[case["kind"]][2]
    return None if f is None else f(case, seed)


def _sparse_work(case, shape, miss, values=True):
    """Bytes and operations of one layer's rebuild + attention: the missed chunks' U rows read once
    per head, SV, the rebuilt keys written and every live key and value row read once."""
    B, Hq, H, budget = case["batch"], shape.heads, shape.kv_heads, case["budget"]
    _, _, start = _geometry(case)
    L, m = start + budget + 1, B * H * budget * miss
    b = m * RANK * 2 + B * H * D * RANK * 2 + m * D * 2 + 2 * B * H * L * D * 2 + 2 * B * Hq * D * 2
    return b, 2 * m * RANK * D + 4 * B * Hq * L * D


def _score_work(case, shape):
    B, Hq, H = case["batch"], shape.heads, shape.kv_heads
    n = _geometry(case)[0]
    return B * H * n * D * 2 + B * Hq * D * 2 + B * H * n * 2, 2 * B * Hq * n * D


def _dense_work(shape, rows, n, k):
    return 2 * (n * k + rows * (n + k)), 2 * rows * n * k


def work(case):
    shape, kind = MODELS[case["model"]], case["kind"]
    hid, ffn = shape.hidden, shape.ffn
    if kind == "layer":  # about half of the selected chunks are missed
        (b1, f1), (b2, f2) = _sparse_work(case, shape, 0.5), _score_work(case, shape)
        return {"bytes": b1 + b2, "flops": f1 + f2}
    if kind == "attend":
        b, f = _sparse_work(case, shape, 1 - case["hits"] * 8 / case["budget"])
        return {"bytes": b, "flops": f}
    if kind == "mlp":
        b = f = 0
        for n, k in ((2 * ffn, hid), (hid, ffn)):
            x = _dense_work(shape, case["rows"], n, k)
            b, f = b + x[0], f + x[1]
        return {"bytes": b * case["layers"], "flops": f * case["layers"]}
    if kind == "step":
        B = case["batch"]
        n = _geometry(case)[0]
        b = f = 0
        dense = ((shape.heads + 2 * shape.kv_heads) * D, hid), (hid, shape.heads * D), (2 * ffn, hid), (hid, ffn)
        parts = [_sparse_work(case, shape, max(0.0, 1 - case["budget"] / 8 / n)), _score_work(case, shape)]
        parts += [_dense_work(shape, B, *d) for d in dense]
        for x in parts:
            b, f = b + x[0] * case["layers"], f + x[1] * case["layers"]
        x = _dense_work(shape, B, shape.vocab, hid)
        return {"bytes": (b + x[0]) * case["steps"], "flops": (f + x[1]) * case["steps"]}
    # A prompt: keys and values read once, U, SV, landmarks and the host store written; the factors'
    # Gram matrix and projection; for prefill the causal half of the attention.
    B, ctx, H, Hq = case["batch"], case["ctx"], shape.kv_heads, shape.heads
    cols = H * D
    b = B * (2 * ctx * cols * 2 + ctx * RANK * 2 + cols * RANK * 2 + ctx // 8 * cols * 2 + ctx * cols * 2)
    f = B * (ctx * cols * (cols + 1) + 2 * ctx * cols * RANK)
    if kind == "prefill":
        b += 2 * B * ctx * Hq * D * 2
        f += 2 * B * Hq * D * ctx * (ctx + 1)
    return {"bytes": b, "flops": f}


def tolerance(case):
    """bf16 results of fp32 sums. In a layer or step a landmark score one rounding away can change
    which of two almost equal chunks is selected last, and the steps carry one layer's roundings
    through the next."""
    return {"layer": {"rel": 2e-2, "max": 0.9}, "step": {"rel": 2.5e-2, "max": 0.9}, "attend": {"rel": 1e-2, "max": 0.4},
            "mlp": {"rel": 2e-2, "max": 0.4}, "prefill": {"rel": 1e-2, "max": 0.4, "differ": 0.005},
            "encode": {"rel": 1e-2, "max": 0.4, "differ": 0.005}}[case["kind"]]
