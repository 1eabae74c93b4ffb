"""ShadowKV attention handler (reference: models/attention/shadow.py:6-50).

decode() keeps the reference's order of operations: RoPE -> append the new token -> select chunks
(score, top-k, reorder) -> value fetch from host beside the low-rank key rebuild + RoPE -> sparse
attention. A cache in its default setting takes the fetch and the rebuild as one launch on the current
stream, after a selection that moves the cached chunks itself; otherwise, and in decode_begin() /
decode_end(), they are the reference's two streams: [copy stream: value fetch] || [current stream: key
compaction + rebuild] -> join. The attention is the gfx950 split-L decode kernel in place of
flash_attn_with_kvcache; prefill attention is the gfx950 prompt attention kernel (fp32 torch operations
where that kernel does not apply).
"""
import math

import torch

from ...kernels import shadowkv
from ..kvcache.shadow import ShadowKVCache_CPU
from ..tensor_op import plain_eager, repeat_kv
from .base import AttentionBase


def _kernel_takes(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> bool:
    """Whether the prompt attention kernel serves this call: bf16 tensors of 128-dim heads and one
    length, outside autograd and tracing."""
    if not (plain_eager(q, k, v) and all(t.dtype == torch.bfloat16 and t.dim() == 4 for t in (q, k, v))):
        return False
    B, Hq, L, D = q.shape
    H = k.shape[1]
    return (D == 128 and k.shape == (B, H, L, D) and v.shape == k.shape and q.numel() > 0 and H > 0 and Hq % H == 0
            and B * Hq * L < 2 ** 31 and B * H <= 65535)


def causal_attention_fp32(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, block: int = 1024) -> torch.Tensor:
    """Causal GQA attention in fp32; q [B, Hq, L, D], k/v [B, Hkv, L, D] -> [B, L, Hq, D]. bf16 device
    prompts of 128-dim heads outside autograd and tracing run on the prompt attention kernel
    (shadowkv.prefill_attn; MI355X, 32 heads over 8 x 8192 tokens: 0.93 ms against 11.5 ms of the
    torch operations); everything else as query-blocked torch operations."""
    if _kernel_takes(q, k, v):
        with torch.cuda.device(q.device):
            return shadowkv.prefill_attn(q, k, v)
    B, Hq, L, D = q.shape
    k = repeat_kv(k, Hq // k.shape[1]).float()
    v = repeat_kv(v, Hq // v.shape[1]).float()
    kt = k.transpose(-1, -2).contiguous()
    out = torch.empty(B, L, Hq, D, dtype=q.dtype, device=q.device)
    for s in range(0, L, block):
        e = min(L, s + block)
        scores = torch.matmul(q[:, :, s:e].float(), kt[..., :e]) / math.sqrt(D)
        mask = torch.arange(e, device=q.device)[None, :] > torch.arange(s, e, device=q.device)[:, None]
        scores.masked_fill_(mask, float("-inf"))
        p = torch.softmax(scores, dim=-1)
        out[:, s:e] = torch.matmul(p, v[:, :, :e]).transpose(1, 2).to(q.dtype)
    return out


def _unreplaced(obj, steps: dict) -> bool:
    """Whether obj's methods named in steps are the functions that steps holds: not another class's, not a
    subclass's and not the instance's own."""
    cls = type(obj)
    for name, function in steps.items():
        if getattr(cls, name, None) is not function or name in obj.__dict__:
            return False
    return True


# Selected tokens (sparse_budget) up to which the joined chain is taken, by value store: its selection moves both
# buffers' hits before the fetch can start, a row's with one workgroup, where the two-stream chain moves the
# keys' beside a host store's fetch, and its moves keep four loads in flight a thread against the compaction
# kernel's eight (MI355X, us per call, two-stream /
# joined, batch 1, 2, 4 of 120000 tokens and 8 kv heads; host, 8192 selected: 254 / 250, 393 / 384, 660 / 655; 16384:
# 375 / 402, 599 / 630, 1051 / 1112; device, 16384: 173 / 142, 173 / 168, 217 / 222, gathered from 213 / 212; 32768:
# 189 / 210, 231 / 258, 370 / 402).
JOINED_MAX_BUDGET = {"host": 8192, "device": 16384}


# What prefill() runs in two halves where nobody has replaced it.
_PREFILL_STEPS = {"prefill_kv_cache": ShadowKVCache_CPU.prefill_kv_cache}
# The steps of decode_begin() that the joined chain of decode() does otherwise, and those that it takes in
# their place.
_CACHE_STEPS = {n: getattr(ShadowKVCache_CPU, n) for n in (
    "get_retrieval_position_ids", "get_value_cache", "get_key_cache", "move_value_hits", "one_stream_active",
    "fetch_and_rebuild")}


class ShadowAttention(AttentionBase):

    def prefill(self, query_states, key_states, value_states, position_ids, layer_idx):
        kv_cache = self.kv_cache
        kv_cache.get_svd(key_states, layer_idx=layer_idx)
        query_states, key_states = self.apply_rotary_pos_emb(query_states, key_states, position_ids)
        if not _unreplaced(kv_cache, _PREFILL_STEPS):  # (what it does with the values comes before the attention)
            kv_cache.prefill_kv_cache(value_states, layer_idx, key_states, query_states[:, :, -1:])
            return causal_attention_fp32(query_states, key_states, value_states)
        # prefill_kv_cache in its two halves: the values' copy to the host runs beside the attention, and the
        # attention's launch comes before the state's many small ones, whose issue by the host it covers
        # (MI355X, one layer: 8192 tokens on 8 kv heads 4.17 -> 3.74 ms, 19333 on 2 7.14 -> 6.51 ms).
        pending = kv_cache._begin_prefill(value_states, layer_idx, key_states, query_states[:, :, -1:])
        try:
            return causal_attention_fp32(query_states, key_states, value_states)
        finally:
            kv_cache._end_prefill(pending)

    def decode(self, query_states, key_states, value_states, position_ids, layer_idx):
        """One new token through the layer: decode_begin() and decode_end(). Nothing can overlap the
        value fetch from outside here, so a cache in its default setting takes the shortest chain on the
        current stream: the selection's launch moves both buffers' hits and one launch fetches the missed
        values beside their keys' rebuild, in place of two compaction launches, two stream hops
        and two launches side by side (the same buffer contents). MI355X, values in host memory,
        one sequence of 8192 tokens: 236 -> 144 us, 4 of 122880: 287 -> 242 us."""
        kv_cache = self.kv_cache
        if not self._joined(kv_cache):
            return self.decode_end(self.decode_begin(query_states, key_states, value_states, position_ids, layer_idx))
        query_states, key_states = self.apply_rotary_pos_emb(query_states, key_states, position_ids)
        kv_cache.update_kv_cache(key_states, value_states, layer_idx)
        position_ids = kv_cache.get_retrieval_position_ids(layer_idx=layer_idx, query_states=query_states, fold_all=True)
        workgroups = kv_cache.fused_fetch_workgroups
        if not workgroups and kv_cache.value_store == "host":  # (the default for device memory suits this too)
            workgroups = shadowkv.fetch_workgroups_alone(kv_cache.block_num, kv_cache.select_sets)
        key_states, value_states = kv_cache.fetch_and_rebuild(layer_idx, position_ids, self.cos_sin_cache,
                                                              fetch_workgroups=workgroups)
        return self.decode_end((query_states, key_states, value_states, [], layer_idx))

    def _joined(self, kv_cache) -> bool:
        """Whether decode() takes the joined chain: a ShadowKVCache_CPU in its default setting, no step of either
        chain replaced, in the cache or here (it would not be called, or not as it expects), and a selection
        that it is the faster one for (JOINED_MAX_BUDGET)."""
        return (_unreplaced(kv_cache, _CACHE_STEPS) and _unreplaced(self, _ATTENTION_STEPS) and not kv_cache.pooled
                and not kv_cache.fold_hit_moves and kv_cache.key_stream is None
                and kv_cache.sparse_budget <= JOINED_MAX_BUDGET[kv_cache.value_store])

    def decode_begin(self, query_states, key_states, value_states, position_ids, layer_idx):
        """First half of decode(): RoPE, append, chunk selection, the value fetch launched on the
        cache's copy stream and the key rebuild on the current stream (or on the cache's
        key_stream, when it has one). Returns what decode_end() needs; work issued on the current
        stream in between overlaps the value fetch."""
        kv_cache = self.kv_cache
        query_states, key_states = self.apply_rotary_pos_emb(query_states, key_states, position_ids)
        kv_cache.update_kv_cache(key_states, value_states, layer_idx)
        return self.decode_begin_appended(query_states, layer_idx)

    def decode_begin_appended(self, query_states, layer_idx):
        """decode_begin() for a token already rotated and appended (ShadowKVCache_CPU.rope_and_append):
        query_states [B, Hq, 1, 128] post-RoPE."""
        kv_cache = self.kv_cache
        position_ids = kv_cache.get_retrieval_position_ids(layer_idx=layer_idx, query_states=query_states)

        curr_stream = torch.cuda.current_stream()
        if kv_cache.one_stream_active():
            # the value fetch and the key rebuild as one launch (hits moved by the selection), on this
            # stream or on the cache's lane_stream, joined in decode_end
            lane_stream = getattr(kv_cache, "lane_stream", None)
            if lane_stream is None:
                key_states, value_states = kv_cache.fetch_and_rebuild(layer_idx, position_ids, self.cos_sin_cache)
                return query_states, key_states, value_states, [], layer_idx
            with torch.cuda.stream(lane_stream):
                lane_stream.wait_stream(curr_stream)
                key_states, value_states = kv_cache.fetch_and_rebuild(layer_idx, position_ids, self.cos_sin_cache)
                done = [lane_stream.record_event()]
            return query_states, key_states, value_states, done, layer_idx
        copy_stream = kv_cache.copy_stream
        # The value hits move within the GPU buffer here, so the copy stream (whose transfers
        # follow one another on the host link) carries the host-link gather alone.
        kv_cache.move_value_hits(layer_idx)
        with torch.cuda.stream(copy_stream):
            copy_stream.wait_stream(curr_stream)
            value_states = kv_cache.get_value_cache(layer_idx, position_ids, hits_moved=True)
            done = [copy_stream.record_event()]  # this fetch only, even if the stream is shared
        key_stream = getattr(kv_cache, "key_stream", None)
        if key_stream is None:
            key_states = self._key_path(layer_idx, position_ids)
        else:  # the key rebuild on its own stream too, joined in decode_end
            with torch.cuda.stream(key_stream):
                key_stream.wait_stream(curr_stream)
                key_states = self._key_path(layer_idx, position_ids)
                done.append(key_stream.record_event())
        return query_states, key_states, value_states, done, layer_idx

    def _key_path(self, layer_idx, position_ids):
        return self.kv_cache.get_key_cache(layer_idx=layer_idx, position_ids=position_ids,
                                           rope_func=self.apply_rotary_pos_emb_single,
                                           cos_sin_cache=self.cos_sin_cache)

    def decode_end(self, pending):
        """Second half of decode(), on the stream decode_begin() ran on: wait for the value fetch,
        then sparse attention of the new token over the assembled buffers -> [B, 1, Hq, D] (with
        a value store in device memory read in place, the selected values from the store).
        `pending` is decode_begin()'s result."""
        query_states, key_states, value_states, done, layer_idx = pending
        kv_cache = self.kv_cache
        for event in done:
            torch.cuda.current_stream().wait_event(event)
        if kv_cache.attn_workspace is None:
            kv_cache._alloc_attention()
        B, Hq = query_states.shape[0], query_states.shape[1]
        q = query_states.reshape(B, Hq, -1) if query_states.shape[2] == 1 else None
        if q is None:
            raise ValueError("decode attention takes one query token per step")
        out = torch.empty(B, Hq, query_states.shape[-1], dtype=query_states.dtype, device=query_states.device)
        kv_len, pool = kv_cache.attention_args(key_states.shape[2])
        shadowkv.sparse_attn_decode(q, key_states, value_states, kv_len, out, kv_cache.attn_workspace,
                                    kv_len_dev=kv_cache.kv_len_dev, pool=pool,
                                    vstore=kv_cache.value_store_args(layer_idx))
        return out.view(B, 1, Hq, -1)


_ATTENTION_STEPS = {n: getattr(ShadowAttention, n) for n in ("decode_begin", "decode_begin_appended", "_key_path")}
