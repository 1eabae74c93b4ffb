"""ShadowAttention.decode (selection with folded hit moves, one fetch + rebuild launch) against
decode_begin + decode_end (two streams): the same bits in the output, the selection and both buffers."""
import types

import pytest
import torch

from shadowkv_amd.decode_model import synthesize_state
from shadowkv_amd.models.attention import ShadowAttention, shadow
from shadowkv_amd.models.kvcache import ShadowKVCache_CPU
from shadowkv_amd.models.tensor_op import apply_rotary_pos_emb_cuda, build_cos_sin_cache, build_glm_cos_sin_cache

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


# One chunk size below, at and above the default, both stores, a selection of the largest size
# (2048 chunks), both rotary layouts, fetches of fewer and of more tiles than workgroups.
@pytest.mark.parametrize("B,H,G,ctx,budget,chunk,store,glm", [
    (1, 8, 4, 6000, 1024, 8, "host", False), (2, 2, 16, 5003, 1024, 4, "host", True),
    (3, 3, 1, 9001, 2048, 16, "host", False), (2, 2, 4, 40000, 16384, 8, "host", False),
    (2, 8, 4, 6000, 1024, 8, "device", False), (1, 2, 16, 20011, 2048, 16, "device", True),
    (16, 8, 4, 6000, 4096, 8, "host", False)])
def test_decode_equals_begin_and_end(gpu, monkeypatch, B, H, G, ctx, budget, chunk, store, glm):
    _say(f"decode chain B={B} H={H} G={G} ctx={ctx} budget={budget} chunk={chunk} {store} glm={glm}")
    D, steps = 128, 4
    table = (build_glm_cos_sin_cache(ctx + 64, 10000.0, device=gpu) if glm
             else build_cos_sin_cache(ctx + 64, 500000.0, D, device=gpu))
    cfg = types.SimpleNamespace(num_attention_heads=H * G, num_key_value_heads=H, hidden_size=H * G * D,
                                num_hidden_layers=1)
    g = torch.Generator(device=gpu).manual_seed(ctx)
    base = torch.randn(B, H * G, 1, D, generator=g, device=gpu)
    qs = [(0.95 * base + 0.3 * torch.randn(B, H * G, 1, D, generator=g, device=gpu)).to(torch.bfloat16)
          for _ in range(steps)]
    kv = [torch.randn(2, B, H, 1, D, generator=g, device=gpu).to(torch.bfloat16) for _ in range(steps)]
    half = build_cos_sin_cache(ctx + 64, 500000.0, D, device=gpu)

    def rope(q, k, pos):
        return (apply_rotary_pos_emb_cuda(q, half, pos.expand(B, H * G, 1)),
                apply_rotary_pos_emb_cuda(k, half, pos.expand(B, H, 1)))

    got = []
    for joined in (True, False):
        cache = ShadowKVCache_CPU(cfg, batch_size=B, max_length=ctx, device=str(gpu), sparse_budget=budget,
                                  chunk_size=chunk, rank=64, max_decode_len=steps, value_store=store)
        synthesize_state(cache, ctx, seed=7, cos_sin=table)
        attn = ShadowAttention(cache, G, D, H * G * D, rope, None, table)
        if store == "host" and budget > 8192:  # (not the chain that decode() takes by itself at this width)
            monkeypatch.setitem(shadow.JOINED_MAX_BUDGET, store, budget)
        assert attn._joined(cache)
        outs = []
        for i in range(steps):
            pos = torch.full((1, 1, 1), ctx + i, dtype=torch.int64, device=gpu)
            args = (qs[i], kv[i][0], kv[i][1], pos, 0)
            out = attn.decode(*args) if joined else attn.decode_end(attn.decode_begin(*args))
            live = cache.sparse_end + cache.gen_offset
            v = cache.v_cache_buffer[0, :, :, :live].clone()
            if store == "device":  # (read in place: the selected region of the value buffer is not kept)
                v[:, :, cache.sparse_start:cache.sparse_end] = 0
            outs.append([out.clone(), cache.position_ids.clone(), cache.cnts.clone(),
                         cache.k_cache_buffer[0, :, :, :live].clone(), v])
        torch.cuda.synchronize()
        got.append(outs)
        del cache, attn
    for i in range(steps):
        for a, b, what in zip(got[0][i], got[1][i], ("output", "position_ids", "hits", "keys", "values")):
            assert torch.equal(a, b), (i, what)
    assert any(0 < int(x[2].max()) for x in got[0][1:]), "no cache hits: the moves were not exercised"


def test_replaced_steps_are_called(gpu):
    """A cache or attention whose steps of the two-stream chain are replaced, on the instance or in a
    subclass, keeps that chain."""
    _say("decode chain replaced steps")
    cfg = types.SimpleNamespace(num_attention_heads=8, num_key_value_heads=2, hidden_size=1024, num_hidden_layers=1)
    table = build_cos_sin_cache(3000, 500000.0, 128, device=gpu)

    class Counting(ShadowKVCache_CPU):
        calls = 0

        def get_key_cache(self, *args, **kwargs):
            Counting.calls += 1
            return super().get_key_cache(*args, **kwargs)

    def run(cls, patch):
        cache = cls(cfg, batch_size=1, max_length=2500, device=str(gpu), sparse_budget=1024, rank=64, max_decode_len=4)
        synthesize_state(cache, 2500, seed=7, cos_sin=table)
        attn = ShadowAttention(cache, 4, 128, 1024, lambda q, k, p: (q, k), None, table)
        joined = attn._joined(cache)
        if patch:
            real = cache.get_key_cache
            cache.get_key_cache = lambda *a, **k: (patch.append(1), real(*a, **k))[1]
        q = torch.ones(1, 8, 1, 128, dtype=torch.bfloat16, device=gpu)
        kv = torch.ones(1, 2, 1, 128, dtype=torch.bfloat16, device=gpu)
        out = attn.decode(q, kv, kv, None, 0)
        torch.cuda.synchronize()
        return joined, out

    joined, want = run(ShadowKVCache_CPU, None)
    assert joined
    joined, got = run(Counting, None)
    assert not joined and Counting.calls == 1 and torch.equal(got, want)
    hits = [0]
    _, got = run(ShadowKVCache_CPU, hits)
    assert len(hits) == 2 and torch.equal(got, want)


@pytest.mark.parametrize("form", ["class", "delegating", "fetch_and_rebuild", "attention class"])
def test_other_replacements_keep_the_chain(gpu, form, monkeypatch):
    """A step patched on the class itself, a cache of another class that hands its attributes on, a
    fetch_and_rebuild with the arguments it had, and an attention step patched on the class."""
    _say(f"decode chain: {form}")
    cfg = types.SimpleNamespace(num_attention_heads=8, num_key_value_heads=2, hidden_size=1024, num_hidden_layers=1)
    table = build_cos_sin_cache(3000, 500000.0, 128, device=gpu)
    calls = []

    class Own(ShadowKVCache_CPU):
        def fetch_and_rebuild(self, layer_idx, position_ids, cos_sin_cache):
            raise AssertionError("not a step of the two-stream chain")

    class Delegating:
        def __init__(self, inner):
            self._inner = inner

        def __getattr__(self, name):
            return getattr(self._inner, name)

    def run(patched):
        cls = Own if patched and form == "fetch_and_rebuild" else ShadowKVCache_CPU
        cache = cls(cfg, batch_size=1, max_length=2500, device=str(gpu), sparse_budget=1024, rank=64, max_decode_len=4)
        synthesize_state(cache, 2500, seed=7, cos_sin=table)
        if patched and form == "delegating":
            cache = Delegating(cache)
        attn = ShadowAttention(cache, 4, 128, 1024, lambda q, k, p: (q, k), None, table)
        assert attn._joined(cache) != patched
        q = torch.ones(1, 8, 1, 128, dtype=torch.bfloat16, device=gpu)
        kv = torch.ones(1, 2, 1, 128, dtype=torch.bfloat16, device=gpu)
        out = attn.decode(q, kv, kv, None, 0)
        torch.cuda.synchronize()
        return out

    want = run(False)
    if form in ("class", "attention class"):
        owner, name = {"class": (ShadowKVCache_CPU, "get_key_cache"),
                       "attention class": (ShadowAttention, "_key_path")}[form]
        real = getattr(owner, name)
        monkeypatch.setattr(owner, name, lambda self, *a, **k: (calls.append(1), real(self, *a, **k))[1])
    assert torch.equal(run(True), want)
    assert len(calls) == (form in ("class", "attention class"))


def _fetch_launches(gpu, monkeypatch, **attrs):
    """The fetch workgroups that decode() asks for, of a cache with the given settings."""
    from shadowkv_amd.kernels import shadowkv
    cfg = types.SimpleNamespace(num_attention_heads=8, num_key_value_heads=2, hidden_size=1024, num_hidden_layers=1)
    table = build_cos_sin_cache(3000, 500000.0, 128, device=gpu)
    cache = ShadowKVCache_CPU(cfg, batch_size=1, max_length=2500, device=str(gpu), sparse_budget=1024, rank=64,
                              max_decode_len=4, value_store=attrs.pop("value_store", "host"))
    for name, value in attrs.items():
        setattr(cache, name, value)
    synthesize_state(cache, 2500, seed=7, cos_sin=table)
    attn = ShadowAttention(cache, 4, 128, 1024, lambda q, k, p: (q, k), None, table)
    real, asked = shadowkv.fetch_misses_rebuild_k_rope, []
    with monkeypatch.context() as m:
        m.setattr(shadowkv, "fetch_misses_rebuild_k_rope",
                  lambda *a, fetch_workgroups=0, **k: (asked.append(fetch_workgroups),
                                                       real(*a, fetch_workgroups=fetch_workgroups, **k))[1])
        q = torch.ones(1, 8, 1, 128, dtype=torch.bfloat16, device=gpu)
        kv = torch.ones(1, 2, 1, 128, dtype=torch.bfloat16, device=gpu)
        attn.decode(q, kv, kv, None, 0)
        torch.cuda.synchronize()
    return asked


def test_fetch_workgroups_of_a_gathered_device_store(gpu, monkeypatch):
    """A store in device memory that is gathered from: the library's own count for it, or the cache's."""
    _say("decode chain: fetch workgroups of a device store")
    assert _fetch_launches(gpu, monkeypatch, value_store="device", values_in_place=False) == [0]
    assert _fetch_launches(gpu, monkeypatch, value_store="device", values_in_place=False,
                           fused_fetch_workgroups=40) == [40]


def test_fetch_workgroups_of_a_host_store(gpu, monkeypatch):
    """A store in host memory: the library's count for a launch alone (which the environment overrides), or the
    cache's."""
    from shadowkv_amd.kernels import shadowkv
    _say("decode chain: fetch workgroups of a host store")
    monkeypatch.setattr(shadowkv, "fetch_workgroups_alone", lambda *a: 33)
    assert _fetch_launches(gpu, monkeypatch) == [33]
    assert _fetch_launches(gpu, monkeypatch, fused_fetch_workgroups=40) == [40]


@pytest.mark.parametrize("store,budget,joined", [("host", 8192, True), ("host", 16384, False), ("device", 16384, True),
                                                 ("device", 32768, False)])
def test_wide_selections_keep_the_two_streams(gpu, monkeypatch, store, budget, joined):
    """A selection too wide for its rows' workgroups to move the hits: the two-stream chain, with the bits of
    the joined one."""
    _say(f"decode chain {store} budget={budget}")
    ctx, chunk = 60000, 16
    cfg = types.SimpleNamespace(num_attention_heads=8, num_key_value_heads=2, hidden_size=1024, num_hidden_layers=1)
    table = build_cos_sin_cache(ctx + 8, 500000.0, 128, device=gpu)
    g = torch.Generator(device=gpu).manual_seed(1)
    base = torch.randn(1, 8, 1, 128, generator=g, device=gpu)
    qs = [(0.95 * base + 0.3 * torch.randn(1, 8, 1, 128, generator=g, device=gpu)).to(torch.bfloat16) for _ in range(3)]
    kv = torch.randn(1, 2, 1, 128, generator=g, device=gpu).to(torch.bfloat16)
    got = []
    for force in (False, True):
        cache = ShadowKVCache_CPU(cfg, batch_size=1, max_length=ctx, device=str(gpu), sparse_budget=budget,
                                  chunk_size=chunk, rank=64, max_decode_len=4, value_store=store)
        synthesize_state(cache, ctx, seed=7, cos_sin=table)
        attn = ShadowAttention(cache, 4, 128, 1024, lambda q, k, p: (q, k), None, table)
        if force:
            monkeypatch.setitem(shadow.JOINED_MAX_BUDGET, store, budget if not joined else budget - 1)
        assert attn._joined(cache) == (joined != force)
        got.append([attn.decode(q, kv, kv, None, 0) for q in qs] + [cache.position_ids, cache.cnts])
        torch.cuda.synchronize()
    assert int(got[0][-1].max()) > 0
    assert all(torch.equal(a, b) for a, b in zip(*got))
