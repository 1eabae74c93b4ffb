"""The Gram matrix and the factors of a prompt's keys read in place (skv_keys_gram, skv_keys_factors)
against float64, and get_svd by either route."""
import types

import pytest
import torch

from shadowkv_amd.kernels import shadowkv
from shadowkv_amd.models.kvcache import ShadowKVCache_CPU
from shadowkv_amd.models.kvcache import shadow as kv

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


# Rows around one stage (64), one share and the 256-row blocks; one to eight heads (half, whole and several
# 256-column tiles); ranks of one, a partial and five vector tiles; by head, by token, and padded rows.
@pytest.mark.parametrize("b,rows,H,R,layout", [(1, 1, 1, 4, "token"), (2, 63, 1, 32, "head"), (1, 65, 2, 48, "padded"),
                                               (3, 257, 3, 160, "head"), (1, 511, 8, 36, "token"),
                                               (1, 1025, 4, 320, "padded"), (1, 33000, 1, 128, "head"),
                                               (1, 33001, 2, 160, "token")])
def test_gram_and_factors(gpu, b, rows, H, R, layout):
    """Bounds: a Gram entry is one fp32 sum of exact products (rows * 2^-24 of the sum of magnitudes, ample);
    a factor one fp32 sum of n products, one division and one rounding to bf16."""
    _say(f"gram and factors b={b} rows={rows} H={H} R={R} {layout}")
    g = torch.Generator().manual_seed(rows + H)
    n = H * 128
    k = torch.randn(b, rows, H, 128, generator=g).to(torch.bfloat16)
    if layout == "head":
        dev = k.transpose(1, 2).contiguous().to(gpu).transpose(1, 2)
    elif layout == "padded":
        dev = torch.full((b, rows + 2, H, 136), float("nan"), dtype=torch.bfloat16, device=gpu)[:, 1:-1, :, :128]
        dev.copy_(k)
    else:
        dev = k.to(gpu)
    K = k.view(b, rows, n).double()
    gram = shadowkv.keys_gram(dev)
    want = K.transpose(1, 2) @ K
    assert ((gram.cpu().double() - want).abs() <= rows * 2 ** -24 * (K.abs().transpose(1, 2) @ K.abs()) + 1e-30).all()
    assert torch.equal(gram, gram.transpose(1, 2))

    V = torch.linalg.qr(torch.randn(b, n, max(R, 1), generator=g))[0][..., :R] if R <= n else torch.randn(b, n, R, generator=g)
    if R > n:
        with pytest.raises(RuntimeError):
            shadowkv.keys_factors(dev, torch.ones(b, R, device=gpu), V.transpose(1, 2).contiguous().to(gpu),
                                  torch.empty(b, rows, R, dtype=torch.bfloat16, device=gpu),
                                  torch.empty(b, H, 128, R, dtype=torch.bfloat16, device=gpu))
        return
    w = torch.rand(b, R, generator=g) * 4 + 0.5
    vt = V.transpose(1, 2).contiguous()
    u = torch.full((b, rows, R), 7.0, dtype=torch.bfloat16, device=gpu)
    sv = torch.full((b, H, 128, R), 7.0, dtype=torch.bfloat16, device=gpu)
    shadowkv.keys_factors(dev, w.to(gpu), vt.to(gpu), u, sv)
    s = w.double().sqrt()
    U = (K @ vt.double().transpose(1, 2)) / s.unsqueeze(1)
    lim = U.abs() * (2 ** -8 + 2 ** -20) + n * 2 ** -24 * (K.abs() @ vt.double().abs().transpose(1, 2)) / s.unsqueeze(1)
    assert ((u.cpu().double() - U).abs() <= lim + 1e-30).all()
    S = (s.unsqueeze(-1) * vt.double()).view(b, R, H, 128).permute(0, 2, 3, 1)
    assert ((sv.cpu().double() - S).abs() <= S.abs() * (2 ** -8 + 2 ** -20)).all()


@pytest.mark.parametrize("form", ["head", "token", "odd"])
def test_get_svd_routes(gpu, form, monkeypatch):
    """get_svd through the kernels and through the torch operations: the same reconstruction, for keys by
    head, fused by token, and at an odd offset (which only the torch operations take)."""
    _say(f"get_svd {form}")
    B, H, ctx, R = 2, 2, 700, 64
    g = torch.Generator().manual_seed(3)
    k = (torch.randn(B, ctx, 48, generator=g) @ torch.randn(B, 48, H * 128, generator=g) / 7
         + 0.05 * torch.randn(B, ctx, H * 128, generator=g)).to(torch.bfloat16).to(gpu)
    if form == "head":
        arg = k.view(B, ctx, H, 128).transpose(1, 2).contiguous()
    elif form == "token":
        arg = k
    else:
        arg = torch.empty(B * ctx * H * 128 + 1, dtype=torch.bfloat16, device=gpu)[1:].view(B, ctx, H * 128)
        arg.copy_(k)
    cfg = types.SimpleNamespace(num_attention_heads=2 * H, num_key_value_heads=H, hidden_size=2 * H * 128,
                                num_hidden_layers=1)
    rec = []
    for force in (False, True):
        cache = ShadowKVCache_CPU(cfg, batch_size=B, max_length=ctx, device=str(gpu), sparse_budget=256, rank=R,
                                  value_store="device")
        taken = []
        real = ShadowKVCache_CPU._keys_in_place
        monkeypatch.setattr(ShadowKVCache_CPU, "_keys_in_place",
                            lambda self, x: None if force else (taken.append(real(self, x)) or taken[-1]))
        with monkeypatch.context() as m:
            if not force and form != "odd":  # (the kernels' own factors, and a verdict that takes them)
                m.setattr(kv, "low_rank_factors", lambda *a: pytest.fail("the kernels' factors were not taken"))
            cache.get_svd(arg, 0)
        monkeypatch.setattr(ShadowKVCache_CPU, "_keys_in_place", real)
        if not force:
            assert (taken[0] is None) == (form == "odd")
        rec.append(torch.einsum("bcr,bhdr->bchd", cache.U[0].float(), cache.SV[0].float()).double())
    diff = (rec[0] - rec[1]).norm() / rec[1].norm()
    assert diff < 4e-3, diff  # two bf16 roundings of the same fp32 factors, up to their signs
    err = (rec[0].reshape(B, ctx, -1) - k.double()).norm() / k.double().norm()
    assert err < 0.08  # the noise outside rank 64


def test_get_svd_after_a_refused_verdict(gpu, monkeypatch):
    """Eigenpairs that do not hold up, whose factors are written before the host reads the verdict: replaced by the
    torch operations' factors."""
    _say("get_svd after a refused verdict")
    H, ctx, R = 2, 700, 64
    k = torch.randn(1, H, ctx, 128, generator=torch.Generator().manual_seed(8)).to(torch.bfloat16).to(gpu)
    cfg = types.SimpleNamespace(num_attention_heads=H, num_key_value_heads=H, hidden_size=H * 128, num_hidden_layers=1)
    make = dict(batch_size=1, max_length=ctx, device=str(gpu), sparse_budget=64, rank=R, value_store="device")
    want = ShadowKVCache_CPU(cfg, **make)
    with monkeypatch.context() as m:
        m.setattr(ShadowKVCache_CPU, "_keys_in_place", lambda self, x: None)
        want.get_svd(k, 0)
    got = ShadowKVCache_CPU(cfg, **make)
    real, calls = kv._top_eigenpairs, []

    def refuse_first(gram, rank):
        w, vt, ok = real(gram, rank)
        calls.append(bool(ok))
        return (w, vt, ok) if len(calls) > 1 else (w.fill_(float("nan")), vt.fill_(3.0), torch.zeros_like(ok))

    monkeypatch.setattr(kv, "_top_eigenpairs", refuse_first)
    got.get_svd(k, 0)
    assert calls == [True, True]
    assert torch.equal(got.U, want.U) and torch.equal(got.SV, want.SV)


@pytest.mark.parametrize("ctx,max_length,B,first", [(1400, 1400, 2, 2), (1403, 2048, 2, 1), (1800, 4096, 3, 2)])
def test_prefill_value_copy(gpu, ctx, max_length, B, first):
    """The host store after prefill and prefill_kv_cache, from whole, ragged and padded rows and batches
    prefilled in parts: every value chunk, nothing else; a transposed view of the values too."""
    from shadowkv_amd.models.attention import ShadowAttention
    from shadowkv_amd.models.tensor_op import build_cos_sin_cache
    _say(f"value copy ctx={ctx} max={max_length} B={B} first={first}")
    H, G, D, c = 2, 2, 128, 8
    cfg = types.SimpleNamespace(num_attention_heads=G * H, num_key_value_heads=H, hidden_size=G * H * D,
                                num_hidden_layers=1)
    g = torch.Generator().manual_seed(ctx)
    table = build_cos_sin_cache(max_length, 10000.0, D, device=gpu)
    q, k, v = (torch.randn(B, h, ctx, D, generator=g).to(torch.bfloat16).to(gpu) for h in (G * H, H, H))
    for form in ("prefill", "encode", "view"):
        cache = ShadowKVCache_CPU(cfg, batch_size=B, max_length=max_length, device=str(gpu), sparse_budget=1024, rank=32)
        attn = ShadowAttention(cache, G, D, G * H * D, lambda a, b, p: (a, b), None, table)
        for lo, hi in ((0, first), (first, B)):
            if lo == hi:
                continue
            vv = v[lo:hi] if form != "view" else v[lo:hi].transpose(1, 2).contiguous().transpose(1, 2)
            if form == "prefill":
                attn.prefill(q[lo:hi], k[lo:hi], vv, None, 0)
            else:
                cache.get_svd(k[lo:hi], 0)
                cache.prefill_kv_cache(vv, 0, k[lo:hi], q[lo:hi, :, -1:])
            n = ctx // c
            got = cache.v_cache_cpu[0]  # (read at once: the call has waited for the copy)
            assert torch.equal(got[lo:hi, :, :n], v[lo:hi, :, :n * c].reshape(hi - lo, H, n, c * D).cpu())
            assert not got[:, :, n:].any() and not got[hi:].any()
        del cache, attn


def test_prefill_replaced_kv_cache_step(gpu, monkeypatch):
    """A prefill_kv_cache replaced in a subclass, on the class, on the instance or in another cache
    altogether: the store holds the values that it passed on, not those that prefill was given, and the
    attention takes the values as it left them."""
    from shadowkv_amd.models.attention import ShadowAttention, shadow
    from shadowkv_amd.models.tensor_op import build_cos_sin_cache
    _say("prefill with a replaced prefill_kv_cache")
    H, G, D, ctx, c = 2, 2, 128, 1400, 8
    cfg = types.SimpleNamespace(num_attention_heads=G * H, num_key_value_heads=H, hidden_size=G * H * D,
                                num_hidden_layers=1)
    g = torch.Generator().manual_seed(4)
    q, k, v = (torch.randn(1, h, ctx, D, generator=g).to(torch.bfloat16).to(gpu) for h in (G * H, H, H))
    table = build_cos_sin_cache(ctx, 10000.0, D, device=gpu)
    make = dict(batch_size=1, max_length=ctx, device=str(gpu), sparse_budget=1024, rank=32)
    real = ShadowKVCache_CPU.prefill_kv_cache

    def scaled(self, values, *args):
        real(self, 2 * values, *args)

    def in_place(self, values, *args):
        real(self, values.mul_(2), *args)

    class Delegating:  # the methods that prefill calls, and no others
        def __init__(self, inner):
            self.get_svd, self.prefill_kv_cache = inner.get_svd, inner.prefill_kv_cache

    for form in ("subclass", "class", "instance", "in place", "delegating", "none"):
        factor = 1 if form in ("delegating", "none") else 2
        with monkeypatch.context() as m:
            cls = ShadowKVCache_CPU
            if form in ("subclass", "in place"):
                cls = type("Replacing", (cls,), {"prefill_kv_cache": scaled if form == "subclass" else in_place})
            cache = cls(cfg, **make)
            if form == "class":
                m.setattr(ShadowKVCache_CPU, "prefill_kv_cache", scaled)
            if form == "instance":
                cache.prefill_kv_cache = types.MethodType(scaled, cache)
            attn = ShadowAttention(Delegating(cache) if form == "delegating" else cache, G, D, G * H * D,
                                   lambda a, b, p: (a, b), None, table)
            given = v.clone()
            out = attn.prefill(q, k, given, None, 0)
            want = (factor * v).view(1, H, ctx // c, c * D).cpu()
            assert torch.equal(cache.v_cache_cpu[0][:, :, :ctx // c], want), form
            used = 2 * v if form == "in place" else v
            assert torch.equal(given, used) and torch.equal(out, shadow.causal_attention_fp32(q, k, used)), form


def test_prefill_refusals_leave_the_store(gpu):
    """A prompt that prefill_kv_cache refuses leaves the store as it was, through prefill too."""
    from shadowkv_amd.models.attention import ShadowAttention
    from shadowkv_amd.models.tensor_op import build_cos_sin_cache
    _say("refused prompts")
    H, G, D, ctx = 2, 2, 128, 1400
    cfg = types.SimpleNamespace(num_attention_heads=G * H, num_key_value_heads=H, hidden_size=G * H * D,
                                num_hidden_layers=1)
    q, k, v = (torch.ones(1, h, ctx, D, dtype=torch.bfloat16, device=gpu) for h in (G * H, H, H))
    cache = ShadowKVCache_CPU(cfg, batch_size=1, max_length=ctx, device=str(gpu), sparse_budget=1024, rank=32)
    attn = ShadowAttention(cache, G, D, G * H * D, lambda a, b, p: (a, b.cpu()), None,
                           build_cos_sin_cache(ctx, 10000.0, D, device=gpu))
    with pytest.raises(ValueError, match="device"):  # keys on the host
        attn.prefill(q, k, v, None, 0)
    torch.cuda.synchronize()
    assert not cache.v_cache_cpu[0].any() and cache.prefilled_batch == 0


@pytest.mark.parametrize("rows,R", [(600, 192), (50200, 32), (70000, 64), (50200, 72), (50200, 96), (33000, 128), (44000, 160),
                                    (50200, 132), (50200, 160), (33000, 164), (50200, 192), (50200, 200)])
def test_factors_forms(gpu, rows, R):
    """Each form of the projection (1, 2, 3 and 5 tiles of 32 vectors a workgroup) with whole and partial last groups
    and tiles, at one head; the bound of test_gram_and_factors."""
    _say(f"factors rows={rows} R={R}")
    n = 256 if R > 128 else 128
    g = torch.Generator().manual_seed(rows + R)
    k = torch.randn(1, rows, n // 128, 128, generator=g).to(torch.bfloat16)
    vt = torch.randn(1, R, n, generator=g) / n ** 0.5
    w = torch.rand(1, R, generator=g) * 4 + 0.5
    u = torch.full((1, rows + 1, R), 7.0, dtype=torch.bfloat16, device=gpu)
    sv = torch.empty(1, n // 128, 128, R, dtype=torch.bfloat16, device=gpu)
    shadowkv.keys_factors(k.to(gpu), w.to(gpu), vt.to(gpu), u[:, :rows], sv)
    K, V, s = k.view(rows, n).double(), vt[0].double().T, w[0].double().sqrt()
    want = (K @ V) / s
    lim = want.abs() * (2 ** -8 + 2 ** -20) + n * 2 ** -24 * (K.abs() @ V.abs()) / s
    assert ((u[0, :rows].cpu().double() - want).abs() <= lim + 1e-30).all()
    assert (u[0, rows] == 7).all(), "wrote past the rows"


@pytest.mark.parametrize("max_length", [1400, 1480])
def test_value_copy_of_many_rows(gpu, max_length):
    """More than 64 (sequence, head) rows, as one transfer and row by row."""
    B, H, ctx, D, c = 33, 2, 1400, 128, 8
    _say(f"value copy of {B * H} rows, max={max_length}")
    cfg = types.SimpleNamespace(num_attention_heads=H, num_key_value_heads=H, hidden_size=H * D, num_hidden_layers=1)
    cache = ShadowKVCache_CPU(cfg, batch_size=B, max_length=max_length, device=str(gpu), sparse_budget=1024, rank=32)
    v = torch.randn(B, H, ctx, D, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(gpu)
    copy = cache.start_value_copy(v, 0)
    assert copy is not None
    copy.synchronize()
    assert torch.equal(cache.v_cache_cpu[0][:, :, :ctx // c], v.view(B, H, ctx // c, c * D).cpu())
    assert not cache.v_cache_cpu[0][:, :, ctx // c:].any()


@pytest.mark.parametrize("B,rows", [(11, 700), (9, 2500), (20, 100), (300, 17000)])
def test_gram_of_large_batches(gpu, B, rows):
    """Batches whose sequences' shares begin on another XCD each, with fewer shares than XCDs, one, and several
    because a share is full; the bound of test_gram_and_factors, and equal sequences have equal bits."""
    _say(f"gram of a batch of {B} x {rows}")
    g = torch.Generator().manual_seed(rows)
    k = torch.randn(min(B, 20), rows, 1, 128, generator=g).to(torch.bfloat16)
    dev = k.to(gpu) if B <= 20 else k[:1].to(gpu).expand(B, rows, 1, 128)
    gram = shadowkv.keys_gram(dev)
    K = k[:, :, 0].double() if B <= 20 else k[:1, :, 0].double()
    want = K.transpose(1, 2) @ K
    lim = rows * 2 ** -24 * (K.abs().transpose(1, 2) @ K.abs()) + 1e-30
    assert ((gram[:len(K)].cpu().double() - want).abs() <= lim).all()
    assert B <= 20 or (gram == gram[:1]).all()


def test_get_svd_of_a_large_batch(gpu, monkeypatch):
    """More than 64 sequences at once: by the kernels, the same factors as each sequence's own."""
    B, ctx, R = 67, 300, 32
    _say(f"get_svd of {B} sequences")
    k = torch.randn(B, 1, ctx, 128, generator=torch.Generator().manual_seed(6)).to(torch.bfloat16).to(gpu)
    cfg = types.SimpleNamespace(num_attention_heads=1, num_key_value_heads=1, hidden_size=128, num_hidden_layers=1)
    make = dict(max_length=ctx, device=str(gpu), sparse_budget=64, rank=R, value_store="device")
    monkeypatch.setattr(kv, "low_rank_factors", lambda *a: pytest.fail("not by the kernels"))
    cache = ShadowKVCache_CPU(cfg, batch_size=B, **make)
    cache.get_svd(k, 0)
    for b in (0, 8, 66):
        one = ShadowKVCache_CPU(cfg, batch_size=1, **make)
        one.get_svd(k[b:b + 1], 0)
        assert torch.equal(cache.U[0][b], one.U[0][0]) and torch.equal(cache.SV[0][b], one.SV[0][0])


def test_get_svd_of_regrouped_heads(gpu):
    """Keys by head whose heads are not the cache's: taken as rows of H * D columns, as their transpose gives them."""
    _say("get_svd of regrouped heads")
    H, ctx, R = 4, 300, 32
    cfg = types.SimpleNamespace(num_attention_heads=H, num_key_value_heads=H, hidden_size=H * 128, num_hidden_layers=1)
    make = dict(batch_size=1, max_length=ctx, device=str(gpu), sparse_budget=64, rank=R, value_store="device")
    for heads, rows in ((2, 2 * ctx), (8, ctx // 2)):
        k = torch.randn(1, heads, rows, 128, generator=torch.Generator().manual_seed(heads)).to(torch.bfloat16).to(gpu)
        got, want = ShadowKVCache_CPU(cfg, **make), ShadowKVCache_CPU(cfg, **make)
        got.get_svd(k, 0)
        want.get_svd(k.transpose(1, 2).reshape(1, ctx, H * 128), 0)
        assert got.U.shape == want.U.shape == (1, 1, ctx, R)
        a, b = (torch.einsum("bcr,bhdr->bchd", c.U[0].float().cpu(), c.SV[0].float().cpu()) for c in (got, want))
        assert (a - b).norm() <= 8e-3 * b.norm()  # two roundings to bf16 of either route's factors
