"""The prompt attention kernel (skv_prefill_attn) against float64 causal attention, and the calls that
stay with the torch operations."""
import math

import pytest
import torch

from shadowkv_amd.kernels import shadowkv
from shadowkv_amd.models.attention import shadow

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


def _exact(q, k, v):
    B, Hq, L, D = q.shape
    G = Hq // k.shape[1]
    kk, vv = (x.double().cpu().repeat_interleave(G, dim=1) for x in (k, v))
    s = q.double().cpu() @ kk.transpose(-1, -2) / math.sqrt(D)
    s.masked_fill_(torch.ones(L, L, dtype=torch.bool).triu(1), float("-inf"))
    return (torch.softmax(s, -1) @ vv).transpose(1, 2)


# Lengths around the 64-key tiles and the 32- and 128-query blocks; (batch, kv head) rows that divide
# among the 8 XCDs (once and several times), that the XCDs divide among, and neither.
@pytest.mark.parametrize("L", [1, 31, 64, 65, 127, 129, 300])
@pytest.mark.parametrize("B,Hq,H", [(1, 8, 8), (2, 4, 1), (1, 6, 3), (3, 16, 1), (2, 16, 8), (3, 16, 8), (1, 5, 5)])
def test_prefill_attn_edges(gpu, B, Hq, H, L):
    """Bound: one bf16 rounding (2^-8) of the value; fp32 scores of magnitude <= ~20 err by 20 * 2^-22
    relative in a probability, so 1e-4 of the largest value is ample."""
    _say(f"prefill_attn B={B} Hq={Hq} H={H} L={L}")
    g = torch.Generator().manual_seed(L * 100 + B * 10 + Hq)
    # q as the transposed view of a projection, k and v as slices of a fused one
    q = (torch.randn(B, L, Hq, 128, generator=g) * 1.5).to(torch.bfloat16).to(gpu).transpose(1, 2)
    kv = torch.randn(B, L, 2 * H, 128, generator=g).to(torch.bfloat16).to(gpu).transpose(1, 2)
    k, v = kv[:, :H], kv[:, H:]
    assert shadow._kernel_takes(q, k, v)
    out = shadow.causal_attention_fp32(q, k, v)
    assert out.shape == (B, L, Hq, 128)
    want = _exact(q, k, v)
    err = (out.cpu().double() - want).abs()
    assert (err <= want.abs() * 2 ** -8 + 1e-4 * v.abs().max().item()).all(), err.max()


def test_prefill_attn_growing_scores_and_alignment(gpu):
    """Scores that grow along the keys (the running maximum moves in every tile) and far below the
    first tile's (never moved), keys hidden by causality set to NaN, and rows at an odd offset (copied)."""
    L = 200
    _say("prefill_attn growing scores")
    g = torch.Generator().manual_seed(9)
    q = torch.ones(1, 2, L, 128).to(torch.bfloat16)
    ramp = torch.linspace(-20, 20, L)[None, None, :, None]
    for sign in (1, -1):
        k = (sign * ramp + 0.1 * torch.randn(1, 1, L, 128, generator=g)).to(torch.bfloat16)
        v = torch.randn(1, 1, L, 128, generator=g).to(torch.bfloat16)
        out = shadowkv.prefill_attn(q.to(gpu), k.to(gpu), v.to(gpu)).cpu().double()
        want = _exact(q, k, v)  # scores to +-226: a probability errs by up to 226 * 2^-23 relative
        assert ((out - want).abs() <= want.abs() * 2 ** -8 + 1e-3).all()
    kn = k.clone()
    kn[:, :, 150:] = float("nan")
    flat = torch.zeros(2 * L * 128 + 1, dtype=torch.bfloat16, device=gpu)
    flat[1:] = q.flatten().to(gpu)
    out2 = shadowkv.prefill_attn(flat[1:].view(1, 2, L, 128), kn.to(gpu), v.to(gpu)).cpu().double()
    assert torch.equal(out2[:, :150], out[:, :150])
    assert out2[:, 150:].isnan().all()


def test_differentiated_and_other_calls_stay_with_torch(gpu):
    _say("prefill_attn routing")
    g = torch.Generator().manual_seed(2)
    q, k, v = (torch.randn(1, h, 40, 128, generator=g).to(torch.bfloat16).to(gpu) for h in (4, 2, 2))
    qg = q.clone().requires_grad_()
    assert not shadow._kernel_takes(qg, k, v)
    shadow.causal_attention_fp32(qg, k, v).float().sum().backward()
    assert qg.grad is not None and qg.grad.abs().sum() > 0
    with torch.no_grad():
        assert shadow._kernel_takes(qg, k, v)
    for a in ((q.float(), k.float(), v.float()), (q[..., :64], k[..., :64], v[..., :64]), (q[:, :, :0], k[:, :, :0], v[:, :, :0]),
              (q.cpu(), k.cpu(), v.cpu()), (q, k, v[:, :, :20])):
        assert not shadow._kernel_takes(*a)
    with pytest.raises(RuntimeError, match="vmap"):  # refused by the torch operations' in-place output
        torch.func.vmap(lambda a: shadow.causal_attention_fp32(a[None], k, v)[0])(q)
    with torch.autograd.forward_ad.dual_level():
        dq = torch.autograd.forward_ad.make_dual(q, torch.ones_like(q))
        out = torch.autograd.forward_ad.unpack_dual(shadow.causal_attention_fp32(dq, k, v))
        assert out.tangent is not None


@pytest.mark.parametrize("L,at", [(1, 0), (70, 0), (200, 3), (200, 64), (300, 130)])
def test_prefill_attn_infinite_values(gpu, L, at):
    """An infinite value reaches every query that sees its key, whatever the bits of its probability (the
    first query's is exactly 1), of either sign; both signs of one dim, and a NaN, give NaN. The other
    dims and the queries of earlier tiles (64 keys) are as without."""
    _say(f"prefill_attn infinite values L={L} at={at}")
    g = torch.Generator().manual_seed(L + at)
    q, k, v = (torch.randn(1, h, L, 128, generator=g).to(torch.bfloat16) for h in (4, 2, 2))
    q[:, :, : L // 2] = 0.0  # equal scores: probabilities 1 / (i + 1), half of them short in binary
    plain = shadowkv.prefill_attn(q.to(gpu), k.to(gpu), v.to(gpu)).cpu()
    inf = float("inf")
    v[0, 0, at, 5], v[0, 0, at, 6], v[0, 1, at, 7], v[0, 1, L - 1, 7], v[0, 1, at, 9] = inf, -inf, inf, -inf, float("nan")
    out = shadowkv.prefill_attn(q.to(gpu), k.to(gpu), v.to(gpu)).cpu()
    seen = out[0, at:]  # [queries, heads, dims]: heads 0, 1 read kv head 0 and heads 2, 3 kv head 1
    last = max(0, (L - 1) // 64 * 64 - at)  # from this one on a query's own tile holds the last key's -inf
    assert (seen[:, :2, 5] == inf).all() and (seen[:, :2, 6] == -inf).all()
    if at == L - 1:
        assert (seen[:, 2:, 7] == -inf).all()  # (the same key: overwritten)
    else:
        assert (seen[:last, 2:, 7] == inf).all() and seen[-1, 2:, 7].isnan().all()
    assert seen[:, 2:, 9].isnan().all()
    same = torch.ones(4, 128, dtype=torch.bool)
    same[:2, 5:7] = False
    same[2:, [7, 9]] = False
    assert torch.equal(out[0][:, same], plain[0][:, same])
    first = min(at, L - 1) // 64 * 64
    assert torch.equal(out[0, :first], plain[0, :first])
