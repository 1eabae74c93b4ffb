"""The leading eigenpairs of symmetric positive semidefinite matrices (skv_sym_eig_top) against the
float64 eigendecomposition, and the factors where the kernel's result is not taken."""
import threading
import types

import pytest
import torch

from shadowkv_amd.kernels import shadowkv
from shadowkv_amd.models.kvcache import shadow as kv
from shadowkv_amd.streams import capture_graph

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


def _check(a, rank, scale=1.0):
    """Residuals, orthogonality and eigenvalues within n * 2^-24 of the largest eigenvalue (the backward
    error of a Householder reduction in fp32)."""
    w, vt, status = shadowkv.sym_eig_top(a, rank)
    torch.cuda.synchronize()
    assert (status.cpu() == 1).all()
    b, n, _ = a.shape
    lim = max(n, 64) * 2 ** -24
    A, W, V = a.cpu().double(), w.cpu().double(), vt.cpu().double()
    want = torch.linalg.eigvalsh(A).flip(-1)[:, :rank]
    top = want[:, :1]
    assert ((W - want).abs() <= lim * top).all()
    assert ((V @ A - W.unsqueeze(-1) * V).norm(dim=-1) <= lim * top).all()
    assert ((V @ V.transpose(1, 2) - torch.eye(rank, dtype=torch.float64)).abs() <= lim).all()


# Sizes at, below and past the register tiles (64 NR rows: 128, 256, 512, 1024) and phases.
@pytest.mark.parametrize("b,n,rank", [(1, 2, 2), (1, 3, 1), (8, 17, 17), (1, 64, 16), (2, 127, 40), (1, 128, 128), (1, 129, 7),
                                      (3, 256, 160), (1, 300, 12), (1, 512, 160), (2, 513, 20), (1, 1000, 160),
                                      (1, 1023, 3), (2, 1024, 160)])
def test_sym_eig_top(gpu, b, n, rank):
    _say(f"sym_eig_top b={b} n={n} rank={rank}")
    g = torch.Generator().manual_seed(n + rank)
    x = torch.randn(b, 2 * n + 5, n, generator=g) * torch.logspace(0.5, -0.5, n)
    a = (x.transpose(1, 2) @ x * 2.0 ** (n % 40 - 20)).to(gpu)
    a = (0.5 * (a + a.transpose(1, 2))).contiguous()
    _check(a, rank)


@pytest.mark.parametrize("kind", ["low rank", "diagonal", "steep", "one entry"])
def test_sym_eig_top_special_spectra(gpu, kind):
    """Reflections of zero columns, split tridiagonals and eigenvalues down to rounding noise."""
    _say(f"sym_eig_top {kind}")
    g = torch.Generator().manual_seed(5)
    n = 256
    if kind == "low rank":
        x = torch.randn(1, 600, 40, generator=g) @ torch.randn(1, 40, n, generator=g)
        rank = 40
    elif kind == "diagonal":
        x, rank = torch.diag(torch.linspace(1, 3, n))[None], 30
    elif kind == "steep":
        x, rank = torch.randn(1, 600, n, generator=g) * torch.logspace(0, -6, n), 30
    else:
        x, rank = torch.zeros(1, n, n), 1
        x[0, 70, 70] = 2.0
    _check((x.transpose(1, 2) @ x).contiguous().to(gpu), rank)


def test_factors_fall_back(gpu):
    """A zero or non-finite matrix is refused by its status, an exactly degenerate one by the
    orthogonality check; low_rank_factors then gives what eigh gives, and what eigh refuses stays refused."""
    _say("eigen fallback")
    n = 128
    for a in (torch.zeros(1, n, n), torch.full((1, n, n), float("nan"))):
        _, _, status = shadowkv.sym_eig_top(a.to(gpu), 8)
        assert status.cpu().tolist() == [0]
    eye = torch.eye(n, device=gpu)[None].contiguous()
    assert not bool(kv._top_eigenpairs(eye, 8)[2])
    assert kv._top_eigenpairs(eye[:, :32, :32].contiguous(), 8) is None  # small: eigh
    u, svt = kv.low_rank_factors(torch.eye(n, device=gpu)[None].to(torch.bfloat16), 8)
    assert (svt @ svt.transpose(1, 2) - torch.eye(8, device=gpu)).abs().max() < 1e-5
    assert torch.isfinite(u).all()
    k = torch.randn(1, 300, n, device=gpu, requires_grad=True)
    u, svt = kv.low_rank_factors(k, 8)
    (u @ svt).sum().backward()
    assert torch.isfinite(k.grad).all()


def test_batches_past_the_xcds(gpu):
    """More problems than one call takes (8) are split."""
    _say("eigen batch 9")
    g = torch.Generator().manual_seed(1)
    k = torch.randn(9, 200, 96, generator=g).to(gpu)
    u, svt = kv.low_rank_factors(k, 20)
    uu, s, vh = torch.linalg.svd(k.cpu().double(), full_matrices=False)
    want = (uu[..., :20] * s[:, None, :20]) @ vh[:, :20]
    got = (u @ svt).cpu().double()
    assert ((got - want).norm(dim=(1, 2)) / want.norm(dim=(1, 2))).max() < 1e-3


def test_concurrent_streams(gpu):
    """Calls of several threads and streams, more than an XCD holds together (two at n = 1024), all give
    the result of a call alone, to the bit."""
    _say("eigen: four streams")
    g = torch.Generator().manual_seed(2)
    x = torch.randn(4, 1200, 1024, generator=g).to(gpu)
    grams = [torch.matmul(k.T.contiguous(), k)[None].contiguous() for k in x]
    want = [shadowkv.sym_eig_top(a, 16) for a in grams]
    torch.cuda.synchronize()
    got = [[] for _ in grams]

    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(5):
                got[i].append(shadowkv.sym_eig_top(grams[i], 16))
        stream.synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i, (w, vt, _) in enumerate(want):
        assert len(got[i]) == 5
        for gw, gvt, status in got[i]:
            assert status.tolist() == [1]
            assert torch.equal(gw, w) and torch.equal(gvt, vt)


def test_captured_call(gpu):
    """Replays of a captured call, one after another with eager calls between them, give the eager result."""
    _say("eigen: captured")
    g = torch.Generator().manual_seed(3)
    x = torch.randn(2, 700, 256, generator=g).to(gpu)
    a = torch.matmul(x.transpose(1, 2).contiguous(), x)
    want = shadowkv.sym_eig_top(a, 20)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with capture_graph(graph, gpu):
        got = shadowkv.sym_eig_top(a, 20)
    for _ in range(3):
        for t in got:
            t.fill_(7)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(u, v) for u, v in zip(got, want))
        assert all(torch.equal(u, v) for u, v in zip(shadowkv.sym_eig_top(a, 20), want))
        torch.cuda.synchronize()


def test_part_of_a_device_takes_eigh(gpu, monkeypatch, request):
    """A device that reports fewer CUs than the XCDs of a whole one have: no attempt, eigh's factors."""
    _say("eigen: part of a device")
    g = torch.Generator().manual_seed(4)
    k = torch.randn(1, 300, 128, generator=g).to(gpu)
    u, svt = kv.low_rank_factors(k, 8)
    monkeypatch.setattr(torch.cuda, "get_device_properties", lambda d: types.SimpleNamespace(multi_processor_count=128))
    shadowkv.sym_eig_runs_on.cache_clear()
    request.addfinalizer(shadowkv.sym_eig_runs_on.cache_clear)
    monkeypatch.setattr(shadowkv, "sym_eig_top", lambda *a: pytest.fail("attempted"))
    assert kv._top_eigenpairs(torch.matmul(k.transpose(1, 2).contiguous(), k), 8) is None
    cfg = types.SimpleNamespace(num_attention_heads=2, num_key_value_heads=1, hidden_size=256, num_hidden_layers=1)
    cache = kv.ShadowKVCache_CPU(cfg, batch_size=1, max_length=300, device=str(gpu), sparse_budget=64, rank=8)
    cache.U = torch.empty(1, device=gpu)
    assert cache._keys_in_place(k.to(torch.bfloat16)) is None  # (their Gram matrix is not made for nothing)
    u2, svt2 = kv.low_rank_factors(k, 8)
    assert ((u2 @ svt2) - (u @ svt)).norm() <= 1e-4 * (u @ svt).norm()
