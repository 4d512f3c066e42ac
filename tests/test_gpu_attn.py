"""The attention layer's inference kernels (norm + rotary, causal prefill, one
decode step over a KV cache) against the same layer's torch ops in float64 on
the CPU (model/model_minimind.py:161-256), at the edges of their tiles; and the
rule that chooses them against calls it must leave to torch."""
from __future__ import annotations

import copy

import pytest
import torch

from model import _ops
from model.model_minimind import Attention, MiniMindConfig, precompute_freqs_cis

BF, F16 = torch.bfloat16, torch.float16


def _layer(hd, heads, kv, dtype, seed=0):
    torch.manual_seed(seed)
    cfg = MiniMindConfig(hidden_size=128, num_attention_heads=heads, num_key_value_heads=kv,
                         head_dim=hd, max_position_embeddings=4096)
    m = Attention(cfg).eval()
    with torch.no_grad():
        for p in m.parameters():
            if p.dim() == 1:
                p.add_(torch.randn(p.shape) * 0.3)
            else:
                p.normal_(0.0, 0.15)  # scores of several units: a peaked softmax
    return m.to(dtype)


def _pos(hd, start, T, dtype):
    cos, sin = precompute_freqs_cis(hd, start + T)
    return cos[start:].to(dtype), sin[start:].to(dtype)


def _wide(m, x, pos, past, use_cache):
    ref = copy.deepcopy(m).double()
    up = lambda t: t.double().cpu()  # noqa: E731
    with torch.no_grad():
        return ref(up(x), tuple(map(up, pos)), None if past is None else tuple(map(up, past)),
                   use_cache)


def _bar(dtype):
    # q, k, v, the probabilities and the output are each rounded to the type once, and so
    # are the projections' inputs to o_proj: six half-steps of it, at the largest element
    return 6 * 2.0 ** -(9 if dtype == BF else 12)


def _close(want, got, bar):
    want, got = want.float().cpu(), got.float().cpu()
    assert torch.isfinite(got).all()
    assert float((want - got).abs().max()) <= bar * float(want.abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("hd,heads,kv,dtype,B,T", [
    (96, 8, 4, BF, 2, 1), (96, 8, 4, BF, 1, 63), (96, 8, 4, BF, 1, 64), (96, 8, 4, BF, 3, 65),
    (64, 4, 4, BF, 2, 127), (64, 3, 1, F16, 1, 129), (128, 8, 2, BF, 1, 257), (128, 4, 1, F16, 2, 96),
    (96, 6, 2, BF, 1, 200), (96, 8, 4, F16, 2, 333),
    # more workgroups than the 256 CUs: a part-filled second round (which runs backwards)
    # and a third one, of paired heads and of single ones
    (96, 8, 4, BF, 5, 1000), (64, 8, 2, BF, 16, 520), (64, 8, 8, BF, 6, 700), (64, 6, 2, F16, 16, 700)])
def test_prefill(dev, hd, heads, kv, dtype, B, T):
    m = _layer(hd, heads, kv, dtype)
    x, pos = torch.randn(B, T, 128).to(dtype), _pos(hd, 0, T, dtype)
    want, (wk, wv) = _wide(m, x, pos, None, True)
    m, x, pos = m.to(dev), x.to(dev), tuple(t.to(dev) for t in pos)
    with torch.inference_mode():
        assert _ops.attn_route(m, m.q_proj(x), m.k_proj(x), m.v_proj(x), pos, None) == "prefill"
        got, (gk, gv) = m(x, pos, None, True)
    assert got.shape == want.shape and gk.shape == wk.shape and gv.shape == wv.shape
    _close(want, got, _bar(dtype))
    _close(wk, gk, _bar(dtype))
    _close(wv, gv, _bar(dtype))


@pytest.mark.gpu
@pytest.mark.parametrize("hd,heads,kv,dtype,B,S,cache", [
    (96, 8, 4, BF, 1, 1, True), (96, 8, 4, BF, 3, 15, True), (96, 8, 4, BF, 2, 16, False),
    (64, 4, 4, BF, 2, 17, True), (128, 8, 2, BF, 1, 1000, True), (64, 3, 1, F16, 5, 47, True),
    (96, 8, 4, F16, 64, 130, True), (128, 4, 1, F16, 1, 333, False), (96, 6, 2, BF, 300, 33, True),
    (64, 6, 6, BF, 2, 95, True), (96, 3, 3, BF, 1, 129, True),
    # more than 64 partial results a head
    (96, 8, 4, BF, 1, 4000, True), (64, 3, 1, F16, 1, 2050, False)])
def test_decode(dev, hd, heads, kv, dtype, B, S, cache):
    m = _layer(hd, heads, kv, dtype)
    x, pos = torch.randn(B, 1, 128).to(dtype), _pos(hd, S, 1, dtype)
    past = tuple(torch.randn(B, S, kv, hd).mul_(1.5).to(dtype) for _ in range(2))
    want, grown = _wide(m, x, pos, past, True)
    md, xd, pd = m.to(dev), x.to(dev), tuple(t.to(dev) for t in pos)
    # the cache as a view with other strides than its own size gives
    roomy = tuple(torch.randn(B, S + 5, kv + 1, hd, dtype=dtype, device=dev) for _ in range(2))
    for r, p in zip(roomy, past):
        r[:, 2:2 + S, :kv] = p.to(dev)
    views = tuple(r[:, 2:2 + S, :kv] for r in roomy)
    for cached in (tuple(p.to(dev) for p in past), views):
        with torch.inference_mode():
            assert _ops.attn_route(md, md.q_proj(xd), md.k_proj(xd), md.v_proj(xd), pd,
                                   cached) == "decode"
            got, kvs = md(xd, pd, cached, cache)
        _close(want, got, _bar(dtype))
        assert (kvs is not None) == cache
        if cache:
            for g, w, p in zip(kvs, grown, past):
                assert g.is_contiguous() and torch.equal(g[:, :S].cpu(), p)
                _close(w[:, S:], g[:, S:], _bar(dtype))


@pytest.mark.gpu
def test_decode_rising_scores(dev):
    """Scores that keep rising along the cache (each range and each lane raises
    its maximum many times), and rows whose largest score comes first."""
    hd, heads, kv, S = 96, 8, 4, 400
    m = _layer(hd, heads, kv, BF)
    x, pos = torch.randn(2, 1, 128).to(BF), _pos(hd, S, 1, BF)
    for ramp in (torch.linspace(0, 40, S), torch.linspace(40, 0, S)):
        past = tuple(torch.randn(2, S, kv, hd) for _ in range(2))
        past = ((past[0] * ramp.view(1, S, 1, 1)).to(BF), past[1].to(BF))
        want, _ = _wide(m, x, pos, past, True)
        md = copy.deepcopy(m).to(dev)
        with torch.inference_mode():
            got, _ = md(x.to(dev), tuple(t.to(dev) for t in pos), tuple(t.to(dev) for t in past), True)
        _close(want, got, 2 * _bar(BF))  # scores of 100: q's rounding moves them by up to half a unit


@pytest.mark.gpu
@pytest.mark.parametrize("hd,heads,kv,dtype,S", [
    (96, 8, 4, F16, 1), (96, 8, 4, BF, 15), (64, 4, 2, F16, 37), (128, 3, 3, BF, 70),
    (64, 4, 1, F16, 1000), (96, 8, 4, BF, 2001)])
def test_decode_infinite_value(dev, hd, heads, kv, dtype, S):
    """One infinite element of a V row (the newest position's, or the cache's last, whose
    row the kernel also reads for the rows that are not there) makes its column infinite
    and changes no other."""
    m = _layer(hd, heads, kv, dtype).to(dev)
    pos = tuple(t.to(dev) for t in _pos(hd, S, 1, dtype))
    q, k, v = (torch.randn(2, 1, n * hd, device=dev).to(dtype) for n in (heads, kv, kv))
    past = tuple(torch.randn(2, S, kv, hd, device=dev).to(dtype) for _ in range(2))
    with torch.inference_mode():
        want, _ = _ops.attn_decode(m, q, k, v, pos, past, False)
        for cached in (False, True):
            v2, pv = v.clone(), past[1].clone()
            row = pv[1, S - 1, kv - 1] if cached else v2[1, 0].view(kv, hd)[kv - 1]
            row[5] = float("inf")
            got, _ = _ops.attn_decode(m, q, k, v2, pos, (past[0], pv), False)
            hit = torch.zeros(2, heads, hd, dtype=torch.bool, device=dev)
            hit[1, heads - heads // kv:, 5] = True
            hit = hit.view(got.shape)
            assert bool((got[hit] == float("inf")).all())
            assert torch.equal(got[~hit], want[~hit]) and bool(torch.isfinite(want).all())


@pytest.mark.gpu
@pytest.mark.parametrize("hd,heads,kv,dtype,T", [
    (96, 8, 4, F16, 1), (96, 8, 4, BF, 100), (64, 3, 1, F16, 129), (128, 4, 4, BF, 190), (64, 4, 2, F16, 64)])
def test_prefill_infinite_value(dev, hd, heads, kv, dtype, T):
    """One infinite element of the last position's V row makes the last row's column
    infinite (rows that are not there are read as copies of it); the other columns, and
    the rows of the tiles before, are as without it."""
    m = _layer(hd, heads, kv, dtype).to(dev)
    pos = tuple(t.to(dev) for t in _pos(hd, 0, T, dtype))
    q, k, v = (torch.randn(2, T, n * hd, device=dev).to(dtype) for n in (heads, kv, kv))
    with torch.inference_mode():
        want = _ops.attn_prefill(m, q, k, v, pos)[0].view(2, T, heads, hd)
        v2 = v.clone()
        v2[1, T - 1].view(kv, hd)[kv - 1, 5] = float("inf")
        got = _ops.attn_prefill(m, q, k, v2, pos)[0].view(2, T, heads, hd)
    hit = torch.zeros_like(want, dtype=torch.bool)
    hit[1, (T - 1) // 64 * 64:, heads - heads // kv:, 5] = True  # the tile that holds the position
    assert bool((got[1, T - 1, heads - heads // kv:, 5] == float("inf")).all())
    assert torch.equal(got[~hit], want[~hit]) and bool(torch.isfinite(want).all())


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["q_norm", "k_norm"])
def test_norm_without_eps(dev, name):
    """nn.RMSNorm(eps=None) takes an epsilon of torch's choosing (2^-23 for bf16 input,
    not bf16's own 2^-7): inputs small enough to tell give what torch's ops give."""
    m = _layer(96, 8, 4, BF).to(dev)
    getattr(m, name).eps = None
    with torch.no_grad():
        getattr(m, name[0] + "_proj").weight.mul_(0.01)
        for T, past in ((70, None), (1, tuple(torch.randn(2, 9, 4, 96, device=dev).to(BF) for _ in range(2)))):
            x = torch.randn(2, T, 128, device=dev).to(BF)
            pos = tuple(t.to(dev) for t in _pos(96, 9 if past else 0, T, BF))
            got = m(x, pos, past, True)
            with torch.amp.autocast("cuda", enabled=True, dtype=BF):  # not the kernels' call
                want = m(x, pos, past, True)
            _close(want[0], got[0], _bar(BF))
            _close(want[1][0], got[1][0], _bar(BF))


@pytest.mark.gpu
def test_calls_left_to_torch(dev):
    """Calls the kernels do not take, or that would tell: the route is None."""
    m = _layer(96, 8, 4, BF).to(dev)
    x = torch.randn(2, 8, 128, device=dev, dtype=BF)
    pos = tuple(t.to(dev) for t in _pos(96, 0, 8, BF))

    def route(mm=m, xx=x, p=pos, past=None):
        return _ops.attn_route(mm, mm.q_proj(xx), mm.k_proj(xx), mm.v_proj(xx), p, past)

    assert route() is None  # grad mode
    with torch.no_grad():
        assert route() == "prefill"
        assert route(p=tuple(t.float() for t in pos)) is None
        assert route(p=tuple(t[:4] for t in pos)) is None
        past = tuple(torch.randn(2, 5, 4, 96, device=dev, dtype=BF) for _ in range(2))
        assert route(past=past) is None  # 8 new positions over a cache
        one = tuple(t[:1] for t in pos)
        assert route(xx=x[:, :1], p=one, past=past) == "decode"
        assert route(xx=x[:, :1], p=one, past=tuple(t.float() for t in past)) is None
        assert route(xx=x[:, :1], p=one, past=tuple(t[:, :0] for t in past)) is None
        assert route(xx=x[:, :1], p=one, past=(past[0], past[1][:, :4])) is None
        with torch.amp.autocast("cuda", dtype=BF):
            assert route() is None
        handle = m.q_norm.register_forward_hook(lambda *a: None)
        assert route() is None
        handle.remove()
        m.is_causal = False
        assert route() is None
        m.is_causal = True
        m.train()
        assert route() == "prefill"
        m.dropout = 0.1
        assert route() is None
        m.eval()
        with torch.autograd.forward_ad.dual_level():
            assert route() is None
        assert route(mm=copy.deepcopy(m).float(), xx=x.float()) is None


def test_cpu_calls_take_the_torch_ops():
    m = _layer(96, 8, 4, BF)
    x = torch.randn(1, 4, 128).to(BF)
    with torch.no_grad():
        assert _ops.attn_route(m, m.q_proj(x), m.k_proj(x), m.v_proj(x), _pos(96, 0, 4, BF), None) is None
        assert m(x, _pos(96, 0, 4, BF))[0].shape == (1, 4, 128)
