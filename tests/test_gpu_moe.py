"""The routed-expert layer's inference kernels against the layer's own loop over
experts in float64 on the CPU (model/model_minimind.py:270-298), with the experts
of each token as the 16-bit router picks them; at the edges of the kernels' tiles,
for empty experts and equal probabilities; and calls left to the torch loop."""
from __future__ import annotations

import copy

import pytest
import torch
import torch.nn.functional as F

from model import _ops
from model.model_minimind import FeedForward, MiniMindConfig, MOEFeedForward

pytestmark = pytest.mark.gpu
BF, F16 = torch.bfloat16, torch.float16


def _layer(D, inter, experts, topk, dtype, norm=True):
    torch.manual_seed(D + inter + experts)
    cfg = MiniMindConfig(hidden_size=D, use_moe=True, num_experts=experts, norm_topk_prob=norm,
                         num_experts_per_tok=topk, moe_intermediate_size=inter)
    m = MOEFeedForward(cfg).eval()
    with torch.no_grad():
        for p in m.parameters():
            p.normal_(0.0, 0.06)
    return m.to(dtype)


def _want(m, x, probs):
    """The layer in float64, the picks from the 16-bit probabilities."""
    m, x = copy.deepcopy(m).double().cpu(), x.double().cpu()
    w, at = torch.sort(probs.double().cpu(), dim=-1, descending=True, stable=True)
    k = m.config.num_experts_per_tok
    w, at = w[:, :k], at[:, :k]
    if m.config.norm_topk_prob:
        w = w / w.sum(-1, keepdim=True)
    y = torch.zeros_like(x)
    with torch.no_grad():
        for e, expert in enumerate(m.experts):
            y += (w * (at == e)).sum(-1, keepdim=True) * expert(x)
    return y


def _check(m, x, probs):
    with torch.inference_mode():
        got = _ops.moe_experts(m.experts, x, probs, m.config.num_experts_per_tok,
                               m.config.norm_topk_prob)
    want = _want(m, x, probs)
    got = got.double().cpu()
    assert torch.isfinite(got).all()
    # the hidden row, each expert's row, the weights and the sum are rounded to the type
    bar = 5 * 2.0 ** -(9 if x.dtype == BF else 12)
    assert float((got - want).abs().max()) <= bar * float(want.abs().max())


@pytest.mark.parametrize("D,inter,experts,topk,dtype,M", [
    (768, 1024, 8, 2, BF, 300), (768, 1024, 8, 2, BF, 1), (512, 512, 4, 1, BF, 129),
    (32, 32, 2, 2, BF, 127), (64, 96, 8, 3, BF, 128), (1024, 160, 4, 2, F16, 257),
    (288, 416, 32, 8, BF, 64), (768, 768, 1, 1, F16, 200), (96, 1056, 5, 2, BF, 1025),
    (768, 64, 8, 2, BF, 4100), (32, 2048, 8, 2, BF, 3200), (6400, 32, 4, 2, F16, 2048)])
def test_experts(dev, D, inter, experts, topk, dtype, M):
    m = _layer(D, inter, experts, topk, dtype, norm=M != 129).to(dev)
    x = torch.randn(M, D, device=dev).to(dtype)
    with torch.no_grad():
        probs = F.softmax(m.gate(x), -1)
    _check(m, x, probs)
    with torch.inference_mode():  # the layer takes them
        y = m(x.view(1, M, D))
    assert torch.equal(y.view(M, D), _ops_call(m, x, probs)) and float(m.aux_loss) == 0.0


def _ops_call(m, x, probs):
    with torch.inference_mode():
        return _ops.moe_experts(m.experts, x, probs, m.config.num_experts_per_tok,
                                m.config.norm_topk_prob)


def test_empty_experts_and_ties(dev):
    m = _layer(64, 64, 8, 2, BF).to(dev)
    x = torch.randn(400, 64, device=dev).to(BF)
    probs = torch.zeros(400, 8, device=dev, dtype=BF)
    probs[:, 3], probs[:, 6] = 0.75, 0.25      # six experts without a row
    _check(m, x, probs)
    probs = torch.full((400, 8), 0.125, device=dev, dtype=BF)  # all equal: the first two
    _check(m, x, probs)
    probs[::2, 5] = 0.5
    _check(m, x, probs)
    # the picks are torch.topk's, where equal values compete too
    g = torch.Generator().manual_seed(1)
    probs = (torch.randint(1, 5, (4000, 8), generator=g) / 16).to(BF).to(dev)
    x = torch.randn(4000, 64, device=dev).to(BF)
    fast = _ops_call(m, x, probs).float()
    w, at = torch.topk(probs, 2, -1, sorted=False)
    w = (w / (w.sum(-1, keepdim=True) + 1e-20)).float()
    with torch.no_grad():
        rows = torch.stack([e(x).float() for e in m.experts], 1)
    slow = (w.unsqueeze(-1) * rows.gather(1, at.unsqueeze(-1).expand(-1, -1, 64))).sum(1)
    assert float((fast - slow).abs().max()) <= 0.02 * float(slow.abs().max())


def test_nan_token_stays_its_own(dev):
    m = _layer(64, 64, 4, 2, BF).to(dev)
    x = torch.randn(130, 64, device=dev).to(BF)
    with torch.inference_mode():
        clean = m(x.view(1, 130, 64)).view(130, 64)
        x[77, 5] = float("nan")
        got = m(x.view(1, 130, 64)).view(130, 64)
    assert torch.isnan(got[77]).all()
    rest = torch.arange(130, device=dev) != 77
    assert torch.equal(got[rest], clean[rest])


def test_replay_in_a_graph(dev):
    m = _layer(128, 128, 8, 2, BF).to(dev)
    x = torch.randn(1, 300, 128, device=dev).to(BF)
    with torch.inference_mode():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            m(x)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = m(x)
        for i in range(3):
            x.copy_(torch.randn(1, 300, 128, device=dev))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, m(x)), i


def test_other_experts_keep_their_own_forward(dev):
    class Doubled(FeedForward):
        def forward(self, x):
            return 2 * super().forward(x)

    m = _layer(64, 64, 4, 2, BF).to(dev)
    twice = copy.deepcopy(m)
    for e in twice.experts:
        e.__class__ = Doubled
    x = torch.randn(1, 40, 64, device=dev).to(BF)
    with torch.inference_mode():
        want, got = 2 * m(x).float(), twice(x).float()
    assert float((got - want).abs().max()) <= 0.02 * float(want.abs().max())


def test_calls_left_to_the_loop(dev):
    m = _layer(64, 64, 4, 2, BF).to(dev)
    x = torch.randn(10, 64, device=dev).to(BF)
    with torch.no_grad():
        probs = F.softmax(m.gate(x), -1)
        take = lambda mm=m, xx=x, p=probs, k=2: _ops.moe_experts(mm.experts, xx, p, k, True)  # noqa: E731
        assert take() is not None
        assert take(xx=x[:0], p=probs[:0]) is None
        assert take(xx=torch.randn(10, 128, device=dev).to(BF)[:, ::2]) is None
        h = m.experts[1].register_forward_hook(lambda *a: None)
        assert take() is None
        h.remove()
        old = m.experts[2].up_proj.forward
        m.experts[2].up_proj.forward = lambda t: old(t) * 2
        assert take() is None
        del m.experts[2].up_proj.forward
        assert take(mm=copy.deepcopy(m).float(), xx=x.float(), p=probs.float()) is None
        odd = _layer(64, 48, 4, 2, BF).to(dev)
        assert take(mm=odd) is None and odd(x.view(1, 10, 64)).shape == (1, 10, 64)
    assert take() is None  # grad mode
