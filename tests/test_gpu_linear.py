"""The sublayers' linear kernels against float64 products of the same 16-bit values,
at the edges of their tiles and on both sides of every line of the dispatch; and the
calls that stay with torch."""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F
from torch import nn

from model import _ops

pytestmark = pytest.mark.gpu
BF, F16 = torch.bfloat16, torch.float16


def _linears(K, Ns, dt, dev):
    torch.manual_seed(K + sum(Ns))
    return [nn.Linear(K, n, bias=False).to(dev).to(dt) for n in Ns]


def _close(want, got, dt):
    # one rounding of each output: half a last place is at most 2^-8 of the value at bf16's
    # 8 significant bits, 2^-11 at fp16's 11; fp32 sums of up to 2048 products, whose terms
    # are some sqrt(2048) times the sum, add under 2^-13 of the largest output
    assert torch.isfinite(got).all()
    err = (want - got.double()).abs()
    bound = 2.0 ** -(8 if dt == BF else 11) * want.abs() + 2.0 ** -13 * float(want.abs().max())
    assert bool((err <= bound).all())


@pytest.mark.parametrize("K,Ns,M,dt", [
    # 16 x 16 tiles: one row, ragged rows, ragged columns, both wave counts, the last count
    (32, (4,), 1, BF), (768, (768, 384, 384), 64, BF), (768, (20, 36, 4), 17, F16),
    (2048, (768,), 128, BF), (1536, (100,), 5, BF), (1568, (64,), 33, F16), (96, (112,), 1024, BF),
    # 64 x 64 tiles: just past the count, ragged both ways, K of 64 and of 32
    (768, (768, 384, 384), 75, BF), (64, (1536,), 1025, BF), (160, (516, 68), 300, BF),
    (32, (4096,), 63, F16), (768, (6400,), 65, BF), (2048, (768,), 700, BF),
    # 128 x 64 tiles: the first count, ragged, K of 64 and of 32
    (64, (2048,), 768, BF), (160, (516, 68), 2200, F16), (2048, (768,), 2050, BF),
    # 128 x 128 tiles: one and two slices of K, ragged
    (64, (2048,), 2176, BF), (128, (1540, 260), 2100, F16), (96, (1024, 512), 3001, BF),
    # 128 x 192 tiles: the first count, ragged rows, columns and K
    (64, (768,), 8192, BF), (160, (764, 380), 5400, F16), (768, (768, 384, 384), 4225, BF),
    # 256 x 256 tiles: nearly full rounds, ragged rows, columns and K
    (96, (6396,), 4001, BF), (64, (4096, 2048, 260), 3900, F16)])
def test_products(dev, K, Ns, M, dt):
    mods = _linears(K, Ns, dt, dev)
    x = torch.randn(M, K, device=dev).to(dt)
    with torch.inference_mode():
        outs = _ops.linears(x, *mods)
        assert outs is not None
        for m, o in zip(mods, outs):
            _close(x.double() @ m.weight.double().t(), o, dt)


@pytest.mark.parametrize("K,N,M,dt", [
    (768, 2048, 1, BF), (768, 2048, 48, BF), (768, 2048, 64, BF), (2048, 20, 30, F16), (32, 36, 7, BF),
    (96, 1100, 130, BF), (64, 4100, 600, BF), (768, 2048, 515, F16), (128, 2432, 1111, BF),
    (96, 2052, 1100, BF), (32, 4100, 1500, F16), (64, 4100, 3500, BF), (160, 2048, 7300, F16)])
def test_glu(dev, K, N, M, dt):
    gate, up = _linears(K, (N, N), dt, dev)
    x = torch.randn(1, M, K, device=dev).to(dt)
    with torch.inference_mode():
        got = _ops.glu(x, gate, up)
    z = x.double() @ gate.weight.double().t()
    # silu's exponential and quotient add a few fp32 ulps
    _close(F.silu(z) * (x.double() @ up.weight.double().t()), got, dt)


def test_infinite_and_extreme_inputs(dev):
    """Values past the others' rows stay in their row; silu of large inputs is finite."""
    gate, up = _linears(64, (64, 64), BF, dev)
    x = torch.randn(40, 64, device=dev).to(BF)
    x[3, 5] = float("inf")
    x[7] = float("nan")
    x[9] *= 3000
    with torch.inference_mode():
        got, want = _ops.glu(x, gate, up).float(), F.silu(gate(x).float()) * up(x).float()
        out, = _ops.linears(x, up)
        ref = up(x)
    assert torch.equal(torch.isnan(out), torch.isnan(ref)) and torch.equal(torch.isinf(out), torch.isinf(ref))
    rows = torch.tensor([r for r in range(40) if r not in (3, 7)], device=dev)
    assert torch.isfinite(got[rows]).all()
    assert float((got - want)[rows].abs().max()) <= 0.02 * float(want[rows].abs().max())


def test_calls_left_to_torch(dev):
    a, b, c = _linears(64, (64, 64, 32), BF, dev)
    x = torch.randn(4, 6, 64, device=dev).to(BF)
    assert _ops.linears(x, a) is None  # grad mode
    with torch.no_grad():
        assert _ops.linears(x, a, b, c)[2].shape == (4, 6, 32)
        assert _ops.linears(x.transpose(0, 1), a) is None
        assert _ops.linears(x[:, :0], a) is None
        assert _ops.linears(x.float(), a) is None
        assert _ops.linears(x.cpu(), a) is None
        assert _ops.glu(x, a, c) is None
        assert _ops.linears(x, nn.Linear(64, 64).to(dev).to(BF)) is None  # a bias
        assert _ops.linears(x[..., :48].contiguous(), *_linears(48, (64,), BF, dev)) is None
        old = b.forward
        b.forward = lambda t: old(t) + 1
        assert _ops.linears(x, a, b) is None and _ops.glu(x, a, b) is None
        assert torch.equal(_ops.linear(x, b), old(x) + 1)
        del b.forward
        with torch.amp.autocast("cuda", dtype=BF):
            assert _ops.linears(x, a) is None
        big = torch.empty(6000, 768, device=dev, dtype=BF)
        assert _ops.linears(big, *_linears(768, (4096,), BF, dev)) is None  # faster in the library
