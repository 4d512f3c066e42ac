"""Which calls of the sublayers (attention, feed-forward, routed experts, lm_head) run on
the HIP kernels: every other call has to reach the torch ops, as the layers' plain source
says it would."""
from __future__ import annotations

import importlib.util
import types

import pytest
import torch
from torch import nn

from model import _ops
from model.model_minimind import (Attention, FeedForward, MiniMindConfig, MOEFeedForward,
                                  precompute_freqs_cis)

BF = torch.bfloat16


def _cfg(**kw):
    return MiniMindConfig(hidden_size=128, num_hidden_layers=1, num_attention_heads=2,
                          num_key_value_heads=1, head_dim=64, intermediate_size=64, vocab_size=64,
                          max_position_embeddings=64, **kw)


def _fake(shape, device="cuda:1"):
    """A tensor of that device with no storage: enough for the rules to look at."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        return torch.empty(shape, device=device, dtype=BF)


def _taken(monkeypatch, device, current):
    """What the rules say to calls that nothing but the device speaks against; with the
    device right, they get as far as the first look at the data."""
    monkeypatch.setattr(_ops, "_current_device", lambda: current)
    monkeypatch.setattr(_ops, "plain_tensors", lambda *a: True)
    attn, moe = Attention(_cfg()).to(BF).eval(), MOEFeedForward(_cfg()).to(BF).eval()
    seen = []

    def library():
        seen.append(1)
        raise RuntimeError("the library")

    monkeypatch.setattr(_ops.H, "load", library)
    monkeypatch.setattr(_ops, "_linear_pays", lambda *a: True)
    lin = nn.Linear(128, 64, bias=False).to(BF)
    q, kv, pos = _fake((1, 4, 128), device), _fake((1, 4, 64), device), _fake((4, 64), device)
    out = [_ops._linear_weights(q, (lin,)) is not None,
           _ops.attn_route(attn, q, kv, kv, (pos, pos), None) is not None]
    for call in (lambda: _ops.linears(q, lin), lambda: _ops.glu(q, lin, lin),
                 lambda: _ops.moe_experts(moe.experts, q[0], _fake((4, 4), device), 1, True)):
        seen.clear()
        try:
            call()
        except RuntimeError:
            pass
        out.append(bool(seen))
    return out


@pytest.mark.parametrize("current,taken", [(1, True), (0, False)])
def test_only_tensors_of_the_current_device(monkeypatch, current, taken):
    """The library launches on the current device: tensors of another one are torch's."""
    with torch.no_grad():
        assert _taken(monkeypatch, "cuda:1", current) == [taken] * 5


@pytest.mark.gpu
def test_another_device_current_runs_torch_ops(dev, monkeypatch):
    torch.manual_seed(0)
    ff, moe, attn = FeedForward(_cfg()), MOEFeedForward(_cfg()), Attention(_cfg())
    x = torch.randn(1, 4, 128, device=dev).to(BF)
    pos = tuple(t.to(dev).to(BF) for t in precompute_freqs_cis(64, 4))
    with torch.no_grad():
        for m in (ff, moe, attn):
            m.to(dev).to(BF).eval()
        want = [ff(x), moe(x), attn(x, pos, None, True)[0]]
        monkeypatch.setattr(_ops, "_current_device", lambda: 1)
        q, k, v = attn.q_proj(x), attn.k_proj(x), attn.v_proj(x)
        assert _ops.linears(x, attn.q_proj) is None and _ops.glu(x, ff.gate_proj, ff.up_proj) is None
        assert _ops.attn_route(attn, q, k, v, pos, None) is None
        assert _ops.moe_experts(moe.experts, x[0], torch.softmax(moe.gate(x[0]), -1), 1, True) is None
        got = [ff(x), moe(x), attn(x, pos, None, True)[0]]
    for w, g in zip(want, got):
        # both round sums and intermediates to bf16 (8 bits): a few half-steps of the largest
        assert float((w.float() - g.float()).abs().max()) <= 6 * 2.0 ** -9 * float(w.float().abs().max())


@pytest.mark.parametrize("grad", [False, True])
def test_feed_forward_traces_with_fx(grad):
    ff, x = FeedForward(_cfg()), torch.randn(2, 3, 128)
    with torch.set_grad_enabled(grad):
        gm = torch.fx.symbolic_trace(ff)
        assert torch.equal(gm(x), ff(x))
    called = {n.target for n in gm.graph.nodes if n.op == "call_module"}
    assert called == {"gate_proj", "up_proj", "down_proj"}


@pytest.mark.parametrize("grad", [False, True])
def test_feed_forward_scripts(grad):
    ff, x = FeedForward(_cfg()), torch.randn(2, 3, 128)
    with torch.set_grad_enabled(grad):
        assert torch.equal(torch.jit.script(ff)(x), ff(x))


def _plain_calls():
    """plain_call as each kind of tracer and transform sees it, without grad mode."""
    from torch.fx.experimental.proxy_tensor import make_fx
    seen = {}

    def ask(name, out=None):
        def call(x):
            seen[name] = _ops.plain_call()
            return x + 1
        return call

    x = torch.randn(3)
    with torch.no_grad():
        ask("eager")(x)
        make_fx(ask("make_fx"))(x)
        torch.vmap(ask("vmap"))(x)
        torch.func.jvp(ask("jvp"), (x,), (x,))
        torch.jit.trace(ask("jit.trace"), (x,), check_trace=False)
        with torch.autograd.forward_ad.dual_level():
            ask("dual level")(x)
        seen["compile"] = torch.compile(_ops.plain_call, fullgraph=True, backend="eager")()
    ask("grad mode")(x)
    return seen


def test_plain_call_under_tracers_and_transforms():
    seen = _plain_calls()
    assert seen.pop("eager") is True
    assert len(seen) == 7 and not any(seen.values()), seen


@pytest.mark.gpu
def test_compiled_sublayers_keep_one_graph(dev):
    """16-bit inference under torch.compile: the torch ops in one graph, as in the source."""
    torch.manual_seed(0)
    ff, attn = FeedForward(_cfg()).to(dev).to(BF).eval(), Attention(_cfg()).to(dev).to(BF).eval()
    x = torch.randn(1, 4, 128, device=dev).to(BF)
    pos = tuple(t.to(dev).to(BF) for t in precompute_freqs_cis(64, 4))
    with torch.no_grad():
        for fn in (ff, lambda t: attn(t, pos, None, True)[0]):
            torch._dynamo.reset()
            got, want = torch.compile(fn, fullgraph=True, backend="eager")(x), fn(x)
            # the compiled call's torch ops round intermediates that the kernels do not
            assert float((want.float() - got.float()).abs().max()) <= 6 * 2.0 ** -9 * float(want.float().abs().max())


def test_plain_call_under_torch_function_modes():
    """A mode that could observe or replace the ops is not a plain call; the default
    device's own mode is one."""
    from torch.overrides import TorchFunctionMode

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with torch.no_grad():
        with Mode():
            assert not _ops.plain_call()
            with torch.device("cpu"):
                assert not _ops.plain_call()
        with torch.device("cpu"):
            assert _ops.plain_call()
        assert _ops.plain_call()


@pytest.mark.gpu
def test_function_mode_sees_the_sublayers_ops(dev):
    from torch.overrides import TorchFunctionMode
    seen = set()

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.add(getattr(func, "__name__", ""))
            return func(*args, **(kwargs or {}))

    x = torch.randn(1, 4, 128, device=dev).to(BF)
    pos = tuple(t.to(dev).to(BF) for t in precompute_freqs_cis(64, 4))
    ff, moe, attn = (m.to(dev).to(BF).eval() for m in (FeedForward(_cfg()), MOEFeedForward(_cfg()), Attention(_cfg())))
    for call, ops in ((lambda: ff(x), {"linear", "silu"}), (lambda: moe(x), {"linear", "silu", "topk"}),
                      (lambda: attn(x, pos), {"linear", "rms_norm", "scaled_dot_product_attention"})):
        seen.clear()
        with torch.no_grad(), Mode():
            call()
        assert ops <= seen, (ops, seen)


def _again(module):
    """A second copy of a module of the package, imported now."""
    spec = importlib.util.spec_from_file_location(module.__name__ + "_again", module.__file__)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


@pytest.mark.parametrize("owner,name", [
    ("torch._C", "_len_torch_dispatch_stack"), ("torch._C", "_len_torch_function_stack"),
    ("torch._C._functorch", "peek_interpreter_stack"),
    ("torch.autograd.forward_ad", "_current_level"),
    ("torch.nn.modules.module", "_global_forward_hooks"),
    ("torch.overrides", "_get_current_function_mode_stack"),
    ("torch.utils._device", "DeviceContext")])
def test_no_call_is_plain_on_a_torch_without_a_name(monkeypatch, owner, name):
    with torch.no_grad():
        assert _again(_ops).plain_call()
        monkeypatch.delattr(f"{owner}.{name}")
        ops = _again(_ops)
        assert not ops.plain_call()


def test_stream_on_a_torch_without_the_raw_handle(monkeypatch):
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d: types.SimpleNamespace(cuda_stream=77))
    assert _again(_ops.H).stream(torch.device("cuda:0")) == 77


def test_decode_past_the_librarys_limit_is_torchs(monkeypatch):
    """mhc_attn_decode_fwd takes up to 2^20 sequences x kv heads and raises past that."""
    monkeypatch.setattr(_ops, "_current_device", lambda: 1)
    monkeypatch.setattr(_ops, "plain_tensors", lambda *a: True)
    attn = Attention(_cfg()).to(BF).eval()
    pos = _fake((1, 64))
    with torch.no_grad():
        for B, want in ((1 << 20, "decode"), ((1 << 20) + 1, None)):
            kv, past = _fake((B, 1, 64)), _fake((B, 7, 1, 64))
            got = _ops.attn_route(attn, _fake((B, 1, 128)), kv, kv, (pos, pos), (past, past))
            assert got == want, B


@pytest.mark.parametrize("n,taken", [(0, False), (2, False), (4, True)])
def test_linear_widths(monkeypatch, n, taken):
    """mhc_linear_fwd takes multiples of four output features, and none of zero."""
    monkeypatch.setattr(_ops, "_current_device", lambda: 1)
    monkeypatch.setattr(_ops, "plain_tensors", lambda *a: True)
    lin = nn.utils.skip_init(nn.Linear, 128, n, bias=False).to(BF)
    with torch.no_grad():
        assert (_ops._linear_weights(_fake((4, 128)), (lin,)) is not None) == taken


PRODUCTS = [
    # (rows, K, outputs, glu), whether the kernels are no slower than the library there
    # 16 x 16 tiles: one a CU, more
    ((64, 768, (768,), False), True), ((64, 6464, (1024,), False), True), ((64, 6496, (1024,), False), False),
    ((64, 2560, (1536,), False), True), ((64, 2592, (1536,), False), False),
    # 64 x 64 tiles: one a CU, more
    ((512, 2048, (2048,), False), True), ((512, 2080, (2048,), False), False),
    ((512, 1024, (2432,), False), True), ((512, 1536, (2432,), False), False),
    # 128 x 64 tiles
    ((512, 768, (6400,), False), True), ((2048, 2048, (768,), False), False),
    # 128 x 128 tiles: one round, two
    ((8192, 512, (1024,), False), True), ((2048, 512, (6400,), False), False),
    ((8192, 768, (2048,), False), False), ((2048, 768, (6400,), False), False),
    # 128 x 192 tiles, 256 x 256 tiles
    ((8192, 768, (768,), False), True), ((8192, 2048, (768,), False), False),
    ((4096, 768, (6400,), False), False),
    # q, k, v
    ((64, 768, (768, 384, 384), False), True), ((8192, 768, (768, 384, 384), False), True),
    ((16384, 768, (768, 384, 384), False), True), ((65536, 768, (768, 384, 384), False), False),
    ((16384, 1024, (1024, 1024, 1024), False), False), ((8192, 2048, (2048, 512, 512), False), False),
    ((2051, 1984, (2688, 2688, 2688), False), False), ((2930, 3296, (2496, 2496, 2496), False), False), ((4225, 768, (768, 384, 384), False), True),
    ((300, 4096, (4096, 1024, 1024), False), True), ((3000, 4096, (4096, 1024, 1024), False), False),
    # gate and up
    ((64, 768, (2048, 2048), True), True), ((8192, 768, (2432, 2432), True), True),
    ((8192, 2048, (6464, 6464), True), True), ((3000, 2048, (4096, 4096), True), False),
    ((1024, 4096, (12928, 12928), True), False)]


@pytest.mark.parametrize("size,pays", PRODUCTS)
def test_products_go_where_they_are_faster(monkeypatch, size, pays):
    M, K, ns, glu = size
    calls, lib = [], _ops.H.load()

    class Lib:
        mhc_linear_pays = lib.mhc_linear_pays if hasattr(lib, "mhc_linear_pays") else None

        def __getattr__(self, name):
            calls.append(name)
            raise RuntimeError(name)

    class Layer(nn.Linear):  # what plain_module is told is an nn.Linear; the library's call
        def __init__(self, n):
            super().__init__(32, 4, bias=False, dtype=BF)
            self.out_features = n
            self.weight = nn.Parameter(_fake((n, K)), requires_grad=False)

        def forward(self, x):
            calls.append("torch")
            return None

    monkeypatch.setattr(_ops, "_current_device", lambda: 1)
    monkeypatch.setattr(_ops, "plain_tensors", lambda *a: True)
    monkeypatch.setattr(_ops, "plain_module", lambda *a: True)
    monkeypatch.setattr(_ops.H, "load", lambda: Lib())
    monkeypatch.setattr(_ops.H, "stream", lambda dev: 0)
    monkeypatch.setattr(_ops.H, "dtype_tag", lambda t: 1)
    x, mods = _fake((M, K)), [Layer(n) for n in ns]
    with torch.no_grad():
        try:
            if glu:
                taken = _ops.glu(x, *mods) is not None
            else:
                taken = (_ops.linear(x, mods[0]) if len(ns) == 1 else _ops.linears(x, *mods)) is not None
        except RuntimeError:
            taken = True
    assert taken == pays and (not calls or calls == ["torch"] or pays), (taken, calls)


@pytest.mark.parametrize("tokens,hidden,inter,experts,topk,taken", [
    (8192, 4096, 14336, 4, 1, False), (8188, 4096, 14336, 4, 1, True), (8192, 4096, 8192, 4, 1, True),
    (8192, 8192, 8192, 4, 1, False), (1, 8192, 8192, 4, 1, True), (65536, 2048, 6464, 4, 2, True)])
def test_experts_go_where_they_are_faster(monkeypatch, tokens, hidden, inter, experts, topk, taken):
    """Wide experts with many rows each: the library's products, in the loop."""
    def proj(n, k):
        return types.SimpleNamespace(out_features=n, in_features=k, bias=None, weight=_fake((n, k)))

    def library():
        raise RuntimeError("the library")

    monkeypatch.setattr(_ops, "_current_device", lambda: 1)
    monkeypatch.setattr(_ops, "plain_tensors", lambda *a: True)
    monkeypatch.setattr(_ops, "plain_module", lambda *a: True)
    monkeypatch.setattr(_ops.H, "load", library)
    mods = [types.SimpleNamespace(gate_proj=proj(inter, hidden), up_proj=proj(inter, hidden),
                                  down_proj=proj(hidden, inter)) for _ in range(experts)]
    with torch.no_grad():
        try:
            got = _ops.moe_experts(mods, _fake((tokens, hidden)), _fake((tokens, experts)), topk, True) is not None
        except RuntimeError:
            got = True
    assert got == taken


@pytest.mark.gpu
def test_experts_without_room_for_all_rows_loop(dev, monkeypatch):
    """The kernels hold every expert's rows at once: where that does not fit, the loop
    over the experts, which needs less, runs as it did."""
    torch.manual_seed(0)
    moe, x = MOEFeedForward(_cfg()).to(dev).to(BF).eval(), torch.randn(1, 40, 128, device=dev).to(BF)
    empty = torch.empty

    def full(*args, **kwargs):
        if kwargs.get("dtype") is torch.uint8:
            raise torch.OutOfMemoryError("no room")
        return empty(*args, **kwargs)

    with torch.no_grad():
        want = moe(x)
        monkeypatch.setattr(torch, "empty", full)
        got = moe(x)
    assert float(moe.aux_loss) == 0
    assert float((want.float() - got.float()).abs().max()) <= 6 * 2.0 ** -9 * float(want.float().abs().max())
