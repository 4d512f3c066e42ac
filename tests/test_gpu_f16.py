"""fp16 streams on the K-streamed MFMA pre kernel: every output against the fp32
oracle and against the VALU kernel that served fp16 before (no image), at the
edges of its tiles and chunks; and the C ABI's image flag."""
from __future__ import annotations

import pytest
import torch

from oracle import mhc_ref as R
from tests._util import make_params, maxrel, tol

pytestmark = pytest.mark.gpu

from model import _hip as H  # noqa: E402
from model import _ops  # noqa: E402
from model.mhc_common import MHCHead  # noqa: E402
from model.mhc_fused import MHCConnection_Fused  # noqa: E402

F16 = torch.float16
MODES = {"full": H.MODE_FULL, "nohres": H.MODE_NOHRES, "head": H.MODE_HEAD}


def _run(kind, x, p, packed, n, C, iters, norm):
    d = p["phi_weight"].device
    kw = dict(want_saved=True, norm=None if norm is None else (norm, 1e-6))
    if kind == "full":
        return _ops.pre_full(x, p["phi_weight"], packed, p["alpha_pre"], p["bias_pre"],
                             p["alpha_post"], p["bias_post"], p["alpha_res"], p["bias_res"], n, C,
                             2.0, 1e-6, 1e-6, iters, 1e-6, want_h_pre=True, want_raw=True, **kw)
    if kind == "nohres":
        return _ops.pre_nohres(x, p["phi_weight"], packed, p["alpha_pre"], p["bias_pre"],
                               p["alpha_post"], p["bias_post"], n, C, 2.0, 1e-6, 1e-6,
                               want_h_pre=True, **kw)
    out, inv, mix = _ops.head(x, p["phi_weight"], packed, p["alpha"], p["bias"], n, C, 1e-6, 1e-6, **kw)
    return {"sub_in": out, "inv_rms": inv, "mixes_raw": mix}


@pytest.mark.parametrize("kind,n,C,M,iters,norm", [
    ("full", 4, 768, 1, 20, True), ("full", 4, 768, 33, 10, False), ("full", 4, 768, 1000, 10, True),
    ("full", 8, 768, 31, 20, True), ("full", 8, 200, 65, 1, False), ("full", 2, 64, 32, 10, True),
    ("full", 2, 40, 70, 10, False), ("full", 4, 8, 5, 3, True), ("full", 16, 96, 17, 10, True),
    ("full", 4, 1032, 40, 10, True), ("full", 2, 1536, 9, 10, False),
    ("nohres", 4, 768, 47, 0, True), ("nohres", 8, 72, 64, 0, False), ("nohres", 2, 512, 3, 0, True),
    ("head", 4, 768, 90, 0, True), ("head", 8, 136, 33, 0, False), ("head", 2, 64, 1, 0, True)])
def test_matches_oracle_and_valu_kernel(dev, kind, n, C, M, iters, norm):
    g = torch.Generator().manual_seed(n * C + M)
    x = torch.randn(1, M, n * C, generator=g).to(F16)
    p = make_params(kind, n, C, F16, g)
    w = (1.0 + 0.5 * torch.randn(C, generator=g)).to(F16) if norm else None
    pd, xd = {k: v.to(dev) for k, v in p.items()}, x.to(dev)
    wd = None if w is None else w.to(dev)
    packed = _ops.packed_phi(pd["phi_weight"], n, C, MODES[kind])
    assert packed is not None
    fast = _run(kind, xd, pd, packed, n, C, iters, wd)
    slow = _run(kind, xd, pd, None, n, C, iters, wd)
    for k, v in fast.items():
        if v is not None:
            # the sums run in another order: a gate may round to the other neighbour, and
            # what it multiplies with it
            bar = 1e-5 if v.dtype == torch.float32 and k == "inv_rms" else tol(F16)
            assert maxrel(slow[k], v) <= bar, k
    pf, xf = {k: v.float() for k, v in p.items()}, x.float()
    if kind == "full":
        sub, h_pre, h_post, raw, inv, mixes = R.pre_full(xf, pf, n, C)
        want = {"h_pre": h_pre, "h_post": h_post, "h_res_raw": raw, "mixes_raw": mixes,
                "h_res": R.sinkhorn(raw, max(iters, 1), 1e-6)}
    elif kind == "nohres":
        sub, h_pre, h_post, inv, mixes = R.pre_nohres(xf, pf, n, C)
        want = {"h_pre": h_pre, "h_post": h_post, "mixes_raw": mixes}
    else:
        sub, want = R.head(xf, pf, n, C), {}
    if norm:
        sub = torch.nn.functional.rms_norm(sub, (C,), w.float(), 1e-6)
    want["sub_in"] = sub
    for k, v in want.items():
        assert maxrel(v.reshape(fast[k].shape), fast[k]) <= 2 * tol(F16), k


def test_modules_take_the_image_and_train_through(dev):
    """A module's forward equals the Functions' outputs with the image, and its
    gradients still flow."""
    torch.manual_seed(3)
    m = MHCConnection_Fused(4, 64).to(dev).to(F16)
    head = MHCHead(4, 64).to(dev).to(F16)
    x = torch.randn(2, 19, 256, device=dev).to(F16).requires_grad_()
    head(m(x, lambda z: z)).float().sum().backward()
    assert torch.isfinite(x.grad).all() and m._phi_pack.get(m.phi_weight.detach(), 4, 64) is not None


def test_without_the_flag_the_image_is_ignored(dev):
    """phi_packed beside a plain fp16 phi tag is not read (it was not before)."""
    g = torch.Generator().manual_seed(1)
    p = {k: v.to(dev) for k, v in make_params("head", 4, 64, F16, g).items()}
    x = torch.randn(8, 256, generator=g).to(F16).to(dev)
    lib, junk = H.load(), torch.zeros(1 << 16, dtype=torch.uint8, device=dev)
    outs = []
    for image in (None, junk.data_ptr()):
        out = torch.empty(8, 64, dtype=F16, device=dev)
        H.check(lib.mhc_head_fwd(x.data_ptr(), 2, p["phi_weight"].data_ptr(), 2, image,
                                 p["alpha"].data_ptr(), p["bias"].data_ptr(), 2, out.data_ptr(), None,
                                 None, 8, 4, 64, 1e-6, 1e-6, None, H.stream(dev)), "mhc_head_fwd")
        outs.append(out)
    assert torch.equal(*outs)
