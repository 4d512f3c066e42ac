"""Tensor-level wrappers of the C-ABI entry points.

Each function validates shapes, allocates the outputs with torch.empty on the
input's device (the library never allocates), and enqueues the kernel on the
current stream.  Inputs are made contiguous, as the reference's Functions do
(model/mhc_fused.py:585-586, :729-732).
"""
from __future__ import annotations

import ctypes
import functools
import threading
import weakref
from typing import Optional

import torch

from . import _hip as H

# What plain_call looks at has no public name.  On a torch where one is missing no call
# counts as plain, and the torch ops run.
try:
    from torch._C import _len_torch_dispatch_stack, _len_torch_function_stack
    from torch._C._functorch import peek_interpreter_stack
    from torch.autograd import forward_ad
    from torch.nn.modules.module import _global_forward_hooks, _global_forward_pre_hooks
    from torch.overrides import _get_current_function_mode_stack
    from torch.utils._device import DeviceContext
    CAN_TELL = isinstance(forward_ad._current_level, int)
except (ImportError, AttributeError):
    CAN_TELL = False

_GRAD = threading.local()


class GradAwareFunction(torch.autograd.Function):
    """An autograd Function whose forward can tell whether the caller had grad
    mode on.  ctx.needs_input_grad follows requires_grad alone, also under
    torch.no_grad(), so a forward that keys on it alone would save tensors,
    write backward-only outputs and repack trainable weights on every
    inference call."""

    @classmethod
    def apply(cls, *args, **kwargs):
        prev = getattr(_GRAD, "on", True)
        _GRAD.on = torch.is_grad_enabled()
        try:
            return super().apply(*args, **kwargs)
        finally:
            _GRAD.on = prev


def grad_wanted(ctx, index: Optional[int] = None) -> bool:
    """Inside a GradAwareFunction's forward: whether a gradient of any input
    (or of input `index`) will be asked for."""
    if not getattr(_GRAD, "on", True):
        return False
    return any(ctx.needs_input_grad) if index is None else bool(ctx.needs_input_grad[index])


def _contiguous(t: torch.Tensor) -> torch.Tensor:
    """t itself where its data already lie in order (only its pointer is used)."""
    return t if t.is_contiguous() else t.detach().contiguous()


class PhiPack:
    """MFMA operand image of a projection weight, rebuilt when the weight changes.

    Policy:
      * A weight that trains (grad mode on and phi.requires_grad) is repacked
        on every call.  Its values change every optimizer step, and in-place
        writes through .data (p.data.copy_ / normal_) do not bump the version
        counter, so no cache key could see them.  The pack is one small launch.
      * Otherwise (inference, frozen weights) the image is cached for one weight
        tensor object (held by weak reference, so a replaced parameter never
        aliases a freed one) at one value of its version counter, which
        optimizer steps, load_state_dict and copy_ bump.  A write through .data
        is invisible to that key: call invalidate() after one.  Inference
        tensors, which have no version counter, are repacked on every call.
    The cache is not pickled or deep-copied; a copy rebuilds it lazily.
    No reference counterpart: the reference's kernels read the row-major weight
    directly (model/mhc_fused.py:217-229).
    """

    def __init__(self, mode: int):
        self.mode = mode
        self.invalidate()

    def invalidate(self) -> None:
        """Drop the cached image; the next call repacks."""
        self._src = None
        self._key = None
        self._buf: Optional[torch.Tensor] = None

    def __getstate__(self):
        return {"mode": self.mode}

    def __setstate__(self, state):
        self.mode = state["mode"]
        self.invalidate()

    def get(self, phi: torch.Tensor, n: int, C: int,
            training: Optional[bool] = None) -> Optional[torch.Tensor]:
        """The image of phi (None when (n, C, dtype) has no MFMA kernel): the
        bf16 operand image for a bf16 phi (kernels for bf16 streams), the
        split hi / lo image for an fp32 phi (kernels for fp32 streams), the
        fp16 image for an fp16 phi (kernels for fp16 streams).
        training: whether phi trains in this call; default grad mode and
        phi.requires_grad (inside an autograd Function's forward, where grad
        mode is off, pass grad_wanted(ctx, <phi's index>))."""
        if training is None:
            training = torch.is_grad_enabled() and phi.requires_grad
        try:
            version = None if training else phi._version
        except RuntimeError:
            version = None
        key = (phi.data_ptr(), version, phi.device, phi.dtype, n, C)
        if (version is not None and self._buf is not None and self._src() is phi
                and key == self._key):
            return self._buf
        lib = H.load()
        if phi.dtype == torch.bfloat16:
            nbytes = lib.mhc_phi_packed_bytes(n, C, self.mode)
            pack = lib.mhc_phi_pack
        elif phi.dtype == torch.float32:
            nbytes = lib.mhc_phi_split_bytes(n, C, self.mode)
            pack = lib.mhc_phi_pack_split
        elif phi.dtype == torch.float16 and n > 1:
            nbytes = lib.mhc_phi_packed_bytes(n, C, self.mode)

            def pack(w, _dtype, buf, *rest):
                return lib.mhc_phi_pack_f16(w, buf, *rest)
        else:
            return None
        if nbytes <= 0:
            return None
        w = _contiguous(phi)
        buf = torch.empty(nbytes, dtype=torch.uint8, device=phi.device)
        H.check(pack(w.data_ptr(), H.dtype_tag(w), buf.data_ptr(), n, C, self.mode,
                     H.stream(phi.device)), "mhc_phi_pack")
        if version is None:
            self.invalidate()
        else:
            self._src = weakref.ref(phi)
            self._key = key
            self._buf = buf
        return buf


# Packs of weights that no module owns (the reference-style autograd Functions
# called directly): id(phi), mode -> (weak reference to phi, PhiPack).  An entry
# goes (with its device image) as soon as its weight is freed.
_PACKS: dict = {}


def _drop_pack(key, ref) -> None:
    ent = _PACKS.get(key)
    if ent is not None and ent[0] is ref:
        del _PACKS[key]


def packed_phi(phi: torch.Tensor, n: int, C: int, mode: int,
               training: Optional[bool] = None) -> Optional[torch.Tensor]:
    """MFMA image of phi for a caller without a PhiPack of its own (None when
    the shape or dtype has no MFMA kernel); training as in PhiPack.get."""
    if not phi.is_cuda:
        return None
    key = (id(phi), mode)
    ent = _PACKS.get(key)
    if ent is None or ent[0]() is not phi:
        ent = (weakref.ref(phi, lambda ref, key=key: _drop_pack(key, ref)), PhiPack(mode))
        _PACKS[key] = ent
    return ent[1].get(phi, n, C, training)


# ---------------------------------------------- sums of squares along a chain
SSQ_COLS = 128  # one fp32 partial per 128 columns of C (kSsqCols)


def ssq_wanted(dtype: torch.dtype, n: int, C: int) -> bool:
    """Whether a stream of this shape carries its rows' sums of squares from the
    launch that writes it to the pre launch that reads it: bf16, C a multiple
    of 128, and a pre kernel that would otherwise read the stream once more
    to form them (n = 8, n = 16, or C > 1024)."""
    return (dtype == torch.bfloat16 and C % SSQ_COLS == 0
            and (n in (8, 16) or (n >= 2 and C > 1024)))


class StreamChain:
    """Carries per-row sums of squares along a chain of mHC calls.

    The launch that writes a stream (the post phase, or the entry RMSNorm +
    StreamExpand) also writes its rows' partial sums of squares
    ([M, C / 128] fp32); the next pre launch that reads that exact tensor
    takes them instead of a pass over x of its own.  A caller that hands
    each call's output unchanged to the next call (as the MiniMind blocks do)
    creates one chain per forward and passes it to every mHC call; the sums
    are used only when the next call's input is the very tensor object the
    previous call returned.  Writing into that tensor in place between the
    calls is the caller's to avoid (the chain cannot see it).
    No reference counterpart."""

    __slots__ = ("src", "ssq")

    def __init__(self):
        self.src = None
        self.ssq = None

    def take(self, x: torch.Tensor, n: int, C: int) -> Optional[torch.Tensor]:
        """The sums of squares of x's rows, or None when x is not the tensor the
        chain last recorded (or the shape carries none)."""
        if self.ssq is None or self.src is not x:
            return None
        M = x.numel() // (n * C) if n * C else 0
        if tuple(self.ssq.shape) != (M, C // SSQ_COLS) or self.ssq.device != x.device:
            return None
        return self.ssq

    def buffer(self, like: torch.Tensor, n: int, C: int,
               rows: Optional[int] = None) -> Optional[torch.Tensor]:
        """A buffer for the sums of squares of an n-stream of `rows` tokens
        (default: `like` is such a stream, [..., n*C]) with like's dtype and
        device, or None when that shape carries none."""
        if not like.is_cuda or not ssq_wanted(like.dtype, n, C):
            return None
        M = like.numel() // (n * C) if rows is None else rows
        return torch.empty(M, C // SSQ_COLS, dtype=torch.float32, device=like.device)

    def put(self, out: torch.Tensor, ssq: Optional[torch.Tensor]) -> torch.Tensor:
        """Record out (the tensor handed to the next call) and its sums."""
        self.src = out
        self.ssq = ssq
        return out


def _phi_tag(phi: torch.Tensor, packed: Optional[torch.Tensor]) -> int:
    """phi's dtype tag, saying that `packed` is an fp16 image where it is one."""
    tag = H.dtype_tag(phi)
    return tag | H.PHI_F16_IMAGE if packed is not None and tag == H.DTYPE_F16 else tag


def _check_numel(name: str, t: torch.Tensor, want: int) -> None:
    # The kernels index biases by stream / matrix element; a short tensor would be
    # read out of bounds, so sizes are enforced here (the C ABI sees only pointers).
    if t.numel() != want:
        raise ValueError(f"mhc_amd: {name} has {t.numel()} elements, expected {want}")


def _rows(x_flat: torch.Tensor, NC: int) -> torch.Tensor:
    if x_flat.shape[-1] != NC:
        raise ValueError(f"mhc_amd: last dim {x_flat.shape[-1]} != n*C = {NC}")
    return _contiguous(x_flat).view(-1, NC)


def _flat(t: torch.Tensor, name: str, numel: int) -> torch.Tensor:
    """t in order, with that many elements (only its pointer is used)."""
    if t.numel() != numel:
        raise RuntimeError(f"mhc_amd: {name} of shape {tuple(t.shape)} has {t.numel()} elements, "
                           f"not {numel}")
    return _contiguous(t)


def _norm_args(norm, C: int, dev):
    """(weight pointer, dtype tag, eps, keep-alive tensor) of an RMSNorm over C
    fused into a pre-phase / head launch, or Nones without one."""
    if norm is None:
        return None, 0, 0.0, None
    w, eps = norm
    H.require_device(w)
    wc = _contiguous(w)
    _check_numel("norm weight", wc, C)
    if wc.device != dev:
        raise ValueError("mhc_amd: norm weight is on another device")
    return wc.data_ptr(), H.dtype_tag(wc), float(eps), wc


def _ssq_ptr(ssq, M: int, C: int):
    if ssq is None:
        return None
    if ssq.dtype != torch.float32 or tuple(ssq.shape) != (M, C // SSQ_COLS) or not ssq.is_contiguous():
        raise ValueError(f"mhc_amd: sums of squares must be contiguous fp32 [{M}, {C // SSQ_COLS}]")
    return ssq.data_ptr()


def pre_full(x_flat, phi, packed, a_pre, b_pre, a_post, b_post, a_res, b_res, n, C,
             post_mult, pre_eps, rms_eps, sk_iters, sk_eps, *, sinkhorn=True,
             want_h_pre=False, want_raw=False, want_saved=False, norm=None, ssq=None):
    """Fused pre phase (+ Sinkhorn).  Returns a dict of [M, ...] tensors.
    norm=(weight [C], eps): "sub_in" is RMSNorm(pre-aggregate) instead.
    ssq: x's per-row partial sums of squares ([M, C / 128] fp32, from the
    launch that wrote x), or None."""
    dev = H.require_device(x_flat, phi, a_pre, b_pre, a_post, b_post, a_res, b_res)
    NC = n * C
    FD = 2 * n + n * n
    if tuple(phi.shape) != (NC, FD):
        raise ValueError(f"mhc_amd: phi_weight shape {tuple(phi.shape)} != ({NC}, {FD})")
    x2 = _rows(x_flat, NC)
    M = x2.shape[0]
    phi_c = _contiguous(phi)
    a_pre, b_pre, a_post, b_post, a_res, b_res = H.params_like(
        x2, a_pre, b_pre, a_post, b_post, a_res, b_res)
    _check_numel("alpha_pre", a_pre, 1)
    _check_numel("alpha_post", a_post, 1)
    _check_numel("alpha_res", a_res, 1)
    _check_numel("bias_pre", b_pre, n)
    _check_numel("bias_post", b_post, n)
    _check_numel("bias_res", b_res, n * n)
    new = x2.new_empty
    f32 = torch.float32
    out = {
        "sub_in": new((M, C)),
        "h_post": new((M, n)),
        "h_pre": new((M, n)) if want_h_pre else None,
        "h_res_raw": new((M, n, n)) if want_raw else None,
        "h_res": new((M, n, n)) if sinkhorn else None,
        "inv_rms": new((M,), dtype=f32) if want_saved else None,
        "mixes_raw": new((M, FD), dtype=f32) if want_saved else None,
    }
    args = (x2.data_ptr(), H.dtype_tag(x2), phi_c.data_ptr(), _phi_tag(phi_c, packed), H.ptr(packed),
            a_pre.data_ptr(), b_pre.data_ptr(), a_post.data_ptr(), b_post.data_ptr(),
            a_res.data_ptr(), b_res.data_ptr(), H.dtype_tag(a_pre),
            out["sub_in"].data_ptr(), H.ptr(out["h_pre"]), out["h_post"].data_ptr(),
            H.ptr(out["h_res_raw"]), H.ptr(out["h_res"]), H.ptr(out["inv_rms"]),
            H.ptr(out["mixes_raw"]), M, n, C, float(post_mult), float(pre_eps), float(rms_eps),
            int(sk_iters), float(sk_eps))
    sp = _ssq_ptr(ssq, M, C)
    if norm is None:
        H.check(H.load().mhc_pre_fwd(*args, sp, H.stream(dev)), "mhc_pre_fwd")
    else:
        wp, wdt, weps, _keep = _norm_args(norm, C, dev)
        H.check(H.load().mhc_pre_norm_fwd(*args, wp, wdt, weps, sp, H.stream(dev)),
                "mhc_pre_norm_fwd")
    return out


def pre_nohres(x_flat, phi, packed, a_pre, b_pre, a_post, b_post, n, C, post_mult, pre_eps,
               rms_eps, *, want_h_pre=False, want_saved=False, norm=None, ssq=None):
    dev = H.require_device(x_flat, phi, a_pre, b_pre, a_post, b_post)
    NC = n * C
    FD = 2 * n
    if tuple(phi.shape) != (NC, FD):
        raise ValueError(f"mhc_amd: phi_weight shape {tuple(phi.shape)} != ({NC}, {FD})")
    x2 = _rows(x_flat, NC)
    M = x2.shape[0]
    phi_c = _contiguous(phi)
    a_pre, b_pre, a_post, b_post = H.params_like(x2, a_pre, b_pre, a_post, b_post)
    _check_numel("alpha_pre", a_pre, 1)
    _check_numel("alpha_post", a_post, 1)
    _check_numel("bias_pre", b_pre, n)
    _check_numel("bias_post", b_post, n)
    new = x2.new_empty
    f32 = torch.float32
    out = {
        "sub_in": new((M, C)),
        "h_post": new((M, n)),
        "h_pre": new((M, n)) if want_h_pre else None,
        "inv_rms": new((M,), dtype=f32) if want_saved else None,
        "mixes_raw": new((M, FD), dtype=f32) if want_saved else None,
    }
    args = (x2.data_ptr(), H.dtype_tag(x2), phi_c.data_ptr(), _phi_tag(phi_c, packed), H.ptr(packed),
            a_pre.data_ptr(), b_pre.data_ptr(), a_post.data_ptr(), b_post.data_ptr(),
            H.dtype_tag(a_pre), out["sub_in"].data_ptr(), H.ptr(out["h_pre"]),
            out["h_post"].data_ptr(), H.ptr(out["inv_rms"]), H.ptr(out["mixes_raw"]),
            M, n, C, float(post_mult), float(pre_eps), float(rms_eps))
    sp = _ssq_ptr(ssq, M, C)
    if norm is None:
        H.check(H.load().mhc_pre_nohres_fwd(*args, sp, H.stream(dev)), "mhc_pre_nohres_fwd")
    else:
        wp, wdt, weps, _keep = _norm_args(norm, C, dev)
        H.check(H.load().mhc_pre_nohres_norm_fwd(*args, wp, wdt, weps, sp, H.stream(dev)),
                "mhc_pre_nohres_norm_fwd")
    return out


def head(x_flat, phi, packed, alpha, bias, n, C, pre_eps, rms_eps, *, want_saved=False,
         norm=None, ssq=None):
    """MHCHead forward; n == 1 is the plain RMSNorm (phi/alpha/bias unused).
    norm=(weight [C], eps): the model's final RMSNorm applied in the same launch."""
    NC = n * C
    x2 = _rows(x_flat, NC)
    M = x2.shape[0]
    if n == 1:
        dev = H.require_device(x_flat)
        phi_p = a_p = b_p = None
        phi_dt = pdt = H.DTYPE_F32
    else:
        dev = H.require_device(x_flat, phi, alpha, bias)
        if tuple(phi.shape) != (NC, n):
            raise ValueError(f"mhc_amd: phi_weight shape {tuple(phi.shape)} != ({NC}, {n})")
        phi_c = _contiguous(phi)
        alpha_c, bias_c = H.params_like(x2, alpha, bias)
        _check_numel("alpha", alpha_c, 1)
        _check_numel("bias", bias_c, n)
        phi_p, a_p, b_p = phi_c.data_ptr(), alpha_c.data_ptr(), bias_c.data_ptr()
        phi_dt, pdt = _phi_tag(phi_c, packed), H.dtype_tag(alpha_c)
    out = torch.empty(M, C, dtype=x2.dtype, device=dev)
    inv = torch.empty(M, dtype=torch.float32, device=dev) if want_saved else None
    mix = torch.empty(M, n, dtype=torch.float32, device=dev) if (want_saved and n > 1) else None
    args = (x2.data_ptr(), H.dtype_tag(x2), phi_p, phi_dt, H.ptr(packed), a_p, b_p, pdt,
            out.data_ptr(), H.ptr(inv), H.ptr(mix), M, n, C, float(pre_eps), float(rms_eps))
    sp = _ssq_ptr(ssq, M, C) if n > 1 else None
    if norm is None:
        H.check(H.load().mhc_head_fwd(*args, sp, H.stream(dev)), "mhc_head_fwd")
    else:
        wp, wdt, weps, _keep = _norm_args(norm, C, dev)
        H.check(H.load().mhc_head_norm_fwd(*args, wp, wdt, weps, sp, H.stream(dev)),
                "mhc_head_norm_fwd")
    return out, inv, mix


def post(x_flat, h_res, h_post, f_out, n, C, ssq_out=None):
    """out = H_res . x + H_post (x) F; h_res None means identity (use_mhc = 2).
    ssq_out: an [M, C / 128] fp32 buffer that receives out's per-row partial
    sums of squares (for the next pre launch), or None."""
    dev = H.require_device(x_flat, h_res, h_post, f_out)
    NC = n * C
    x2 = _rows(x_flat, NC)
    M = x2.shape[0]
    hp = _flat(h_post, "h_post", M * n)
    f2 = _flat(f_out, "f_out", M * C)
    if hp.dtype != (h_res.dtype if h_res is not None else hp.dtype):
        raise TypeError("mhc_amd: h_res and h_post must share a dtype")
    out = torch.empty_like(x2)
    lib = H.load()
    sp = _ssq_ptr(ssq_out, M, C)
    if h_res is not None:
        hr = _flat(h_res, "h_res", M * n * n)
        rc = lib.mhc_post_fwd(x2.data_ptr(), H.dtype_tag(x2), hr.data_ptr(), hp.data_ptr(),
                              H.dtype_tag(hp), f2.data_ptr(), H.dtype_tag(f2), out.data_ptr(),
                              M, n, C, sp, H.stream(dev))
        H.check(rc, "mhc_post_fwd")
    else:
        rc = lib.mhc_post_nohres_fwd(x2.data_ptr(), H.dtype_tag(x2), hp.data_ptr(),
                                     H.dtype_tag(hp), f2.data_ptr(), H.dtype_tag(f2),
                                     out.data_ptr(), M, n, C, sp, H.stream(dev))
        H.check(rc, "mhc_post_nohres_fwd")
    return out


def sinkhorn(m: torch.Tensor, iters: int, eps: float) -> torch.Tensor:
    dev = H.require_device(m)
    N = m.shape[-1]
    if m.dim() < 2 or m.shape[-2] != N:
        raise ValueError(f"mhc_amd: last two dims must be square, got {tuple(m.shape)}")
    mc = m.contiguous()
    out = torch.empty_like(mc)
    batch = mc.numel() // (N * N) if N > 0 else 0
    rc = H.load().mhc_sinkhorn_fwd(mc.data_ptr(), out.data_ptr(), H.dtype_tag(mc), batch, N,
                                   int(iters), float(eps), H.stream(dev))
    H.check(rc, "mhc_sinkhorn_fwd")
    return out


def expand_norm(x: torch.Tensor, weight: torch.Tensor, eps: float, n: int,
                ssq_out=None) -> torch.Tensor:
    """RMSNorm over the last dim (gain weight) followed by StreamExpand to n
    copies, one launch: [B, L, C] -> [B, L, n*C].  ssq_out as in post."""
    dev = H.require_device(x, weight)
    B, L, C = x.shape
    xc = x.contiguous()
    wp, wdt, weps, _keep = _norm_args((weight, eps), C, dev)
    out = torch.empty(B, L, n * C, dtype=x.dtype, device=dev)
    rc = H.load().mhc_expand_norm_fwd(xc.data_ptr(), H.dtype_tag(xc), wp, wdt, out.data_ptr(),
                                      B * L, n, C, weps, _ssq_ptr(ssq_out, B * L, C),
                                      H.stream(dev))
    H.check(rc, "mhc_expand_norm_fwd")
    return out


def pre_token_threshold(max_tokens: int = -1) -> int:
    """Set (max_tokens >= 0) or query the batch size at or below which the
    pre-phase launches use the small-batch group kernel (bit-identical to the
    large-batch kernels); returns the previous value."""
    return int(H.load().mhc_pre_token_threshold(int(max_tokens)))


def pre_row_staging(on: int = -1) -> int:
    """Set (on >= 0) or query whether the persistent pre kernel loads x tiles
    as whole rows staged through LDS where the shape allows; returns the
    previous setting (0 or 1).  The two agree to rounding (the row sums of
    squares are added in another order)."""
    return int(H.load().mhc_pre_row_staging(int(on)))


def pre_group_split_tokens(max_tokens: int = -1) -> int:
    """Set (max_tokens >= 0) or query the batch size at or below which the
    n = 8 small-batch pre phase runs as two launches (the projection split
    over the output tiles; bit-identical); returns the previous value."""
    return int(H.load().mhc_pre_group_split_tokens(int(max_tokens)))


def stream_expand(x: torch.Tensor, n: int) -> torch.Tensor:
    dev = H.require_device(x)
    B, L, D = x.shape
    xc = x.contiguous()
    out = torch.empty(B, L, n * D, dtype=x.dtype, device=dev)
    rc = H.load().mhc_stream_expand_fwd(xc.data_ptr(), out.data_ptr(), xc.element_size(),
                                        B * L, n, D, H.stream(dev))
    H.check(rc, "mhc_stream_expand_fwd")
    return out


# ------------------------------------------------------------------ backward
# Gradients come back in the dtypes the reference's backward kernels store:
# the forward inputs' dtypes, with the per-token g_raw in fp32.

def post_bwd(x_flat, h_res, h_post, f_out, n, C, g_out):
    """(g_x, g_h_res, g_h_post, g_f) of out = H_res . x + H_post (x) F.  With
    h_res None (use_mhc = 2) g_x is g_out itself and g_h_res is None."""
    dev = H.require_device(g_out, h_post, f_out, h_res, x_flat if h_res is not None else None)
    NC = n * C
    M = g_out.numel() // NC
    hp = _contiguous(h_post).view(M, n)
    f2 = _contiguous(f_out).view(M, C)
    g_hp = torch.empty_like(hp)
    g_f = torch.empty_like(f2)
    lib = H.load()
    if h_res is None:
        g2 = _rows(g_out, NC)
        rc = lib.mhc_post_nohres_bwd(hp.data_ptr(), H.dtype_tag(hp), f2.data_ptr(), H.dtype_tag(f2),
                                     g2.data_ptr(), H.dtype_tag(g2), None, g_hp.data_ptr(),
                                     g_f.data_ptr(), M, n, C, H.stream(dev))
        H.check(rc, "mhc_post_nohres_bwd")
        return g2, None, g_hp, g_f
    x2 = _rows(x_flat, NC)
    g2 = _rows(g_out, NC)
    if g2.dtype != x2.dtype:
        g2 = g2.to(x2.dtype)
    hr = _contiguous(h_res).view(M, n, n)
    if hr.dtype != hp.dtype:
        raise TypeError("mhc_amd: h_res and h_post must share a dtype")
    g_x = torch.empty_like(x2)
    g_hr = torch.empty_like(hr)
    rc = lib.mhc_post_bwd(x2.data_ptr(), H.dtype_tag(x2), hr.data_ptr(), hp.data_ptr(),
                          H.dtype_tag(hp), f2.data_ptr(), H.dtype_tag(f2), g2.data_ptr(),
                          g_x.data_ptr(), g_hr.data_ptr(), g_hp.data_ptr(), g_f.data_ptr(),
                          M, n, C, H.stream(dev))
    H.check(rc, "mhc_post_bwd")
    return g_x, g_hr, g_hp, g_f


def pre_bwd(x2, phi, alphas, biases, inv_rms, mixes, n, C, mode, post_mult, pre_eps,
            g_sub=None, g_hpre=None, g_hpost=None, g_hres=None, g_x_in=None):
    """Per-token pre-phase backward.  alphas / biases: (pre, post, res) with
    None for absent segments.  g_x_in: a gradient of x from elsewhere, added to
    g_x in the same launch.  Returns (g_x [M, n*C] x dtype, g_raw [M, FD] fp32
    or None for mode RMS)."""
    grads = [g for g in (g_sub, g_hpre, g_hpost, g_hres) if g is not None]
    dev = H.require_device(x2, inv_rms, *grads)
    M = x2.shape[0]
    gdt = grads[0].dtype if grads else x2.dtype
    g_sub, g_hpre, g_hpost, g_hres = (
        g if g is None or (g.dtype == gdt and g.is_contiguous()) else g.to(gdt).contiguous()
        for g in (g_sub, g_hpre, g_hpost, g_hres))
    if g_x_in is not None:
        H.require_device(x2, g_x_in)
        g_x_in = g_x_in.to(x2.dtype).reshape(x2.shape).contiguous()
        if g_x_in.data_ptr() % 16:  # a caller's view; the MFMA kernels load 16 bytes
            g_x_in = g_x_in.clone()
    g_x = torch.empty_like(x2)
    if mode == H.MODE_RMS:
        phi_p = phi_dt = None
        ps = [None] * 5
        pdt = H.DTYPE_F32
        g_raw = None
    else:
        FD = {H.MODE_FULL: 2 * n + n * n, H.MODE_NOHRES: 2 * n, H.MODE_HEAD: n}[mode]
        phi_c = _contiguous(phi)
        phi_p, phi_dt = phi_c.data_ptr(), H.dtype_tag(phi_c)
        present = [p for p in (alphas[0], biases[0], alphas[1], biases[1], alphas[2]) if p is not None]
        conv = iter(H.params_like(x2, *present))
        ps = [None if p is None else next(conv)
              for p in (alphas[0], biases[0], alphas[1], biases[1], alphas[2])]
        pdt = H.dtype_tag(ps[0])
        g_raw = torch.empty(M, FD, dtype=torch.float32, device=dev)
    rc = H.load().mhc_pre_bwd_add(
        x2.data_ptr(), H.dtype_tag(x2), phi_p, phi_dt if phi_dt is not None else H.DTYPE_F32,
        *[H.ptr(p) for p in ps], pdt, inv_rms.data_ptr(), H.ptr(mixes),
        H.ptr(g_sub), H.ptr(g_hpre), H.ptr(g_hpost), H.ptr(g_hres),
        H.dtype_tag(g_sub if g_sub is not None else x2), H.ptr(g_x_in), g_x.data_ptr(), H.ptr(g_raw),
        M, n, C, mode, float(post_mult), float(pre_eps), H.stream(dev))
    H.check(rc, "mhc_pre_bwd")
    return g_x, g_raw


def pre_bwd_weights(x2, inv_rms, mixes, g_raw, phi, alphas, n, C, mode):
    """(g_phi, [g_alpha_seg], [g_bias_seg]) from pre_bwd's g_raw; alphas as in
    pre_bwd.  g_alpha_* are 0-dim, g_bias_* flat, all in the alphas' dtype."""
    dev = H.require_device(x2, inv_rms, mixes, g_raw, phi)
    M = x2.shape[0]
    present = [a for a in alphas if a is not None]
    conv = iter(H.params_like(x2, *present))
    al = [None if a is None else next(conv) for a in alphas]
    pdt = al[0].dtype
    lib = H.load()
    g_phi = torch.empty(phi.shape, dtype=phi.dtype, device=dev)
    sizes = (n, n, n * n)
    g_alpha = [None if a is None else torch.empty((), dtype=pdt, device=dev) for a in al]
    g_bias = [None if a is None else torch.empty(sizes[i], dtype=pdt, device=dev)
              for i, a in enumerate(al)]
    if M == 0:
        g_phi.zero_()
        for t in g_alpha + g_bias:
            if t is not None:
                t.zero_()
        return g_phi, g_alpha, g_bias
    nbytes = lib.mhc_pre_bwd_weights_workspace_bytes(M, n, C, mode)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    rc = lib.mhc_pre_bwd_weights(
        x2.data_ptr(), H.dtype_tag(x2), inv_rms.data_ptr(), mixes.data_ptr(), g_raw.data_ptr(),
        *[H.ptr(a) for a in al], H.dtype_tag(al[0]), g_phi.data_ptr(), H.dtype_tag(g_phi),
        H.ptr(g_alpha[0]), H.ptr(g_bias[0]), H.ptr(g_alpha[1]), H.ptr(g_bias[1]),
        H.ptr(g_alpha[2]), H.ptr(g_bias[2]), ws.data_ptr(), nbytes, M, n, C, mode,
        H.stream(dev))
    H.check(rc, "mhc_pre_bwd_weights")
    return g_phi, g_alpha, g_bias


def check_sinkhorn_bwd_iters(n: int, iters: int) -> None:
    """Raise, before a forward whose Sinkhorn will need a gradient, when the
    backward kernel cannot take `iters` iterations for n (it would otherwise
    fail only at backward)."""
    cap = int(H.load().mhc_sinkhorn_bwd_max_iters(int(n)))
    if iters > cap:
        raise ValueError(f"mhc_amd: sinkhorn_iters={iters} exceeds what the Sinkhorn backward "
                         f"takes for n={n} ({cap}); train with sinkhorn_iters <= {cap}")


def sinkhorn_bwd(m: torch.Tensor, g: torch.Tensor, iters: int, eps: float,
                 out_dtype=None) -> torch.Tensor:
    """d sinkhorn(m) / d m applied to g, stored in out_dtype (default m's)."""
    dev = H.require_device(m, g)
    N = m.shape[-1]
    mc = m.contiguous()
    gc = g.contiguous()
    out = torch.empty(mc.shape, dtype=out_dtype or mc.dtype, device=dev)
    batch = mc.numel() // (N * N) if N > 0 else 0
    rc = H.load().mhc_sinkhorn_bwd(mc.data_ptr(), H.dtype_tag(mc), gc.data_ptr(), H.dtype_tag(gc),
                                   out.data_ptr(), H.dtype_tag(out), batch, N, int(iters),
                                   float(eps), H.stream(dev))
    H.check(rc, "mhc_sinkhorn_bwd")
    return out


# ------------------------------------------- the model's sublayers, inference
# Kernels in place of the torch ops of the sublayers.  They record no autograd
# graph and see only data pointers, so a call takes them only when nothing but
# the numbers could tell: no grad mode, no forward-mode level, no functorch
# transform, no tracing or compiling, no dispatch or function mode, no autocast, and
# submodules that nobody has hooked or patched.

# torch.cuda.current_device also looks whether torch's GPU side is set up, which a GPU
# tensor answers: 0.3 us a call.
_current_device = getattr(torch._C, "_cuda_getDevice", None) or torch.cuda.current_device


def on_current_device(t: torch.Tensor) -> bool:
    """Whether t, a GPU tensor, lies on the device the library would launch on.  Its entry points set no
    device, and a device's default stream is handle 0 on every device, so for a tensor
    of another one the launch would go to the wrong GPU; torch ops set the device."""
    return t.get_device() == _current_device()


def _function_modes() -> bool:
    """Whether one of the torch-function modes on the stack could see or replace the torch
    ops.  The one that torch.set_default_device and `with torch.device(...)` leave there
    only changes factory calls without a device, of which the sublayers make none."""
    return any(type(m) is not DeviceContext for m in _get_current_function_mode_stack())


def plain_call() -> bool:
    """Whether nothing is recording, transforming or tracing torch ops here.
    Compiling is asked first: Dynamo knows that answer, and cannot trace the rest."""
    return not (torch.compiler.is_compiling() or not CAN_TELL
                or torch.is_grad_enabled() or torch.is_autocast_enabled("cuda")
                or forward_ad._current_level >= 0
                or _len_torch_dispatch_stack() > 0
                or (_len_torch_function_stack() > 0 and _function_modes())
                or peek_interpreter_stack() is not None
                or torch.jit.is_tracing())


def plain_module(m: torch.nn.Module, kind: type) -> bool:
    """Whether m is exactly a `kind` whose call is its class's forward: no hooks
    on it or on all modules, no forward of its own."""
    return (type(m) is kind and "forward" not in m.__dict__
            and not (m._forward_hooks or m._forward_pre_hooks)
            and not (_global_forward_hooks or _global_forward_pre_hooks))


_PLAIN = (torch.Tensor, torch.nn.Parameter)


def plain_tensors(dtype: torch.dtype, dev: torch.device, *ts) -> bool:
    """Whether every tensor is a plain one of that dtype on that GPU, its data
    16-byte aligned."""
    index = dev.index
    for t in ts:
        if (type(t) not in _PLAIN or t.dtype != dtype or not t.is_cuda or t.get_device() != index
                or t.data_ptr() % 16):
            return False
    return True


# Multiply-adds past which one linear layer is the library's at every K.
LINEAR_MAX_MACS = 13_000_000_000


@functools.lru_cache(maxsize=4096)
def _linear_pays(M: int, K: int, ns: tuple, glu: bool = False) -> bool:
    """Whether the kernels are no slower than the library for these sizes."""
    if M * K * sum(ns) >= 1 << 62 or max(M, K, *ns) >= 1 << 31:
        return False
    return bool(H.load().mhc_linear_pays((ctypes.c_int * len(ns))(*ns), len(ns), M, K, int(glu)))


_HALF = (torch.bfloat16, torch.float16)


def _linear_weights(x: torch.Tensor, mods, glu: bool = False, closely: bool = True):
    """The weights of bias-free nn.Linear layers the kernels can apply to x, or None; also
    None where the library is faster (not closely: where it is at every K).  That is asked
    before what takes longer to look at: a call left to torch waits for this."""
    if not isinstance(x, torch.Tensor):  # an fx Proxy: the torch ops are traced
        return None
    if not x.is_cuda or x.dtype not in _HALF or not plain_call():
        return None
    total = x.numel()
    if x.dim() < 2 or total == 0:
        return None
    K = x.shape[-1]
    if K % 32 != 0 or K > 1 << 22:
        return None
    try:
        ns = tuple([m.out_features for m in mods])
    except AttributeError:
        return None
    if not (_linear_pays(total // K, K, ns, glu) if closely else total * ns[0] <= LINEAR_MAX_MACS):
        return None
    if not on_current_device(x) or not x.is_contiguous():
        return None
    ws = []
    for m in mods:
        if not plain_module(m, torch.nn.Linear) or m.bias is not None:
            return None
        w = m.weight
        if w.dim() != 2 or w.shape[1] != K or not 4 <= w.shape[0] <= 1 << 30 or w.shape[0] % 4 != 0 or not w.is_contiguous():
            return None
        ws.append(w)
    return ws if plain_tensors(x.dtype, x.device, x, *ws) else None


def _launch_linears(x: torch.Tensor, ws):
    K, n = x.shape[-1], len(ws)
    outs = [x.new_empty(*x.shape[:-1], w.shape[0]) for w in ws]
    H.check(H.load().mhc_linear_fwd(
        x.data_ptr(), (ctypes.c_void_p * n)(*[w.data_ptr() for w in ws]),
        (ctypes.c_void_p * n)(*[o.data_ptr() for o in outs]),
        (ctypes.c_int * n)(*[w.shape[0] for w in ws]), n, x.numel() // K, K, H.dtype_tag(x),
        H.stream(x.device)), "mhc_linear_fwd")
    return outs


def linears(x: torch.Tensor, *mods):
    """[m(x) for m in mods] for one to three bias-free nn.Linear layers in one
    launch, or None for a call the kernels do not take or that is faster in the
    library (`linear` looks closer at a single layer)."""
    ws = _linear_weights(x, mods, closely=len(mods) > 1)
    return None if ws is None else _launch_linears(x, ws)


def linear(x: torch.Tensor, m: torch.nn.Module) -> torch.Tensor:
    """m(x), on mhc_linear_fwd for a call that it takes and that is not faster in the
    library."""
    ws = _linear_weights(x, (m,))
    return m(x) if ws is None else _launch_linears(x, ws)[0]


def glu(x: torch.Tensor, gate: torch.nn.Module, up: torch.nn.Module) -> Optional[torch.Tensor]:
    """silu(gate(x)) * up(x) for bias-free nn.Linear layers in one launch, or None
    for a call the kernels do not take."""
    ws = _linear_weights(x, (gate, up), glu=True)
    if ws is None or ws[0].shape != ws[1].shape:
        return None
    K, N = x.shape[-1], ws[0].shape[0]
    out = x.new_empty(*x.shape[:-1], N)
    H.check(H.load().mhc_glu_fwd(x.data_ptr(), ws[0].data_ptr(), ws[1].data_ptr(), out.data_ptr(),
                                 x.numel() // K, K, N, H.dtype_tag(x), H.stream(x.device)),
            "mhc_glu_fwd")
    return out


ATTN_HEAD_DIMS = (64, 96, 128)
ATTN_MAX_ROWS = 1 << 20  # sequences x kv heads of a decode step; mhc_attn_decode_fwd refuses more


def attn_route(m, q, k, v, position_embeddings, past) -> Optional[str]:
    """Which kernel serves this call of the attention layer m between its
    projections (q, k, v): "prefill", "decode", or None (the torch ops).
    q [B, T, heads * head_dim]; k, v [B, T, kv_heads * head_dim]."""
    H_, KV, hd = m.n_local_heads, m.n_local_kv_heads, m.head_dim
    if (not q.is_cuda or q.dtype not in _HALF or hd not in ATTN_HEAD_DIMS
            or q.dim() != 3 or H_ % KV != 0 or not plain_call() or not on_current_device(q)):
        return None
    B, T, _ = q.shape
    if B * T == 0 or (m.training and m.dropout > 0) or (T > 1 and not m.is_causal):
        return None
    if not (plain_module(m.q_norm, torch.nn.RMSNorm) and plain_module(m.k_norm, torch.nn.RMSNorm)):
        return None
    if m.q_norm.eps is None or m.k_norm.eps is None:  # torch's own choice, which its versions differ in
        return None
    cos, sin = position_embeddings
    gq, gk = m.q_norm.weight, m.k_norm.weight
    if gq is None or gk is None or not plain_tensors(q.dtype, q.device, q, k, v, gq, gk, cos, sin):
        return None
    if not (q.shape == (B, T, H_ * hd) and k.shape == v.shape == (B, T, KV * hd)
            and gq.shape == gk.shape == (hd,) and cos.shape == sin.shape == (T, hd)
            and all(t.is_contiguous() for t in (q, k, v, gq, gk, cos, sin))):
        return None
    if past is None:
        return "prefill"
    pk, pv = past[0], past[1]
    if (T != 1 or H_ // KV > 4 or not plain_tensors(q.dtype, q.device, pk, pv)
            or pk.dim() != 4 or pk.shape != pv.shape
            or pk.shape[0] != B or pk.shape[1] < 1 or tuple(pk.shape[2:]) != (KV, hd)
            or B * KV > ATTN_MAX_ROWS):
        return None
    for t in (pk, pv):
        if t.stride(3) != 1 or any(s % 8 for s in t.stride()[:3]):
            return None
    return "decode"


def attn_prefill(m, q, k, v, position_embeddings):
    """(attention output [B, T, heads * head_dim], normed and rotated k); the
    call is one attn_route calls "prefill"."""
    B, T, _ = q.shape
    H_, KV, hd = m.n_local_heads, m.n_local_kv_heads, m.head_dim
    cos, sin = position_embeddings
    kr, out = torch.empty_like(k), torch.empty_like(q)
    H.check(H.load().mhc_attn_prefill_fwd(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), m.q_norm.weight.data_ptr(),
        m.k_norm.weight.data_ptr(), cos.data_ptr(), sin.data_ptr(), kr.data_ptr(), out.data_ptr(),
        B, T, H_, KV, hd, H.dtype_tag(q), float(m.q_norm.eps), float(m.k_norm.eps),
        H.stream(q.device)), "mhc_attn_prefill_fwd")
    return out, kr


def attn_decode(m, q, k, v, position_embeddings, past, use_cache: bool):
    """(attention output [B, 1, heads * head_dim], grown (k, v) caches or None);
    the call is one attn_route calls "decode"."""
    B = q.shape[0]
    H_, KV, hd = m.n_local_heads, m.n_local_kv_heads, m.head_dim
    cos, sin = position_embeddings
    pk, pv = past[0], past[1]
    S = pk.shape[1]
    lib = H.load()
    out = torch.empty_like(q)
    grown = None
    if use_cache:
        grown = tuple(torch.empty(B, S + 1, KV, hd, dtype=q.dtype, device=q.device)
                      for _ in range(2))
    nbytes = lib.mhc_attn_decode_workspace_bytes(B, S, H_, KV, hd)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=q.device) if nbytes > 0 else None
    H.check(lib.mhc_attn_decode_fwd(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), m.q_norm.weight.data_ptr(),
        m.k_norm.weight.data_ptr(), cos.data_ptr(), sin.data_ptr(),
        pk.data_ptr(), *pk.stride()[:3], pv.data_ptr(), *pv.stride()[:3],
        grown[0].data_ptr() if grown else None, grown[1].data_ptr() if grown else None,
        out.data_ptr(), H.ptr(ws), max(nbytes, 0), B, S, H_, KV, hd, H.dtype_tag(q),
        float(m.q_norm.eps), float(m.k_norm.eps), H.stream(q.device)),
        "mhc_attn_decode_fwd")
    return out, grown


# Past both, the experts' products by the library, one expert after another, are as fast
# or faster with all the passes around them: 4096 x 14336, 8192 tokens, 4 experts, top 1,
# 3.55 ms on the kernels and 3.25 in the loop (4096 tokens 1.92 and 2.08); 8192 x 8192 3.67
# and 3.48 (4096 tokens 2.02 and 2.18); 4096 x 8192, 8192 tokens, 8 experts, top 2, 3.75 and
# 4.39; at hidden 768 to 3072 the loop takes 1.08 to 6 times as long at every size measured.
MOE_LOOP_WEIGHT = 1 << 25   # elements of one weight
MOE_LOOP_ROWS = 2048        # rows an expert, on average


def moe_experts(experts, x: torch.Tensor, probs: torch.Tensor, topk: int, norm_topk: bool,
                zero: Optional[torch.Tensor] = None):
    """The routed experts' weighted sum for x [M, hidden] on the HIP kernels, or
    None for a call they do not take.  experts: modules with gate_proj, up_proj
    and down_proj (plain nn.Linear without bias) and SiLU between them; probs
    [M, experts], the router's softmax; zero: a tensor of x's type whose one element
    the last launch sets to 0."""
    if (not x.is_cuda or x.dtype not in _HALF or not plain_call()
            or not on_current_device(x) or x.dim() != 2 or x.shape[0] == 0 or not x.is_contiguous()
            or probs.shape != (x.shape[0], len(experts)) or not probs.is_contiguous()):
        return None
    if zero is not None and (zero.numel() != 1 or zero.dtype != x.dtype or zero.device != x.device):
        return None
    M, D = x.shape
    inter = getattr(experts[0].gate_proj, "out_features", 0)
    if D * inter > MOE_LOOP_WEIGHT and M * topk >= MOE_LOOP_ROWS * len(experts):
        return None
    kind, ws = type(experts[0]), ([], [], [])
    for e in experts:
        if not plain_module(e, kind):
            return None
        for lin, w in zip((e.gate_proj, e.up_proj, e.down_proj), ws):
            if not plain_module(lin, torch.nn.Linear) or lin.bias is not None:
                return None
            w.append(lin.weight)
    inter = ws[0][0].shape[0]
    if (any(t.shape != (inter, D) or not t.is_contiguous() for t in ws[0] + ws[1])
            or any(t.shape != (D, inter) or not t.is_contiguous() for t in ws[2])
            or not plain_tensors(x.dtype, x.device, x, probs, *ws[0], *ws[1], *ws[2])):
        return None
    lib = H.load()
    nbytes = lib.mhc_moe_workspace_bytes(M, D, inter, len(experts), topk)
    if nbytes < 0:
        return None
    try:  # every expert's rows at once; the loop needs one expert's at a time
        work = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
    except torch.OutOfMemoryError:
        return None
    out = torch.empty_like(x)
    ptrs = [(ctypes.c_void_p * len(w))(*[t.data_ptr() for t in w]) for w in ws]
    H.check(lib.mhc_moe_fwd(x.data_ptr(), probs.data_ptr(), *ptrs, out.data_ptr(), H.ptr(zero),
                            work.data_ptr(), nbytes, M, D, inter, len(experts), topk,
                            int(norm_topk), H.dtype_tag(x), H.stream(x.device)), "mhc_moe_fwd")
    return out
