"""Torch-facing operators over the C ABI (HIP kernels on gfx950).

``cheby_ema_forward``   fused forward (static or dynamic lambda, EMA carry).
``cheby_ema_ttt``       fused forward + TTT coefficient gradient.
``cheby_ema_backward``  dL/dx, dL/dc, dL/d ema_init from dL/dout (+ dL/d ema_final).
``cheby_ema``           the forward as a differentiable op (autograd.Function
                        whose backward is ``cheby_ema_backward``).
``v10_chunked_ttt``     the reference's full path: online TTT over chunks with
                        an inline Lion update, in one launch.
``cheby_ema_lut_forward`` the fixed-coefficient LUT/Clenshaw forward of the
                        reference's _fused_clenshaw_ema_kernel (x_norm,
                        tanh_y, out and the carried state), in one launch.

All run on the current torch stream of the input's device and never
synchronise the host.  Inputs are not modified.  There is no CPU path: a
tensor that is not on a ROCm device raises.
"""
from __future__ import annotations

import ctypes
import os
import threading
from typing import Sequence

import torch

from . import _native as nat

_ws_lock = threading.Lock()
_ws_cache: dict[tuple[int, int, int], torch.Tensor] = {}
# Workspaces whose address a captured graph holds: the keys whose current one
# does, and those that a larger one has replaced since (see _workspace).
_ws_in_graph: set[tuple[int, int, int]] = set()
_ws_kept: list[tuple[tuple[int, int, int], torch.Tensor]] = []

# With fault checks on (environment OSM_CHECK_FAULTS=1, or set_fault_check),
# every launch that uses a workspace is followed by a read of the workspace's
# fault word, which synchronises the host: a look-back wait that gave up (its
# launch's results are invalid) then raises instead of passing silently.
_check_faults = os.environ.get("OSM_CHECK_FAULTS", "0") not in ("", "0")


def set_fault_check(on: bool) -> bool:
    """Turns the per-launch fault check on or off; returns the old setting."""
    global _check_faults
    old, _check_faults = _check_faults, bool(on)
    return old


# Test aid: with timing jitter on, the forward, TTT, backward and table-forward
# scan launches carry OSM_FLAG_TIMING_JITTER (every workgroup sleeps a pseudo-random time
# before it publishes to the look-back); results must not change.
_timing_jitter = False


def set_timing_jitter(on: bool) -> bool:
    """Turns OSM_FLAG_TIMING_JITTER on or off for later launches; returns the old setting."""
    global _timing_jitter
    old, _timing_jitter = _timing_jitter, bool(on)
    return old


# Test aid: with the poll limit at zero, the forward, TTT, backward and
# table-forward scan launches carry OSM_FLAG_POLL_LIMIT_ZERO: a look-back wait whose word is not
# yet published gives up at once (the fault word is set and the outputs that
# depend on the missing value are NaN), as a wait that passes its poll limit
# does.
_poll_limit_zero = False


def set_poll_limit_zero(on: bool) -> bool:
    """Turns OSM_FLAG_POLL_LIMIT_ZERO on or off for later launches; returns the old setting."""
    global _poll_limit_zero
    old, _poll_limit_zero = _poll_limit_zero, bool(on)
    return old


def workspace_status(ws: torch.Tensor, *, reset: bool = False, stream: int | None = None) -> tuple[int, int]:
    """(fault word, launch counter) of a workspace, read on ``stream`` (the
    current stream of its device by default) through osm_workspace_status;
    synchronises the host.  A non-zero fault word is the fault tag of the
    last launch whose look-back wait gave up; ``reset`` clears it."""
    lib = nat.load()
    cur = _current_stream(ws.device)
    if stream is None:
        stream = cur
    # The status buffer is allocated on the current stream.  When the status
    # kernel runs on another stream, the current stream is drained first (its
    # earlier work may still use that memory) and the other stream after the
    # launch, so the read-back sees the kernel's values.
    st = torch.empty(2, dtype=torch.int32, device=ws.device)
    if stream != cur:
        torch.cuda.current_stream(ws.device).synchronize()
    nat.check(lib.osm_workspace_status(ctypes.c_void_p(ws.data_ptr()), ctypes.c_void_p(st.data_ptr()),
                                       1 if reset else 0, ctypes.c_void_p(stream)))
    if stream != cur:
        torch.cuda.ExternalStream(stream, device=ws.device).synchronize()
    fault, epoch = (int(v) & 0xFFFFFFFF for v in st.cpu().tolist())
    return fault, epoch


def workspace_faults(reset: bool = True) -> list[tuple[tuple[int, int, int], int]]:
    """Fault words of every workspace this module has created, as
    [((device, stream, op), fault word)] for the non-zero ones.  Each device
    is synchronised first and the words are read on its current stream (the
    stream a workspace was made for may no longer exist).  ``reset`` clears
    the words it reports."""
    with _ws_lock:
        items = list(_ws_cache.items()) + _ws_kept
    bad = []
    for key, ws in items:
        torch.cuda.synchronize(ws.device)
        fault, _ = workspace_status(ws, reset=reset)
        if fault:
            bad.append((key, fault))
    return bad


def _after_launch(ws: torch.Tensor, stream: int, what: str) -> None:
    if _check_faults:
        fault, epoch = workspace_status(ws, reset=True, stream=stream)
        if fault:
            raise nat.OsmError(nat.OSM_E_FAULT, f"{what}: a look-back wait gave up (fault word 0x{fault:08x}, "
                                                f"launch counter {epoch}); the results of that launch are invalid")


# The raw handle of a device's current stream: torch's C accessor when this
# torch has it (a tenth of the host time of building a Stream object, which
# shows on launches of small inputs), else the public API.
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _current_stream(dev: torch.device) -> int:
    if _raw_stream is not None:
        return _raw_stream(dev.index if dev.index is not None else torch.cuda.current_device())
    return torch.cuda.current_stream(dev).cuda_stream


# Whether the current stream of the current device is being captured, and that
# device (torch's C accessors where this torch has them, as above).
_current_capturing = getattr(torch._C, "_cuda_isCurrentStreamCapturing", torch.cuda.is_current_stream_capturing)
_current_device = getattr(torch._C, "_cuda_getDevice", torch.cuda.current_device)


def _capturing(dev: torch.device) -> bool:
    if dev.index is None or dev.index == _current_device():
        return _current_capturing()
    with torch.cuda.device(dev):
        return _current_capturing()


# The native launch path (csrc/osm_torch.cpp) and the library it was
# initialised for.  Its functions return None for what is not in the kernel's
# own form; the Python code below each call then converts, or raises.
_ext = None
_ext_for = None
_DTYPE_CODE = {None: None, torch.float32: nat.F32, torch.bfloat16: nat.BF16}


def _fast():
    """The native launch path, or None where the Python path has to run: with
    fault checks on, a library object that is not the loaded one, or without
    the extension."""
    global _ext, _ext_for
    lib = nat.load()
    if _ext_for is not lib:
        if _raw_stream is None or not isinstance(lib, ctypes.CDLL):
            return None
        ext = nat.load_ext()
        if ext is not None:
            ext.init(tuple(ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in nat.EXT_FUNCTIONS), _raw_stream,
                     _ws_cache, _workspace, nat.check)
        _ext, _ext_for = ext, lib
    return None if _check_faults else _ext


def _test_flags() -> int:
    return (nat.FLAG_TIMING_JITTER if _timing_jitter else 0) | (nat.FLAG_POLL_LIMIT_ZERO if _poll_limit_zero else 0)


def _flags(clamp: bool, nan_policy: str) -> int:
    if nan_policy not in ("zero_z", "zero_u"):
        raise ValueError("nan_policy must be 'zero_z' or 'zero_u'")
    return ((0 if clamp else nat.FLAG_NO_CLAMP) | (nat.FLAG_NAN_ZERO_U if nan_policy == "zero_u" else 0) |
            _test_flags())


def _workspace(device: torch.device, stream: int, nbytes: int, op: int) -> torch.Tensor:
    """Zero-initialised workspace reused per (device, stream, entry point).
    Calls on one stream are ordered, so they never overlap on a workspace;
    one workspace per entry point keeps its layout fixed across alternating
    forward/backward calls (a layout change costs a clear).

    A graph holds the address of the workspace that its capture used, so that
    one is never freed; the one that replaces it is at least twice its size, so
    those kept stay smaller together than the one in use.  A capture that finds
    none large enough gets memory of the graph, cleared in every replay."""
    key = (device.index, stream, op)
    capturing = _capturing(device)
    with _ws_lock:
        ws = _ws_cache.get(key)
        if ws is None or ws.numel() < nbytes:
            if capturing:
                return torch.zeros(nbytes, dtype=torch.uint8, device=device)
            size = max(nbytes, 1 << 20)
            if key in _ws_in_graph:
                _ws_in_graph.discard(key)
                _ws_kept.append((key, ws))
                size = max(size, 2 * ws.numel())
            size = (size + (1 << 20) - 1) & ~((1 << 20) - 1)
            ws = torch.zeros(size, dtype=torch.uint8, device=device)
            _ws_cache[key] = ws
        elif capturing:
            _ws_in_graph.add(key)
        return ws


def _as_param(v, H: int, device, name: str) -> torch.Tensor:
    if (isinstance(v, torch.Tensor) and v.dtype is torch.float32 and v.dim() == 1 and v.is_contiguous()
            and v.device == device):
        t = v   # already in the kernel's form: no conversion calls (host time per launch)
    else:
        t = v if isinstance(v, torch.Tensor) else torch.as_tensor(v, dtype=torch.float32)
        t = t.to(device=device, dtype=torch.float32).reshape(-1).contiguous()
    if t.numel() != H:
        raise ValueError(f"{name} must have H={H} entries, got {t.numel()}")
    return t


def _dtype_code(dt: torch.dtype) -> int:
    if dt == torch.float32:
        return nat.F32
    if dt == torch.bfloat16:
        return nat.BF16
    raise TypeError(f"unsupported dtype {dt}; use float32 or bfloat16")


def _prepare(x, coeffs, damping, lam, g, lam_shift, lam_min, lam_max, ema_init, clamp, out_dtype, out,
             nan_policy="zero_z", alloc_out=True):
    if not isinstance(x, torch.Tensor) or x.dim() != 3:
        raise ValueError("x must be a [B,S,D] tensor")
    if x.device.type != "cuda":
        raise RuntimeError("orthossm_amd runs on a ROCm GPU only; x is on " + str(x.device))
    dev = x.device
    if x.dtype not in (torch.float32, torch.bfloat16):
        x = x.float()
    if x.stride(2) != 1 or min(x.stride()) < 0:
        x = x.contiguous()
    B, S, D = x.shape
    if coeffs.dim() != 4:
        raise ValueError("coeffs must be [B,H,K,hd]")
    Bc, H, K, hd = coeffs.shape
    if Bc != B or H * hd != D:
        raise ValueError(f"coeffs {tuple(coeffs.shape)} does not match x {tuple(x.shape)}")
    c = coeffs if (coeffs.dtype is torch.float32 and coeffs.device == dev) else coeffs.to(device=dev,
                                                                                            dtype=torch.float32)
    if c.stride(3) != 1:
        c = c.contiguous()
    damp = _as_param(damping, H, dev, "damping")
    lamt = _as_param(lam, H, dev, "lam")
    gt = None
    if g is not None:
        gt = g.to(device=dev, dtype=torch.float32)
        if gt.dim() == 2:
            gt = gt.unsqueeze(0).expand(B, S, H)
        if tuple(gt.shape) != (B, S, H):
            raise ValueError(f"g must be [S,H] or [B,S,H], got {tuple(g.shape)}")
    init = None
    if ema_init is not None:
        init = ema_init.to(device=dev, dtype=torch.float32).reshape(B, D).contiguous()
    odt = x.dtype if out_dtype is None else out_dtype
    if out is None:
        if alloc_out:
            out = torch.empty((B, S, D), device=dev, dtype=odt)
    elif tuple(out.shape) != (B, S, D) or out.dtype != odt or out.device != dev:
        raise ValueError("out has the wrong shape, dtype or device")
    if out is not None and (out.stride(2) != 1 or min(out.stride()) < 0):
        raise ValueError("out must have a contiguous lane dimension and non-negative strides")
    a = nat.ChebyArgs()
    a.abi_version = nat.ABI_VERSION
    a.flags = _flags(clamp, nan_policy)
    a.B, a.S, a.H, a.hd, a.K = B, S, H, hd, K
    a.x, a.x_dtype, a.x_stride_b, a.x_stride_s = x.data_ptr(), _dtype_code(x.dtype), x.stride(0), x.stride(1)
    a.out_dtype = _dtype_code(odt)
    if out is not None:
        a.out = out.data_ptr()
        a.out_stride_b, a.out_stride_s = out.stride(0), out.stride(1)
    a.coeffs, a.c_stride_b, a.c_stride_h, a.c_stride_k = c.data_ptr(), c.stride(0), c.stride(1), c.stride(2)
    a.damping, a.lam = damp.data_ptr(), lamt.data_ptr()
    if gt is not None:
        a.g, a.g_stride_b, a.g_stride_s, a.g_stride_h = gt.data_ptr(), gt.stride(0), gt.stride(1), gt.stride(2)
    a.lam_shift, a.lam_min, a.lam_max = float(lam_shift), float(lam_min), float(lam_max)
    a.ema_init = init.data_ptr() if init is not None else None
    keep = (x, c, damp, lamt, gt, init)  # keeps every pointed-to tensor alive across the call
    return a, out, keep


def cheby_ema_forward(x: torch.Tensor, coeffs: torch.Tensor, damping: Sequence[float] | torch.Tensor,
                      lam: Sequence[float] | torch.Tensor, *, g: torch.Tensor | None = None,
                      lam_shift: float = 0.004, lam_min: float = 0.9, lam_max: float = 0.9999,
                      ema_init: torch.Tensor | None = None, clamp: bool = True,
                      out_dtype: torch.dtype | None = None, out: torch.Tensor | None = None,
                      return_state: bool = False, state_out: torch.Tensor | None = None,
                      nan_policy: str = "zero_z"):
    """Fused softsign -> Clenshaw -> damping -> tanh -> EMA on the GPU.

    x [B,S,D] fp32|bf16, coeffs [B,H,K,hd] fp32, damping/lam [H], g optional
    [S,H] or [B,S,H] (dynamic lambda), ema_init optional [B,D].
    Returns out [B,S,D] (dtype of x unless out_dtype), and ema_final [B,D]
    fp32 when return_state.  ``state_out`` (contiguous [B,D] fp32 on the
    device) receives ema_final instead of a new tensor.  ``nan_policy``: a
    NaN input gives z = 0 ('zero_z', the reference's Triton kernels) or counts
    as u = 0 ('zero_u', the reference's PyTorch fast path).
    """
    fast = _fast()
    if fast is not None and out_dtype in _DTYPE_CODE:
        res = fast.forward(x, coeffs, damping, lam, g, lam_shift, lam_min, lam_max, _flags(clamp, nan_policy), ema_init,
                           _DTYPE_CODE[out_dtype], out, return_state, state_out)
        if res is not None:
            return res if return_state else res[0]
    lib = nat.load()
    a, out, keep = _prepare(x, coeffs, damping, lam, g, lam_shift, lam_min, lam_max, ema_init, clamp,
                            out_dtype, out, nan_policy)
    dev = out.device
    ema_final = _state_buffer(a, dev, return_state, state_out)
    stream = _current_stream(dev)
    nbytes = lib.osm_workspace_bytes(ctypes.byref(a), 0)
    if nbytes == 0:
        nat.check(_rc_from_error(lib, a, 0))
    ws = _workspace(dev, stream, nbytes, nat.OP_FWD)
    nat.check(lib.osm_cheby_ema_fwd(ctypes.byref(a), ctypes.c_void_p(ws.data_ptr()), ws.numel(),
                                    ctypes.c_void_p(stream)))
    _after_launch(ws, stream, "osm_cheby_ema_fwd")
    del keep
    return (out, ema_final) if return_state else out


def cheby_ema_ttt(x: torch.Tensor, coeffs: torch.Tensor, damping, lam, *, g: torch.Tensor | None = None,
                  lam_shift: float = 0.004, lam_min: float = 0.9, lam_max: float = 0.9999,
                  ema_init: torch.Tensor | None = None, target: str = "x", clamp: bool = True,
                  out_dtype: torch.dtype | None = None, out: torch.Tensor | None = None,
                  return_state: bool = False, state_out: torch.Tensor | None = None,
                  grad_out: torch.Tensor | None = None, nan_policy: str = "zero_z"):
    """Fused forward plus the TTT coefficient gradient
    grad[b,h,k,j] = d/dc MSE(out[:, :-1], y[:, 1:]) / (k+1)^2, y = x ('x') or
    softsign(x) ('softsign').  Returns (out, grad) or (out, grad, ema_final).
    ``grad_out`` (contiguous [B,H,K,hd] fp32) and ``state_out`` receive the
    results instead of new tensors."""
    lib = nat.load()
    tgt = {"x": nat.TARGET_X, "softsign": nat.TARGET_SOFTSIGN}.get(target)
    if tgt is None:
        raise ValueError("target must be 'x' or 'softsign'")
    fast = _fast()
    if fast is not None and grad_out is None and out_dtype in _DTYPE_CODE:
        res = fast.ttt(x, coeffs, damping, lam, g, lam_shift, lam_min, lam_max, _flags(clamp, nan_policy), ema_init,
                       _DTYPE_CODE[out_dtype], out, return_state, state_out, tgt)
        if res is not None:
            return res if return_state else res[:2]
    a, out, keep = _prepare(x, coeffs, damping, lam, g, lam_shift, lam_min, lam_max, ema_init, clamp,
                            out_dtype, out, nan_policy)
    dev = out.device
    if grad_out is None:
        grad = torch.empty((a.B, a.H, a.K, a.hd), device=dev, dtype=torch.float32)
    else:
        _check_dest(grad_out, (a.B, a.H, a.K, a.hd), dev, "grad_out")
        grad = grad_out
    ema_final = _state_buffer(a, dev, return_state, state_out)
    stream = _current_stream(dev)
    nbytes = lib.osm_workspace_bytes(ctypes.byref(a), 1)
    if nbytes == 0:
        nat.check(_rc_from_error(lib, a, 1))
    ws = _workspace(dev, stream, nbytes, nat.OP_TTT)
    nat.check(lib.osm_cheby_ema_ttt(ctypes.byref(a), ctypes.c_void_p(grad.data_ptr()), tgt,
                                    ctypes.c_void_p(ws.data_ptr()), ws.numel(), ctypes.c_void_p(stream)))
    _after_launch(ws, stream, "osm_cheby_ema_ttt")
    del keep
    return (out, grad, ema_final) if return_state else (out, grad)


def cheby_ema_backward(x: torch.Tensor, coeffs: torch.Tensor, damping, lam, out: torch.Tensor | None,
                       grad_out: torch.Tensor, *, g: torch.Tensor | None = None, lam_shift: float = 0.004,
                       lam_min: float = 0.9, lam_max: float = 0.9999, grad_state: torch.Tensor | None = None,
                       clamp: bool = True, nan_policy: str = "zero_z", need_coeffs: bool = True,
                       need_init: bool = False, grad_x_out: torch.Tensor | None = None,
                       grad_coeffs_out: torch.Tensor | None = None, grad_init_out: torch.Tensor | None = None,
                       z_saved: torch.Tensor | None = None, full_jacobian: bool = False):
    """Backward of ``cheby_ema_forward``.

    ``out`` is the saved forward output (its clamp mask |out| < 1 - 1e-6
    gates the adjoint, as the reference's reverse scan does; it may be None
    with clamp=False), ``grad_out`` = dL/dout [B,S,D] and ``grad_state`` =
    dL/d ema_final [B,D] or None.  Returns (grad_x [B,S,D] in x's dtype,
    grad_coeffs [B,H,K,hd] fp32 or None, grad_init [B,D] fp32 or None).
    lambda and damping are treated as constants.  ``grad_x_out``,
    ``grad_coeffs_out`` and ``grad_init_out`` (contiguous, on the device)
    receive the results instead of new tensors.  ``z_saved`` (bf16 [B,S,D],
    the forward's z) makes the backward take 1 - z^2 from it, and
    ``full_jacobian`` uses 1/(1+|x|)^2 everywhere, as the reference's
    full-path backward does.
    """
    lib = nat.load()
    if out is None and clamp:
        raise ValueError("the saved forward output is needed for the clamp mask")
    fast = _fast()
    if fast is not None and z_saved is None and grad_x_out is None and grad_coeffs_out is None and \
            grad_init_out is None:
        res = fast.backward(x, coeffs, damping, lam, g, lam_shift, lam_min, lam_max,
                            _flags(clamp, nan_policy) | (nat.FLAG_FULL_JACOBIAN if full_jacobian else 0), out, grad_out,
                            grad_state, need_coeffs, need_init)
        if res is not None:
            return res
    a, _, keep = _prepare(x, coeffs, damping, lam, g, lam_shift, lam_min, lam_max, None, clamp,
                          out.dtype if out is not None else None, out, nan_policy, alloc_out=False)
    xin = keep[0]
    dev = xin.device
    B, S, D = a.B, a.S, a.H * a.hd
    out_dt = out.dtype if out is not None else xin.dtype
    go = grad_out.to(device=dev, dtype=out_dt)
    if tuple(go.shape) != (B, S, D):
        raise ValueError(f"grad_out must be [B,S,D]=({B},{S},{D}), got {tuple(grad_out.shape)}")
    if go.stride(2) != 1 or min(go.stride()) < 0:
        go = go.contiguous()
    if grad_x_out is None:
        gx = torch.empty((B, S, D), device=dev, dtype=xin.dtype)
    else:
        if tuple(grad_x_out.shape) != (B, S, D) or grad_x_out.dtype != xin.dtype or \
                grad_x_out.device != dev or not grad_x_out.is_contiguous():
            raise ValueError(f"grad_x_out must be a contiguous {xin.dtype} tensor of shape {(B, S, D)} on {dev}")
        gx = grad_x_out
    gc = gi = None
    if grad_coeffs_out is not None:
        _check_dest(grad_coeffs_out, (B, a.H, a.K, a.hd), dev, "grad_coeffs_out")
        gc = grad_coeffs_out
    elif need_coeffs:
        gc = torch.empty((B, a.H, a.K, a.hd), device=dev, dtype=torch.float32)
    if grad_init_out is not None:
        _check_dest(grad_init_out, (B, D), dev, "grad_init_out")
        gi = grad_init_out
    elif need_init:
        gi = torch.empty((B, D), device=dev, dtype=torch.float32)
    gs = None
    if grad_state is not None:
        gs = grad_state.to(device=dev, dtype=torch.float32).reshape(B, D).contiguous()
    bw = nat.BwdArgs()
    bw.grad_out, bw.go_stride_b, bw.go_stride_s = go.data_ptr(), go.stride(0), go.stride(1)
    bw.grad_state = gs.data_ptr() if gs is not None else None
    bw.grad_x, bw.gx_stride_b, bw.gx_stride_s = gx.data_ptr(), gx.stride(0), gx.stride(1)
    bw.grad_coeffs = gc.data_ptr() if gc is not None else None
    bw.grad_init = gi.data_ptr() if gi is not None else None
    if z_saved is not None:
        if tuple(z_saved.shape) != (B, S, D) or z_saved.dtype != torch.bfloat16 or z_saved.stride(2) != 1:
            raise ValueError("z_saved must be a bf16 [B,S,D] tensor with a contiguous lane dimension")
        bw.z_saved, bw.z_stride_b, bw.z_stride_s = z_saved.data_ptr(), z_saved.stride(0), z_saved.stride(1)
    if full_jacobian:
        a.flags |= nat.FLAG_FULL_JACOBIAN
    stream = _current_stream(dev)
    nbytes = lib.osm_workspace_bytes(ctypes.byref(a), nat.OP_BWD)
    if nbytes == 0:
        nat.check(lib.osm_cheby_ema_bwd(ctypes.byref(a), ctypes.byref(bw), None, 0, None))
    ws = _workspace(dev, stream, nbytes, nat.OP_BWD)
    nat.check(lib.osm_cheby_ema_bwd(ctypes.byref(a), ctypes.byref(bw), ctypes.c_void_p(ws.data_ptr()), ws.numel(),
                                    ctypes.c_void_p(stream)))
    _after_launch(ws, stream, "osm_cheby_ema_bwd")
    del keep, go, gs
    return gx, gc, gi


class _ChebyEMAFunction(torch.autograd.Function):
    """Differentiable forward: saves x, coeffs and the output; the backward
    is one ``osm_cheby_ema_bwd`` call."""

    @staticmethod
    def forward(ctx, x, coeffs, ema_init, damping, lam, g, lam_shift, lam_min, lam_max, clamp, out_dtype,
                nan_policy):
        ctx.set_materialize_grads(False)   # an unused output's gradient stays None
        out, fin = cheby_ema_forward(x, coeffs, damping, lam, g=g, lam_shift=lam_shift, lam_min=lam_min,
                                     lam_max=lam_max, ema_init=ema_init, clamp=clamp, out_dtype=out_dtype,
                                     return_state=True, nan_policy=nan_policy)
        ctx.save_for_backward(x, coeffs, out if clamp else None, g)
        ctx.params = (damping, lam, lam_shift, lam_min, lam_max, clamp, nan_policy)
        ctx.has_init = ema_init is not None
        return out, fin

    @staticmethod
    def backward(ctx, grad_out, grad_fin):
        x, coeffs, out, g = ctx.saved_tensors
        damping, lam, lam_shift, lam_min, lam_max, clamp, nan_policy = ctx.params
        need_x, need_c, need_i = ctx.needs_input_grad[0], ctx.needs_input_grad[1], ctx.needs_input_grad[2]
        if grad_out is None:
            grad_out = torch.zeros(x.shape, device=x.device, dtype=out.dtype if out is not None else x.dtype)
        gx, gc, gi = cheby_ema_backward(x, coeffs, damping, lam, out, grad_out, g=g, lam_shift=lam_shift,
                                        lam_min=lam_min, lam_max=lam_max, grad_state=grad_fin, clamp=clamp,
                                        nan_policy=nan_policy, need_coeffs=need_c, need_init=need_i)
        if need_x and gx.dtype != x.dtype:
            gx = gx.to(x.dtype)
        if need_c and gc.dtype != coeffs.dtype:
            gc = gc.to(coeffs.dtype)
        return (gx if need_x else None, gc, gi if ctx.has_init else None,
                None, None, None, None, None, None, None, None, None)


def cheby_ema(x: torch.Tensor, coeffs: torch.Tensor, damping, lam, *, g: torch.Tensor | None = None,
              lam_shift: float = 0.004, lam_min: float = 0.9, lam_max: float = 0.9999,
              ema_init: torch.Tensor | None = None, clamp: bool = True, out_dtype: torch.dtype | None = None,
              return_state: bool = False, nan_policy: str = "zero_z"):
    """``cheby_ema_forward`` as a differentiable op: gradients flow to x,
    coeffs and ema_init (lambda, g and damping are constants).  Returns out,
    or (out, ema_final) when return_state."""
    out, fin = _ChebyEMAFunction.apply(x, coeffs, ema_init, damping, lam, g, lam_shift, lam_min, lam_max, clamp,
                                       out_dtype, nan_policy)
    return (out, fin) if return_state else out


# Per-head Lion forget factors of the reference (MULTI_SCALE_LAMBDA,
# sdpc_kernel.py:1416); heads past the eighth use 0.995 (1429-1432).
V10_LION_LAMBDA = (0.9995, 0.9995, 0.997, 0.997, 0.995, 0.995, 0.97, 0.95)
# Half-table of the full path's LUT mode: points on [0, 1], terms T_0..T_7
# (sdpc_kernel.py:58-59).
LUT_POINTS = 256
LUT_TERMS = 8
_v10_lock = threading.Lock()
_v10_cache: dict = {}


def chebyshev_lut_table(points: int = LUT_POINTS, terms: int = LUT_TERMS) -> torch.Tensor:
    """[terms, points] fp32 CPU tensor: T_k on ``torch.linspace(0, 1, points)``
    by the three-term recurrence T_k = 2u T_{k-1} - T_{k-2} in fp32, the
    construction the kernels' table values must reproduce bit for bit
    (sdpc_kernel.py:63-81)."""
    grid = torch.linspace(0.0, 1.0, points)
    T = torch.zeros(terms, points)
    T[0] = 1.0
    if terms > 1:
        T[1] = grid
    for k in range(2, terms):
        T[k] = 2.0 * grid * T[k - 1] - T[k - 2]
    return T


def v10_tables(device: torch.device, n_heads: int, K: int):
    """(lut [8,256], lion_lambda [H], spectral_scale [K], lr_scale [H]) fp32 on
    ``device``: the Chebyshev table T_k(linspace(0, 1, 256)) built in fp32 by
    the recurrence (sdpc_kernel.py:63-81) and the Lion constants
    (sdpc_kernel.py:1423-1437).  Cached per (device, H, K)."""
    key = (device.type, device.index, n_heads, K)
    with _v10_lock:
        hit = _v10_cache.get(key)
        if hit is not None:
            return hit
        T = chebyshev_lut_table()
        n_active = min(n_heads, len(V10_LION_LAMBDA))
        lam = torch.tensor(list(V10_LION_LAMBDA[:n_active]) + [0.995] * max(0, n_heads - n_active))
        ss = 1.0 / (torch.arange(K, dtype=torch.float32) + 1.0) ** 1.5
        h = torch.arange(n_heads, dtype=torch.float32)
        lr_scale = 1.0 + 0.25 * (h - n_heads / 2.0) / max(n_heads, 1)
        hit = tuple(t.to(device=device, dtype=torch.float32).contiguous() for t in (T, lam, ss, lr_scale))
        _v10_cache[key] = hit
        return hit


def device_momentum(mu, dev: torch.device):
    """ema_momentum as (float, None), or, given a one-element tensor, as
    (0.0, that value in a [1] fp32 tensor on ``dev``): a momentum computed on
    the device stays there, with no host synchronisation."""
    if isinstance(mu, torch.Tensor):
        if mu.numel() != 1:
            raise ValueError(f"ema_momentum must be a number or a one-element tensor, got shape {tuple(mu.shape)}")
        return 0.0, mu.detach().to(device=dev, dtype=torch.float32).reshape(1).contiguous()
    return float(mu), None


def head_momentum(mu, n_heads: int, dev: torch.device) -> torch.Tensor:
    """[n_heads] fp32 on ``dev``, every entry the scalar momentum ``mu`` (a
    number or a one-element tensor, which is not read back to the host)."""
    val, t = device_momentum(mu, dev)
    if t is not None:
        return t.expand(n_heads).contiguous()
    return torch.full((n_heads,), val, dtype=torch.float32, device=dev)


def v10_chunked_ttt(x: torch.Tensor, coeffs: torch.Tensor, momentum: torch.Tensor, *, n_heads: int,
                    base_lr: float = 0.005, ema_momentum: float | torch.Tensor = 0.9, beta1: float = 0.9, beta2: float = 0.99,
                    weight_decay: float = 0.01, chunk_size: int = 256, gate_global: torch.Tensor | None = None,
                    dynamic_lambda: torch.Tensor | None = None, use_lut: bool = True,
                    save_for_backward: bool = False):
    """The reference's full apply_cheby_rkv_v10 path in one launch: chunks of
    ``chunk_size`` tokens, each with the coefficients and Lion momentum the
    previous chunk left (see osm_v10_args in include/osm.h).

    x [B,S,D] fp32|bf16, coeffs and momentum [B,H,K,hd] (cast to fp32; K > 8:
    coefficients past the eighth are returned unchanged, as the reference's
    kernel leaves them), gate_global / dynamic_lambda optional [B];
    ema_momentum a number or a one-element device tensor.  Returns
    (out [B,S,D] fp32 holding bf16 values, coeffs_new, momentum_new) and, with
    save_for_backward, also (z [B,S,D] bf16, coeff_hist [n_chunks,B,H,K,hd]).
    """
    lib = nat.load()
    fast = _fast()
    if fast is not None and isinstance(x, torch.Tensor) and x.is_cuda and isinstance(coeffs, torch.Tensor) and \
            coeffs.dim() == 4 and coeffs.shape[1] == n_heads:
        lut, lion_lambda, ss, lr_scale = v10_tables(x.device, n_heads, min(coeffs.shape[2], nat.MAX_K_V10))
        res = fast.v10(x, coeffs, momentum, n_heads, gate_global, dynamic_lambda, ema_momentum, lut, lion_lambda, ss,
                       lr_scale, base_lr, beta1, beta2, weight_decay, chunk_size, use_lut, save_for_backward)
        if res is not None:
            return res
    if not isinstance(x, torch.Tensor) or x.dim() != 3:
        raise ValueError("x must be a [B,S,D] tensor")
    if x.device.type != "cuda":
        raise RuntimeError("orthossm_amd runs on a ROCm GPU only; x is on " + str(x.device))
    if momentum is None:
        raise ValueError("the full path needs a momentum buffer [B,H,K,hd]")
    dev = x.device
    B, S, D = x.shape
    if S == 0:
        raise ValueError("the full path needs S >= 1")
    if x.dtype not in (torch.float32, torch.bfloat16):
        x = x.float()
    if x.stride(2) != 1:
        x = x.contiguous()
    c_full = coeffs.to(device=dev, dtype=torch.float32)
    m_full = momentum.to(device=dev, dtype=torch.float32)
    if c_full.dim() != 4 or c_full.shape[0] != B or c_full.shape[1] != n_heads or \
            c_full.shape[1] * c_full.shape[3] != D or m_full.shape != c_full.shape:
        raise ValueError(f"coeffs/momentum must be [B,H,K,hd] matching x {tuple(x.shape)} and n_heads={n_heads}")
    H, Kfull, hd = n_heads, c_full.shape[2], c_full.shape[3]
    K = min(Kfull, nat.MAX_K_V10)
    c = c_full[:, :, :K]
    m = m_full[:, :, :K]
    if c.stride(3) != 1:
        c = c.contiguous()
    if m.stride(3) != 1:
        m = m.contiguous()
    lut, lion_lambda, ss, lr_scale = v10_tables(dev, H, K)
    out = torch.empty((B, S, D), device=dev, dtype=torch.float32)
    c_out = torch.empty((B, H, K, hd), device=dev, dtype=torch.float32)
    m_out = torch.empty_like(c_out)
    gate = None if gate_global is None else gate_global.to(device=dev, dtype=torch.float32).reshape(B).contiguous()
    dyn = None if dynamic_lambda is None else \
        dynamic_lambda.to(device=dev, dtype=torch.float32).reshape(B).contiguous()
    n_chunks = (S + chunk_size - 1) // chunk_size
    z = hist = None
    if save_for_backward:
        z = torch.empty((B, S, D), device=dev, dtype=torch.bfloat16)
        hist = torch.empty((n_chunks, B, H, K, hd), device=dev, dtype=torch.float32)
    a = nat.V10Args()
    a.abi_version = nat.ABI_VERSION
    a.flags = nat.V10_USE_LUT if use_lut else 0
    a.B, a.S, a.H, a.hd, a.K, a.chunk = B, S, H, hd, K, int(chunk_size)
    a.x, a.x_dtype, a.x_stride_b, a.x_stride_s = x.data_ptr(), _dtype_code(x.dtype), x.stride(0), x.stride(1)
    a.out, a.out_stride_b, a.out_stride_s = out.data_ptr(), out.stride(0), out.stride(1)
    a.coeffs, a.c_stride_b, a.c_stride_h, a.c_stride_k = c.data_ptr(), c.stride(0), c.stride(1), c.stride(2)
    a.momentum, a.m_stride_b, a.m_stride_h, a.m_stride_k = m.data_ptr(), m.stride(0), m.stride(1), m.stride(2)
    a.coeffs_out, a.momentum_out = c_out.data_ptr(), m_out.data_ptr()
    a.lut, a.lion_lambda, a.lr_scale, a.spectral_scale = lut.data_ptr(), lion_lambda.data_ptr(), \
        lr_scale.data_ptr(), ss.data_ptr()
    a.gate = gate.data_ptr() if gate is not None else None
    a.dyn_lambda = dyn.data_ptr() if dyn is not None else None
    mu_val, mu_dev = device_momentum(ema_momentum, dev)
    a.ema_momentum, a.base_lr, a.beta1, a.beta2, a.weight_decay = (mu_val, float(base_lr),
                                                                   float(beta1), float(beta2), float(weight_decay))
    a.ema_momentum_dev = mu_dev.data_ptr() if mu_dev is not None else None
    if z is not None:
        a.z_save, a.z_stride_b, a.z_stride_s = z.data_ptr(), z.stride(0), z.stride(1)
        a.coeff_hist = hist.data_ptr()
    stream = _current_stream(dev)
    nat.check(lib.osm_v10_chunked_ttt(ctypes.byref(a), ctypes.c_void_p(stream)))
    keep = (x, c, m, gate, dyn, mu_dev)  # noqa: F841  (alive until the launch is queued)
    if Kfull > K:
        c_out = torch.cat([c_out, c_full[:, :, K:]], dim=2)
        m_out = torch.cat([m_out, m_full[:, :, K:]], dim=2)
    if save_for_backward:
        return out, c_out, m_out, z, hist
    return out, c_out, m_out


def engine_prologue(x: torch.Tensor, norm_weight: torch.Tensor, eps: float, w1: torch.Tensor, b1: torch.Tensor,
                    w2: torch.Tensor, b2: torch.Tensor, ema_base: torch.Tensor, tokens_seen: torch.Tensor):
    """The engine's input norm, complexity gate and momentum schedule
    (sdpc_engine.py:163-209) in two launches, without gradients; tokens_seen
    (int64 scalar) is advanced by S in place.  x [B,S,D] fp32 and the weights
    fp32 contiguous on x's device, D a multiple of 4 up to ENGINE_MAX_D.
    Returns (x_normed [B,S,D], gate [B,1], mu, a 0-d tensor)."""
    fast = _fast()
    if fast is not None:
        res = fast.engine(x, norm_weight, eps, w1, b1, w2, b2, ema_base, tokens_seen)
        if res is not None:
            return res
    lib = nat.load()
    if x.dim() != 3 or x.dtype != torch.float32 or x.device.type != "cuda" or x.stride(2) != 1 or x.numel() == 0:
        raise ValueError("x must be a non-empty [B,S,D] float32 tensor on a ROCm device with lane stride 1")
    dev = x.device
    B, S, D = x.shape
    for name, t, n in (("norm_weight", norm_weight, D), ("w1", w1, D // 4 * D), ("b1", b1, D // 4), ("w2", w2, D // 4),
                       ("b2", b2, 1), ("ema_base", ema_base, 1)):
        if t.numel() != n:
            raise ValueError(f"{name} must have {n} entries, got {t.numel()}")
        _check_dest(t, t.shape, dev, name)
    if tokens_seen.dtype != torch.int64 or tokens_seen.numel() != 1 or tokens_seen.device != dev:
        raise ValueError(f"tokens_seen must be an int64 scalar on {dev}")
    xn = torch.empty((B, S, D), device=dev, dtype=torch.float32)
    scratch = torch.empty(lib.osm_engine_scratch_bytes(B, S, D) // 4, device=dev, dtype=torch.float32)
    gate = torch.empty((B, 1), device=dev, dtype=torch.float32)
    mu = torch.empty((), device=dev, dtype=torch.float32)
    a = nat.EngineArgs()
    a.abi_version, a.eps = nat.ABI_VERSION, float(eps)
    a.B, a.S, a.D = B, S, D
    a.x, a.x_stride_b, a.x_stride_s = x.data_ptr(), x.stride(0), x.stride(1)
    a.norm_weight, a.w1, a.b1 = norm_weight.data_ptr(), w1.data_ptr(), b1.data_ptr()
    a.w2, a.b2, a.ema_base, a.tokens_seen = w2.data_ptr(), b2.data_ptr(), ema_base.data_ptr(), tokens_seen.data_ptr()
    a.x_normed, a.gate, a.ema_momentum, a.scratch = xn.data_ptr(), gate.data_ptr(), mu.data_ptr(), scratch.data_ptr()
    nat.check(lib.osm_engine_prologue(ctypes.byref(a), ctypes.c_void_p(_current_stream(dev))))
    return xn, gate, mu


def _rows_dest(t: torch.Tensor | None, shape, dev, name: str) -> torch.Tensor | None:
    """A caller's [B,S,D] or [B,D] fp32 output with lane stride 1, or None."""
    if t is None:
        return None
    if t.shape != torch.Size(shape) or t.dtype != torch.float32 or t.device != dev or t.stride(-1) != 1:
        raise ValueError(f"{name} must be a {tuple(shape)} float32 tensor on {dev} with lane stride 1")
    return t


def cheby_ema_lut_forward(x: torch.Tensor, coeffs: torch.Tensor, *, n_heads: int, ema_momentum: float = 0.9,
                          ema_init: torch.Tensor | None = None, use_lut: bool = True, lut: torch.Tensor | None = None,
                          clamp_tile: int = 128, out: torch.Tensor | None = None,
                          x_norm: torch.Tensor | None = None, tanh_y: torch.Tensor | None = None,
                          ema_final: torch.Tensor | None = None, want_x_norm: bool = True,
                          want_tanh_y: bool = True):
    """The reference's _fused_clenshaw_ema_kernel (sdpc_kernel.py:988-1209)
    through osm_cheby_ema_lut_fwd: per lane, x_norm = softsign(x) (x as
    given, NaN read as 0), y = LUT or Clenshaw series of the fixed
    coefficients, tanh_y = tanh(clamp((0.98 - 0.06 h/H) y, -4, 4)), and the
    EMA s = mu s + (1 - mu) tanh_y from ema_init, out = clamp(s, -1, 1), with
    the carried state clamped every ``clamp_tile`` tokens (the kernel's
    BLOCK_S).  x [B,S,D] fp32|bf16, coeffs [B,H,K<=8,hd], ema_init [B,D] or
    None (0).  ``lut`` is the [8,256] table (the module's own by default).
    Returns (out, x_norm, tanh_y, ema_final) fp32; x_norm / tanh_y are None
    when not wanted and no buffer is given.  ``out``, ``x_norm``, ``tanh_y``
    and ``ema_final`` may be caller buffers (lane stride 1)."""
    lib = nat.load()
    if not isinstance(x, torch.Tensor) or x.dim() != 3:
        raise ValueError("x must be a [B,S,D] tensor")
    if x.device.type != "cuda":
        raise RuntimeError("orthossm_amd runs on a ROCm GPU only; x is on " + str(x.device))
    dev = x.device
    capturing = _capturing(dev)
    fast = None if capturing else _fast()
    if fast is not None and lut is None and out is None and x_norm is None and tanh_y is None and \
            ema_final is None and coeffs.dim() == 4 and coeffs.shape[1] == n_heads:
        table = v10_tables(dev, n_heads, LUT_TERMS)[0] if use_lut else None
        res = fast.lut_forward(x, coeffs, n_heads, ema_momentum, ema_init,
                               (nat.V10_USE_LUT if use_lut else 0) | _test_flags(), table, clamp_tile, want_x_norm,
                               want_tanh_y)
        if res is not None:
            return res
    B, S, D = x.shape
    if x.dtype not in (torch.float32, torch.bfloat16):
        x = x.float()
    if x.stride(2) != 1:
        x = x.contiguous()
    c = coeffs.to(device=dev, dtype=torch.float32)
    H = n_heads
    if c.dim() != 4 or c.shape[0] != B or c.shape[1] != H or H * c.shape[3] != D:
        raise ValueError(f"coeffs must be [B,H,K,hd] matching x {tuple(x.shape)} and n_heads={H}")
    K, hd = c.shape[2], c.shape[3]
    if not 1 <= K <= 8:
        raise ValueError(f"the fused Clenshaw/LUT forward takes 1 to 8 coefficients, got {K}")
    if c.stride(3) != 1:
        c = c.contiguous()
    if use_lut:
        lut = (v10_tables(dev, H, K)[0] if lut is None
               else lut.to(device=dev, dtype=torch.float32).reshape(LUT_TERMS, LUT_POINTS).contiguous())
    init = None
    if ema_init is not None:
        init = ema_init.to(device=dev, dtype=torch.float32).reshape(B, D)
        if init.stride(1) != 1:
            init = init.contiguous()
    out = _rows_dest(out, (B, S, D), dev, "out")
    if out is None:
        out = torch.empty((B, S, D), device=dev, dtype=torch.float32)
    x_norm = _rows_dest(x_norm, (B, S, D), dev, "x_norm")
    if x_norm is None and want_x_norm:
        x_norm = torch.empty((B, S, D), device=dev, dtype=torch.float32)
    tanh_y = _rows_dest(tanh_y, (B, S, D), dev, "tanh_y")
    if tanh_y is None and want_tanh_y:
        tanh_y = torch.empty((B, S, D), device=dev, dtype=torch.float32)
    ema_final = _rows_dest(ema_final, (B, D), dev, "ema_final")
    if ema_final is None:
        ema_final = torch.empty((B, D), device=dev, dtype=torch.float32)
    a = nat.LutFwdArgs()
    a.abi_version = nat.ABI_VERSION
    a.flags = nat.V10_USE_LUT if use_lut else 0
    a.B, a.S, a.H, a.hd, a.K, a.clamp_tile = B, S, H, hd, K, int(clamp_tile)
    a.x, a.x_dtype, a.x_stride_b, a.x_stride_s = x.data_ptr(), _dtype_code(x.dtype), x.stride(0), x.stride(1)
    a.coeffs, a.c_stride_b, a.c_stride_h, a.c_stride_k = c.data_ptr(), c.stride(0), c.stride(1), c.stride(2)
    a.lut = lut.data_ptr() if use_lut else None
    a.ema_momentum = float(ema_momentum)
    if init is not None:
        a.ema_init, a.init_stride_b = init.data_ptr(), init.stride(0)
    a.out, a.out_stride_b, a.out_stride_s = out.data_ptr(), out.stride(0), out.stride(1)
    if x_norm is not None:
        a.x_norm, a.xn_stride_b, a.xn_stride_s = x_norm.data_ptr(), x_norm.stride(0), x_norm.stride(1)
    if tanh_y is not None:
        a.tanh_y, a.ty_stride_b, a.ty_stride_s = tanh_y.data_ptr(), tanh_y.stride(0), tanh_y.stride(1)
    a.ema_final, a.final_stride_b = ema_final.data_ptr(), ema_final.stride(0)
    stream = _current_stream(dev)
    # A capture takes the walk over the tiles, which needs no workspace.
    nbytes = 0 if capturing else lib.osm_lut_fwd_workspace_bytes(ctypes.byref(a))
    if nbytes:
        a.flags |= _test_flags()
        ws = _workspace(dev, stream, nbytes, nat.OP_LUT)
        nat.check(lib.osm_cheby_ema_lut_fwd_ws(ctypes.byref(a), ctypes.c_void_p(ws.data_ptr()), ws.numel(),
                                               ctypes.c_void_p(stream)))
        _after_launch(ws, stream, "osm_cheby_ema_lut_fwd_ws")
    else:
        nat.check(lib.osm_cheby_ema_lut_fwd(ctypes.byref(a), ctypes.c_void_p(stream)))
    keep = (x, c, lut, init)  # noqa: F841  (alive until the launch is queued)
    return out, x_norm, tanh_y, ema_final


def _rows(t: torch.Tensor, dtype: torch.dtype, dev: torch.device) -> torch.Tensor:
    """``t`` as [B,S,D] rows the kernels address: ``dtype`` on ``dev``, lane
    stride 1, non-negative strides of at most 2^20 elements a token."""
    if t.dtype is not dtype or t.device != dev:
        t = t.to(device=dev, dtype=dtype)
    if t.stride(2) != 1 or not 0 <= t.stride(1) <= 1 << 20 or t.stride(0) < 0:
        t = t.contiguous()
    return t


def _v10_backward(x, out, z, hist, grad_out, n_heads, ema_momentum, chunk, need_coeffs):
    """The full path's backward (FusedChebyRKVv10.backward, sdpc_kernel.py:
    2436-2515) on every chunk: the adjoint restarts at each chunk end, the
    chunk's own coefficients enter, 1 - z^2 comes from the saved bf16 z, the
    mask from the output, dL/dx = ... / (1+|x|)^2.  One osm_v10_bwd launch;
    dL/dc (one chunk only) comes from osm_cheby_ema_bwd.  Returns (grad_x,
    grad_coeffs of the first chunk or None)."""
    B, S, D = x.shape
    n_chunks, _, H, K, hd = hist.shape
    dev = x.device
    if need_coeffs:
        h = torch.arange(H, dtype=torch.float32, device=dev)
        damping = (0.98 - 0.06 * h / H).contiguous()
        gx, gc, _ = cheby_ema_backward(x.contiguous(), hist[0], damping, head_momentum(ema_momentum, H, dev), out,
                                       grad_out.to(dtype=torch.float32).contiguous(), clamp=True,
                                       nan_policy="zero_u", z_saved=z, full_jacobian=True)
        return gx, gc
    fast = _fast()
    if fast is not None:
        gx = fast.v10_backward(x, out, z, hist, grad_out, ema_momentum, chunk)
        if gx is not None:
            return gx, None
    lib = nat.load()
    xr = _rows(x, x.dtype if x.dtype in (torch.float32, torch.bfloat16) else torch.float32, dev)
    go, out, z = _rows(grad_out, torch.float32, dev), _rows(out, torch.float32, dev), _rows(z, torch.bfloat16, dev)
    hist = hist.contiguous()
    gx = torch.empty((B, S, D), device=dev, dtype=xr.dtype)
    a = nat.V10BwdArgs()
    a.abi_version, a.x_dtype = nat.ABI_VERSION, _dtype_code(xr.dtype)
    a.B, a.S, a.H, a.hd, a.K, a.chunk = B, S, H, hd, K, int(chunk)
    a.x, a.x_stride_b, a.x_stride_s = xr.data_ptr(), xr.stride(0), xr.stride(1)
    a.grad_out, a.go_stride_b, a.go_stride_s = go.data_ptr(), go.stride(0), go.stride(1)
    a.out, a.out_stride_b, a.out_stride_s = out.data_ptr(), out.stride(0), out.stride(1)
    a.z_saved, a.z_stride_b, a.z_stride_s = z.data_ptr(), z.stride(0), z.stride(1)
    a.coeff_hist = hist.data_ptr()
    a.grad_x, a.gx_stride_b, a.gx_stride_s = gx.data_ptr(), gx.stride(0), gx.stride(1)
    mu_val, mu_dev = device_momentum(ema_momentum, dev)
    a.ema_momentum = mu_val
    a.ema_momentum_dev = mu_dev.data_ptr() if mu_dev is not None else None
    nat.check(lib.osm_v10_bwd(ctypes.byref(a), ctypes.c_void_p(_current_stream(dev))))
    keep = (xr, go, out, z, hist, mu_dev)  # noqa: F841  (alive until the launch is queued)
    return gx, None


class _V10FullFn(torch.autograd.Function):
    """The full path with the reference's backward: dL/dx always, dL/dc when
    the sequence is one chunk (the chunk loop detaches the coefficients,
    sdpc_kernel.py:2593-2594)."""

    @staticmethod
    def forward(ctx, x, coeffs, momentum, kw):
        ctx.set_materialize_grads(False)   # no gradient flows through the Lion state
        out, c_new, m_new, z, hist = v10_chunked_ttt(x, coeffs, momentum, save_for_backward=True, **kw)
        ctx.save_for_backward(x, out, z, hist)
        ctx.kw = kw
        ctx.c_meta = (coeffs.dtype, coeffs.shape)
        return out, c_new, m_new

    @staticmethod
    def backward(ctx, grad_out, grad_c_new, grad_m_new):
        x, out, z, hist = ctx.saved_tensors
        kw = ctx.kw
        need_c = ctx.needs_input_grad[1] and hist.shape[0] == 1
        if grad_out is None:
            grad_out = torch.zeros_like(out)
        gx, gc = _v10_backward(x, out, z, hist, grad_out, kw["n_heads"], kw["ema_momentum"],
                               min(kw["chunk_size"], x.shape[1]), need_c)
        gx = gx.to(x.dtype) if ctx.needs_input_grad[0] else None
        if need_c:
            dt, shape = ctx.c_meta
            if shape[2] > gc.shape[2]:
                gc = torch.cat([gc, gc.new_zeros(shape[0], shape[1], shape[2] - gc.shape[2], shape[3])], dim=2)
            gc = gc.to(dt)
        else:
            gc = None
        return gx, gc, None, None


def v10_full_path(x, coeffs, momentum, *, n_heads: int, base_lr: float = 0.005, ema_momentum: float = 0.9,
                  beta1: float = 0.9, beta2: float = 0.99, weight_decay: float = 0.01, chunk_size: int = 256,
                  gate_global=None, dynamic_lambda=None, use_lut: bool = True):
    """``v10_chunked_ttt`` as a differentiable op with the reference's
    backward of the full path.  Returns (out, coeffs_new, momentum_new)."""
    kw = dict(n_heads=n_heads, base_lr=base_lr, ema_momentum=ema_momentum, beta1=beta1, beta2=beta2,
              weight_decay=weight_decay, chunk_size=chunk_size, gate_global=gate_global,
              dynamic_lambda=dynamic_lambda, use_lut=use_lut)
    if x.dim() == 3 and x.shape[1] > chunk_size:
        coeffs = coeffs.detach()
    return _V10FullFn.apply(x, coeffs, momentum, kw)


def _check_dest(t: torch.Tensor, shape, dev, name: str) -> None:
    if t.dtype != torch.float32 or tuple(t.shape) != tuple(shape) or t.device != dev or not t.is_contiguous():
        raise ValueError(f"{name} must be a contiguous float32 tensor of shape {tuple(shape)} on {dev}")


def _state_buffer(a, dev, return_state: bool, state_out: torch.Tensor | None):
    """ema_final destination: state_out if given, a new [B,D] tensor if
    return_state, else none (the kernel then skips the store)."""
    if state_out is not None:
        _check_dest(state_out, (a.B, a.H * a.hd), dev, "state_out")
        buf = state_out
    elif return_state:
        buf = torch.empty((a.B, a.H * a.hd), device=dev, dtype=torch.float32)
    else:
        buf = None
    a.ema_final = buf.data_ptr() if buf is not None else None
    return buf


def _rc_from_error(lib, a, ttt: int) -> int:
    """osm_workspace_bytes returned 0: re-run validation through the entry
    point with no workspace to obtain the status code and message."""
    if ttt:
        return lib.osm_cheby_ema_ttt(ctypes.byref(a), None, 0, None, 0, None)
    return lib.osm_cheby_ema_fwd(ctypes.byref(a), None, 0, None)
