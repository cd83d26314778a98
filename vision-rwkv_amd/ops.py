"""Operator boundary: the reference's autograd Functions and RUN_* entry points, backed by
libvrwkv_hip.so.

Mirrors
  WKV / RUN_CUDA(w,u,k,v)                 classification/mmcls_custom/models/backbones/vrwkv.py:29-65
  legacy RUN_CUDA(B,T,C,w,u,k,v)          classification/mae/vrwkv/vrwkv.py:30-90
  WKV_6 / RUN_CUDA_RWKV6(B,T,C,H,r,k,v,w,u)  classification/mmcls_custom/models/backbones/vrwkv6.py:34-73
with the same argument meaning, output dtype rule and error behaviour (RuntimeError for
non-device / non-contiguous tensors).
"""
import ctypes

import torch

from . import _lib

_DT = {torch.float32: _lib.VRWKV_F32, torch.bfloat16: _lib.VRWKV_BF16, torch.float16: _lib.VRWKV_F16}


def _check_input(x, name):
    # CHECK_INPUT of bi_wkv.cpp:6-8
    if not x.is_cuda:
        raise RuntimeError(f"{name} must be a CUDA tensor")
    if not x.is_contiguous():
        raise RuntimeError(f"{name} must be contiguous")


def _check_out(t, name, shape, dtype, like):
    """A caller-allocated result (the legacy / wkv6 extension interfaces pass them in)."""
    if not (t.is_cuda and t.is_contiguous() and t.device == like.device):
        raise RuntimeError(f"{name} must be a contiguous CUDA tensor on the inputs' device")
    if tuple(t.shape) != tuple(shape) or t.dtype != dtype:
        raise RuntimeError(f"{name} must have shape {tuple(shape)} and dtype {dtype}")
    return t


def _stream_ptr(device):
    # the handle itself: building a Stream object around it takes 2 us of every call
    return torch._C._cuda_getCurrentRawStream(device.index)


class _on:
    """torch.cuda.device for a tensor's device, without the look-up of device arguments of other kinds."""
    __slots__ = ("index", "previous")

    def __init__(self, device):
        self.index = device.index

    def __enter__(self):
        self.previous = torch._C._cuda_exchangeDevice(self.index)

    def __exit__(self, *exc):
        torch._C._cuda_maybeExchangeDevice(self.previous)
        return False


def bi_wkv_forward(w, u, k, v, out=None, gate=None):
    """Extension-level entry (bi_wkv.cpp:23-33): w,u (C,) fp32; k,v (B,T,C) of one dtype
    (fp32, bf16 or fp16); returns y (B,T,C) of that dtype.  State and arithmetic are fp32.
    out: a caller-allocated y (the legacy interface, wkv_op.cpp:6-8).
    gate: None, or the receptance r (B,T,C) of the same dtype: the result is sigmoid(r) * y, the step that follows the
    operator in VRWKV_SpatialMix.forward (vrwkv.py:185-186 without key_norm), applied before y is stored
    (vrwkv_biwkv_fwd_gate; forward only: it has no autograd)."""
    for t, n in ((w, "w"), (u, "u"), (k, "k"), (v, "v")) + (((gate, "gate"),) if gate is not None else ()):
        _check_input(t, n)
    if k.dim() != 3 or v.shape != k.shape or (gate is not None and (gate.shape != k.shape or gate.dtype != k.dtype)):
        raise RuntimeError("k and v (and the gate) must all be (B,T,C) of one dtype")
    B, T, C = k.shape
    if w.numel() != C or u.numel() != C:
        raise RuntimeError("w and u must have C elements")
    if w.dtype != torch.float32 or u.dtype != torch.float32:
        raise RuntimeError("w and u must be float32")
    if k.dtype not in _DT or v.dtype != k.dtype:
        raise RuntimeError("k and v must share one of float32 / bfloat16 / float16")
    L = _lib.lib()
    dt = _DT[k.dtype]
    y = torch.empty_like(k) if out is None else _check_out(out, "y", k.shape, k.dtype, k)
    if y.numel() == 0:
        return y
    ws_bytes = L.vrwkv_biwkv_fwd_workspace_bytes(B, T, C, dt)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=k.device) if ws_bytes else None
    with _on(k.device):
        tail = (B, T, C, dt, ws.data_ptr() if ws is not None else None, ws_bytes, _stream_ptr(k.device))
        if gate is None:
            _lib.check(L.vrwkv_biwkv_fwd(w.data_ptr(), u.data_ptr(), k.data_ptr(), v.data_ptr(), y.data_ptr(), *tail))
        else:
            _lib.check(L.vrwkv_biwkv_fwd_gate(w.data_ptr(), u.data_ptr(), k.data_ptr(), v.data_ptr(), gate.data_ptr(),
                                              y.data_ptr(), *tail))
    return y


def bi_wkv_backward(w, u, k, v, gy, out=None, like_inputs=False):
    """Extension-level entry (bi_wkv.cpp:35-47): w,u (C,) fp32; k,v,gy (B,T,C) of one dtype;
    returns [gw, gu, gk, gv] with gw, gu (C,) fp32 summed over batch and tokens and gk, gv of the
    dtype of k.  out: caller-allocated (gw, gu, gk, gv).  like_inputs: gw, gu of the dtype of k as well, rounded from the
    fp32 sums by the kernel.  A sample's gk and gv are the same whatever else is in the call, but for the last bits of fp32 ones of more than
    224 tokens: how those are cut goes by the number of samples and channels too."""
    for t, n in ((w, "w"), (u, "u"), (k, "k"), (v, "v"), (gy, "gy")):
        _check_input(t, n)
    if k.dim() != 3 or v.shape != k.shape or gy.shape != k.shape:
        raise RuntimeError("k, v and gy must all be (B,T,C)")
    B, T, C = k.shape
    if w.numel() != C or u.numel() != C or w.dtype != torch.float32 or u.dtype != torch.float32:
        raise RuntimeError("w and u must be float32 with C elements")
    if k.dtype not in _DT or v.dtype != k.dtype or gy.dtype != k.dtype:
        raise RuntimeError("k, v and gy must share one of float32 / bfloat16 / float16")
    L = _lib.lib()
    dt = _DT[k.dtype]
    if out is None:
        gw = torch.empty(C, dtype=k.dtype if like_inputs else torch.float32, device=k.device)
        gu = torch.empty_like(gw)
        gk = torch.empty_like(k)
        gv = torch.empty_like(k)
    else:
        gw, gu = (_check_out(t, n, (C,), torch.float32, k) for t, n in zip(out[:2], ("gw", "gu")))
        gk, gv = (_check_out(t, n, k.shape, k.dtype, k) for t, n in zip(out[2:], ("gk", "gv")))
    if k.numel() == 0:
        return [gw.zero_(), gu.zero_(), gk, gv]
    ws_bytes = L.vrwkv_biwkv_bwd_workspace_bytes(B, T, C, dt)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=k.device)
    with _on(k.device):
        fn = L.vrwkv_biwkv_bwd_like if like_inputs and out is None else L.vrwkv_biwkv_bwd
        _lib.check(fn(w.data_ptr(), u.data_ptr(), k.data_ptr(), v.data_ptr(), gy.data_ptr(),
                      gw.data_ptr(), gu.data_ptr(), gk.data_ptr(), gv.data_ptr(),
                      B, T, C, dt, ws.data_ptr(), ws_bytes, _stream_ptr(k.device)))
    return [gw, gu, gk, gv]


def _wkv_forward(w, u, k, v, factor=1.0):
    """bi_wkv_forward with w and u of one type as they are, times factor in that type (vrwkv_biwkv_fwd_as)."""
    for t, n in ((w, "w"), (u, "u"), (k, "k"), (v, "v")):
        _check_input(t, n)
    if k.dim() != 3 or v.shape != k.shape:
        raise RuntimeError("k and v must all be (B,T,C) of one dtype")
    B, T, C = k.shape
    if w.numel() != C or u.numel() != C:
        raise RuntimeError("w and u must have C elements")
    if k.dtype not in _DT or v.dtype != k.dtype:
        raise RuntimeError("k and v must share one of float32 / bfloat16 / float16")
    L = _lib.lib()
    dt = _DT[k.dtype]
    y = torch.empty_like(k)
    if y.numel() == 0:
        return y
    ws_bytes = L.vrwkv_biwkv_fwd_workspace_bytes(B, T, C, dt)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=k.device) if ws_bytes else None
    with _on(k.device):
        _lib.check(L.vrwkv_biwkv_fwd_as(w.data_ptr(), u.data_ptr(), _DT[w.dtype], factor, k.data_ptr(), v.data_ptr(), y.data_ptr(), B, T, C, dt,
                                        ws.data_ptr() if ws is not None else None, ws_bytes, _stream_ptr(k.device)))
    return y


def _wkv_backward(w, u, k, v, gy, factor=1.0):
    """The gradients of _wkv_forward, gw and gu of the type of w (vrwkv_biwkv_bwd_as)."""
    gw, gu, gk, gv = torch.empty_like(w), torch.empty_like(u), torch.empty_like(k), torch.empty_like(k)
    if gy.shape != k.shape or gy.dtype != k.dtype:
        raise RuntimeError("gy must have the shape and dtype of k")
    if k.numel() == 0:
        return gw.zero_(), gu.zero_(), gk, gv
    B, T, C = k.shape
    L = _lib.lib()
    dt = _DT[k.dtype]
    ws_bytes = L.vrwkv_biwkv_bwd_workspace_bytes(B, T, C, dt)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=k.device)
    with _on(k.device):
        _lib.check(L.vrwkv_biwkv_bwd_as(w.data_ptr(), u.data_ptr(), _DT[w.dtype], factor, k.data_ptr(), v.data_ptr(), gy.data_ptr(), gw.data_ptr(),
                                        gu.data_ptr(), gk.data_ptr(), gv.data_ptr(), B, T, C, dt, ws.data_ptr(), ws_bytes, _stream_ptr(k.device)))
    return gw, gu, gk, gv


class WKV(torch.autograd.Function):
    """Bi-WKV with the reference's dtype rule: arithmetic in fp32, the result is fp32 unless
    the *parameter* w is half / bfloat16, in which case it has w's dtype (vrwkv.py:31-44).
    When k and v already arrive in that 16-bit dtype they are consumed as they are
    (no up-cast copies, no separate down-cast of y), and w and u as well when they share a type."""

    @staticmethod
    def forward(ctx, w, u, k, v):
        out_dtype = w.dtype if w.dtype in (torch.half, torch.bfloat16) else torch.float32
        ctx.out_dtype = out_dtype
        ctx.as_held = w.dtype == u.dtype == k.dtype == v.dtype == out_dtype
        if ctx.as_held:
            wc, uc = w.contiguous(), u.contiguous()
            ctx.save_for_backward(wc, uc, k, v)
            return _wkv_forward(wc, uc, k.contiguous(), v.contiguous())
        wf = w.float().contiguous()
        uf = u.float().contiguous()
        ctx.save_for_backward(wf, uf, k, v)                # the fp32 copies serve the backward too
        if k.dtype == out_dtype and v.dtype == out_dtype:
            return bi_wkv_forward(wf, uf, k.contiguous(), v.contiguous())
        y = bi_wkv_forward(wf, uf, k.float().contiguous(), v.float().contiguous())
        return y if out_dtype == torch.float32 else y.to(out_dtype)

    @staticmethod
    def backward(ctx, gy):
        # vrwkv.py:47-61: gradients in fp32, returned in w's dtype when that is half / bfloat16
        wf, uf, k, v = ctx.saved_tensors
        out_dtype = ctx.out_dtype
        if ctx.as_held:
            return _wkv_backward(wf.contiguous(), uf.contiguous(), k.contiguous(), v.contiguous(), gy.to(out_dtype).contiguous())
        if k.dtype == out_dtype and v.dtype == out_dtype and out_dtype != torch.float32:
            return tuple(bi_wkv_backward(wf, uf, k.contiguous(), v.contiguous(), gy.to(out_dtype).contiguous(), like_inputs=True))
        gw, gu, gk, gv = bi_wkv_backward(wf, uf, k.float().contiguous(), v.float().contiguous(), gy.float().contiguous())
        if out_dtype == torch.float32:
            return (gw, gu, gk, gv)
        gwu = torch.stack((gw, gu)).to(out_dtype)           # one cast for both parameter gradients
        return (gwu[0], gwu[1], gk.to(out_dtype), gv.to(out_dtype))


class _WKVDivided(torch.autograd.Function):
    """WKV of w / n and u / n (vrwkv.py:183) for parameters, k and v of one type: the divisions, and those of their gradients, inside the
    kernels that read the vectors and write the sums.  Tensor ops divide by a number through its fp32 reciprocal; so do the kernels."""

    @staticmethod
    def forward(ctx, w, u, n, k, v):
        ctx.factor = ctypes.c_float(1.0 / n).value
        ctx.save_for_backward(w, u, k, v)
        return _wkv_forward(w, u, k, v, ctx.factor)

    @staticmethod
    def backward(ctx, gy):
        w, u, k, v = _saved(ctx)
        gw, gu, gk, gv = _wkv_backward(w, u, k, v, gy.to(k.dtype).contiguous(), ctx.factor)
        return gw, gu, None, gk, gv


def divided_takes(w, u, k, v):
    """True where wkv_divided computes RUN_CUDA(w / n, u / n, k, v): plain contiguous GPU tensors of one type outside every transform."""
    return (type(w) in (torch.Tensor, torch.nn.Parameter) and type(u) is type(w) and type(k) is type(v) is torch.Tensor and w.is_cuda
            and w.dtype == u.dtype == k.dtype == v.dtype and w.dtype in _DT and w.dim() == 1
            and all(t.is_contiguous() and t.device == w.device for t in (w, u, k, v)) and not _transformed())


def wkv_divided(w, u, n, k, v):
    y = _lib.host().wkv(w, u, k, v, 1.0 / n)
    return _WKVDivided.apply(w, u, n, k, v) if y is None else y


class _WKVLegacy(torch.autograd.Function):
    """Seven-argument form used by the MAE code (classification/mae/vrwkv/vrwkv.py:30-90)."""

    @staticmethod
    def forward(ctx, B, T, C, w, u, k, v):
        if tuple(k.shape) != (B, T, C):
            raise RuntimeError(f"k has shape {tuple(k.shape)}, expected {(B, T, C)}")
        return WKV.forward(ctx, w, u, k, v)

    @staticmethod
    def backward(ctx, gy):
        return (None, None, None) + tuple(WKV.backward(ctx, gy))


def _plain_call(x):
    """Whether to ask the compiled operators (csrc/host/host_ops.cpp), which look at the arguments themselves and answer None where a
    Python class has to decide."""
    return type(x) is torch.Tensor and x.is_cuda and not torch.compiler.is_compiling()


def RUN_CUDA(*args):
    """RUN_CUDA(w, u, k, v) (vrwkv.py:64-65) or legacy RUN_CUDA(B, T, C, w, u, k, v)."""
    if len(args) == 4:
        w, u, k, v = args
        y = _lib.host().wkv(w, u, k, v, 1.0) if _plain_call(k) else None
        if y is not None:
            return y
        return WKV.apply(w.cuda(), u.cuda(), k.cuda(), v.cuda())
    if len(args) == 7:
        B, T, C, w, u, k, v = args
        return _WKVLegacy.apply(B, T, C, w.cuda(), u.cuda(), k.cuda(), v.cuda())
    raise TypeError("RUN_CUDA takes (w, u, k, v) or (B, T, C, w, u, k, v)")


HEAD_SIZE = 64   # vrwkv6.py:23


def wkv6_forward(B, T, C, H, r, k, v, w, u, w_is_ew=False, out=None, whole=False):
    """Extension-level entry (wkv6_op.cpp:7-9): r,k,v (B,T,C) fp32/bf16/fp16, w (B,T,C) fp32 or
    that dtype, u (H,64); returns y (B,T,C) fp32.  With w_is_ew=False, w is the raw decay logit
    (the kernel applies d = exp(-exp(w))); with True it is ew = -exp(w_raw) as the reference
    extension receives it.  Sequences of more than 256 tokens are cut into segments where there are few of them, by their
    number and length; the last bits of y then depend on how many sequences there are.  whole: none is cut and all go 32 tokens at
    a time, and they do not.  (Either is equally far from float64, 5.0e-6 in bf16 at 300 to 1024 tokens.)"""
    for t, n in ((r, "r"), (k, "k"), (v, "v"), (w, "w"), (u, "u")):
        _check_input(t, n)
    if tuple(r.shape) != (B, T, C) or k.shape != r.shape or v.shape != r.shape or w.shape != r.shape:
        raise RuntimeError("r, k, v, w must all be (B,T,C)")
    if u.numel() != C:
        raise RuntimeError("u must have H*64 = C elements")
    if r.dtype not in _DT or k.dtype != r.dtype or v.dtype != r.dtype:
        raise RuntimeError("r, k, v must share one of float32 / bfloat16 / float16")
    if w.dtype != torch.float32 and w.dtype != r.dtype:
        raise RuntimeError("w must be float32 or have the dtype of r, k, v")
    uf = u if u.dtype == torch.float32 else u.float()
    L = _lib.lib()
    y = (torch.empty((B, T, C), device=r.device, dtype=torch.float32) if out is None
         else _check_out(out, "y", (B, T, C), torch.float32, r))      # the reference passes y in (wkv6_op.cpp:7-9)
    if y.numel() == 0:
        return y
    if whole:
        with _on(r.device):
            _lib.check(L.vrwkv_wkv6_fwd_whole(r.data_ptr(), k.data_ptr(), v.data_ptr(), w.data_ptr(), uf.data_ptr(), y.data_ptr(), B, T, C, H,
                                              _DT[r.dtype], _DT[w.dtype], 1 if w_is_ew else 0, _stream_ptr(r.device)))
        return y
    ws_bytes = L.vrwkv_wkv6_fwd_workspace_bytes(B, T, C, H)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=r.device) if ws_bytes else None
    with _on(r.device):
        _lib.check(L.vrwkv_wkv6_fwd(r.data_ptr(), k.data_ptr(), v.data_ptr(), w.data_ptr(), uf.data_ptr(),
                                    y.data_ptr(), B, T, C, H, _DT[r.dtype], _DT[w.dtype], 1 if w_is_ew else 0,
                                    ws.data_ptr() if ws is not None else None, ws_bytes,
                                    _stream_ptr(r.device)))
    return y


def wkv6_backward(B, T, C, H, r, k, v, w, u, gy, w_is_ew=False, out=None, like_inputs=False):
    """Extension-level entry (wkv6_op.cpp:10-12): returns (gr, gk, gv, gw) as (B,T,C) fp32 and gu as
    (H,64) fp32 (already summed over the batch); gw is the gradient w.r.t. the raw decay logit.
    like_inputs: gr, gk, gv, gw of their inputs' types, rounded from the fp32 sums by the kernel (results passed in as `out`
    are fp32 throughout)."""
    like_inputs = like_inputs and out is None
    for t, n in ((r, "r"), (k, "k"), (v, "v"), (w, "w"), (u, "u"), (gy, "gy")):
        _check_input(t, n)
    if tuple(r.shape) != (B, T, C) or any(x.shape != r.shape for x in (k, v, w, gy)):
        raise RuntimeError("r, k, v, w, gy must all be (B,T,C)")
    if r.dtype not in _DT or k.dtype != r.dtype or v.dtype != r.dtype:
        raise RuntimeError("r, k, v must share one of float32 / bfloat16 / float16")
    if w.dtype != torch.float32 and w.dtype != r.dtype:
        raise RuntimeError("w must be float32 or have the dtype of r, k, v")
    uf = u if u.dtype == torch.float32 else u.float()
    gyf = gy if gy.dtype == torch.float32 else gy.float()
    L = _lib.lib()
    if out is None:
        mk = lambda x: torch.empty((B, T, C), device=r.device, dtype=x.dtype if like_inputs else torch.float32)
        gr, gk, gv, gw = mk(r), mk(k), mk(v), mk(w)
        gu = torch.empty((H, C // H), device=r.device, dtype=torch.float32)
    else:                                                             # caller-allocated (gr, gk, gv, gw, gu)
        gr, gk, gv, gw = (_check_out(t, n, (B, T, C), torch.float32, r) for t, n in zip(out[:4], ("gr", "gk", "gv", "gw")))
        gu = _check_out(out[4], "gu", (H, C // H), torch.float32, r)
    if gr.numel() == 0:
        return gr, gk, gv, gw, gu.zero_()
    if like_inputs:
        fn, ws_bytes = L.vrwkv_wkv6_bwd_like, L.vrwkv_wkv6_bwd_like_workspace_bytes(B, T, C, H, _DT[r.dtype], _DT[w.dtype])
    else:
        fn, ws_bytes = L.vrwkv_wkv6_bwd, L.vrwkv_wkv6_bwd_workspace_bytes(B, T, C, H)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=r.device)
    with _on(r.device):
        _lib.check(fn(r.data_ptr(), k.data_ptr(), v.data_ptr(), w.data_ptr(), uf.data_ptr(),
                                    gyf.data_ptr(), gr.data_ptr(), gk.data_ptr(), gv.data_ptr(), gw.data_ptr(),
                                    gu.data_ptr(), B, T, C, H, _DT[r.dtype], _DT[w.dtype], 1 if w_is_ew else 0,
                                    ws.data_ptr(), ws_bytes, _stream_ptr(r.device)))
    return gr, gk, gv, gw, gu


class WKV_6(torch.autograd.Function):
    """Bidirectional RWKV-6 scan with the reference's call contract (vrwkv6.py:34-70): contiguous
    (B,T,C) inputs, raw decay logit w, fp32 (B,T,C) result.  The `ew = -exp(w)` tensor the
    reference materialises is folded into the kernel."""

    @staticmethod
    def forward(ctx, B, T, C, H, r, k, v, w, u):
        with torch.no_grad():
            assert HEAD_SIZE == C // H
            ctx.B, ctx.T, ctx.C, ctx.H = B, T, C, H
            assert r.is_contiguous()
            assert k.is_contiguous()
            assert v.is_contiguous()
            assert w.is_contiguous()
            assert u.is_contiguous()
            ctx.save_for_backward(r, k, v, w, u)
            return wkv6_forward(B, T, C, H, r, k, v, w, u, whole=WKV_6.stays_whole(T, r.dtype) and any(ctx.needs_input_grad))

    # A 16-bit network rounds y again in every block and amplifies last bits: its gradients move by 3e-2 of their norm (twelve
    # blocks, 400 to 1024 tokens, neither side closer to the fp32 model) when the forward is cut instead of whole, those of an fp32
    # network by 4e-4 at most.  So a 16-bit forward that autograd records stays whole up to 33 chunks -- the 32 x 32 patches of a
    # 512 x 512 image and a class token -- and a sample's y is the same in any batch; that costs up to 66 us a layer (3 / 24 / 96
    # sequences of 1056 tokens: 92 / 94 / 95 us whole, 26 / 35 / 67 cut).  Longer chains cost more (2048 tokens: 175 whole, 34 to 115
    # cut) and are cut.  For the same reason it takes up to 256 tokens 32 at a time, not as one or two products: with those the gradients
    # of VRWKV6-B (64 images, 196 tokens) move by 3.3e-2 at a last-bit difference of 7e-6 in y (62 us a layer in place of 46).  The backward is cut from 257 tokens on in either type: gradients depend on the batch there, by 1.4e-2 in
    # 16 bits.
    @staticmethod
    def stays_whole(T, dtype):
        return T <= 33 * 32 and dtype != torch.float32

    @staticmethod
    def backward(ctx, gy):
        # vrwkv6.py:55-70: gu summed over the batch and shaped (H, C//H); the fp32 gradients leave the kernel rounded to
        # their inputs' types, which is what autograd makes of them next
        with torch.no_grad():
            assert gy.is_contiguous()
            r, k, v, w, u = ctx.saved_tensors
            gr, gk, gv, gw, gu = wkv6_backward(ctx.B, ctx.T, ctx.C, ctx.H, r, k, v, w, u, gy, like_inputs=True)
            return (None, None, None, None, gr, gk, gv, gw, gu)


class _WKV_6Unrecorded(WKV_6):
    """WKV_6 where autograd records nothing.  Inside forward that cannot be seen: grad mode is off there anyway, and
    needs_input_grad is set as soon as the bonus is a parameter."""

    @staticmethod
    def forward(ctx, B, T, C, H, r, k, v, w, u):
        assert HEAD_SIZE == C // H
        assert r.is_contiguous() and k.is_contiguous() and v.is_contiguous() and w.is_contiguous() and u.is_contiguous()
        return wkv6_forward(B, T, C, H, r, k, v, w, u)


def RUN_CUDA_RWKV6(B, T, C, H, r, k, v, w, u):
    """vrwkv6.py:72-73."""
    if _plain_call(r):
        y = _lib.host().wkv6(B, T, C, H, r, k, v, w, u, WKV_6.stays_whole(T, r.dtype))
        if y is not None:
            return y
    return (WKV_6 if torch.is_grad_enabled() else _WKV_6Unrecorded).apply(B, T, C, H, r, k, v, w, u)


def q_shift(input, shift_pixel=1, gamma=1 / 4, patch_resolution=None):
    """q_shift of vrwkv.py:68-79 in plain tensor ops (used where gradients are needed)."""
    assert gamma <= 1 / 4
    B, N, C = input.shape
    x = input.transpose(1, 2).reshape(B, C, patch_resolution[0], patch_resolution[1])
    H, W = patch_resolution
    b1, b2, b3, b4 = _shift_bounds(C, gamma)
    out = torch.zeros_like(x)
    out[:, 0:b1, :, shift_pixel:W] = x[:, 0:b1, :, 0:W - shift_pixel]
    out[:, b1:b2, :, 0:W - shift_pixel] = x[:, b1:b2, :, shift_pixel:W]
    out[:, b2:b3, shift_pixel:H, :] = x[:, b2:b3, 0:H - shift_pixel, :]
    out[:, b3:b4, 0:H - shift_pixel, :] = x[:, b3:b4, shift_pixel:H, :]
    out[:, b4:, ...] = x[:, b4:, ...]
    return out.flatten(2).transpose(1, 2)


def _shift_bounds(C, gamma):
    """Upper ends of the four shifted channel groups exactly as the reference cuts them (vrwkv.py:72-76):
    int(C*gamma), int(C*gamma*2), int(C*gamma*3), int(C*gamma*4)."""
    return int(C * gamma), int(C * gamma * 2), int(C * gamma * 3), int(C * gamma * 4)


def _equal_quarters(C, gamma, head_dim):
    """The kernels shift four groups of one width; true when the reference's cuts are of that kind (every
    stock model: C a multiple of 4 with gamma = 1/4, or per-head quarters)."""
    if head_dim:
        return True
    b = _shift_bounds(C, gamma)
    return b == (b[0], 2 * b[0], 3 * b[0], 4 * b[0])


def stack_mixes(mixes, device):
    """The (n_mix, C) fp32 table q_shift_mix hands to the kernel; callers that apply the same mixes again and again
    may build it once and pass it as `mix_table`."""
    return torch.stack([m.detach().reshape(-1).float() for m in mixes]).contiguous().to(device)


def q_shift_mix(x, mixes, shift_pixel=1, gamma=1 / 4, patch_resolution=None, head_dim=0, mix_table=None):
    """One HIP kernel for q_shift + the token-mix lerps: returns [x*m + q_shift(x)*(1-m) for m in mixes]
    (vrwkv.py:160-163 / :248-250).  mixes: 1..3 tensors of C elements.  head_dim=64 gives the per-head
    q_shift_multihead of vrwkv6.py:75-100 (a trailing class token is passed through).  Forward only."""
    _check_input(x, "x")
    if x.dim() != 3 or x.dtype not in _DT:
        raise RuntimeError("x must be (B,T,C) float32 / bfloat16 / float16")
    B, T, C = x.shape
    Hp, Wp = patch_resolution
    if not _equal_quarters(C, gamma, head_dim):
        # unequal channel groups (C*gamma not an integer): the reference's slice copies, then the lerps
        xx = q_shift(x, shift_pixel, gamma, patch_resolution)
        tab = mix_table if mix_table is not None else stack_mixes(mixes, x.device)
        return [(x.float() * m + xx.float() * (1 - m)).to(x.dtype) for m in tab]
    mix = mix_table if mix_table is not None else stack_mixes(mixes, x.device)
    if mix.shape != (len(mixes), C) or mix.dtype != torch.float32 or not mix.is_contiguous() or mix.device != x.device:
        raise RuntimeError("mix_table must be a contiguous float32 (n_mix, C) tensor on x's device")
    if mix.shape[1] != C:
        raise RuntimeError("every mix vector must have C elements")
    outs = [torch.empty_like(x) for _ in mixes]
    if x.numel() == 0:
        return outs
    ptrs = (ctypes.c_void_p * len(outs))(*[o.data_ptr() for o in outs])
    g = head_dim // 4 if head_dim else int(C * gamma)
    with _on(x.device):
        _lib.check(_lib.lib().vrwkv_qshift_mix(x.data_ptr(), mix.data_ptr(), ptrs, len(outs), B, T, C, Hp, Wp,
                                               shift_pixel, g, head_dim, _DT[x.dtype], _stream_ptr(x.device)))
    return outs


PRE_NONE, PRE_RELU_SQ = 0, 1
POST_NONE, POST_SIGMOID_GATE, POST_RESIDUAL = 0, 1, 2
ROW_FUSE_ENABLED = True      # set False to make row_fuse run the tensor-op sequence everywhere (for comparisons)


def _vec_ok(*tensors):
    """True when every given tensor can be read as it lies in 16-byte pieces (dense and 16-byte aligned)."""
    return all(t is None or (t.is_contiguous() and t.data_ptr() % 16 == 0) for t in tensors)


def _dense(t):
    """t as the kernels read it, dense and on 16 bytes."""
    return t if t is None or (t.is_contiguous() and not t.data_ptr() & 15) else t.clone(memory_format=torch.contiguous_format)


def _saved(ctx):
    """The saved tensors as the kernels read them: a hook on saved tensors may hand back other strides or a piece of a larger tensor."""
    return tuple(_dense(t) for t in ctx.saved_tensors)


def row_fuse_tensor_ops(a, other=None, ln_weight=None, ln_bias=None, gamma=None, pre=PRE_NONE, post=POST_NONE, eps=1e-5):
    """The PyTorch-op sequence row_fuse replaces (what the reference runs: vrwkv.py:184-186, :256-261, :300-313);
    used under autograd and wherever the kernel does not apply."""
    y = torch.square(torch.relu(a)) if pre == PRE_RELU_SQ else a
    if ln_weight is not None:
        y = torch.nn.functional.layer_norm(y, (y.shape[-1],), ln_weight, ln_bias, eps)
    if post == POST_SIGMOID_GATE:
        y = torch.sigmoid(other) * y
    elif post == POST_RESIDUAL:
        y = other + (gamma * y if gamma is not None else y)
    return y


class _RowFuse(torch.autograd.Function):
    """row_fuse with a hand-written backward (vrwkv_rowfuse / vrwkv_rowfuse_bwd).  Per-channel inputs arrive in the
    dtype of `a` (the casts outside are differentiated by autograd)."""

    @staticmethod
    def forward(ctx, a, other, ln_weight, ln_bias, gamma, pre, post, eps):
        ctx.save_for_backward(a, other, ln_weight, ln_bias, gamma)
        ctx.meta = (pre, post, eps)
        return _row_fuse_launch(a, other, ln_weight, ln_bias, gamma, pre, post, eps)

    @staticmethod
    def backward(ctx, gout):
        a, other, ln_weight, ln_bias, gamma = _saved(ctx)
        pre, post, eps = ctx.meta
        N = a.shape[-1]
        rows = a.numel() // N
        gout = gout.to(a.dtype).contiguous()
        ga = torch.empty_like(a)
        go = torch.empty_like(a) if post == POST_SIGMOID_GATE else None
        sums = ln_weight is not None or (post == POST_RESIDUAL and gamma is not None)
        L = _lib.lib()
        gparam = ws = None
        ws_bytes = 0
        if sums:
            gparam = torch.empty(3, N, dtype=a.dtype, device=a.device)    # rounded once from the fp32 sums
            ws_bytes = L.vrwkv_rowfuse_bwd_workspace_bytes(rows, N)
            ws = torch.empty(ws_bytes, dtype=torch.uint8, device=a.device)
        ptr = lambda t: t.data_ptr() if t is not None else None
        with _on(a.device):
            _lib.check(L.vrwkv_rowfuse_bwd_like(a.data_ptr(), ptr(other), ptr(ln_weight), ptr(ln_bias), ptr(gamma),
                                           gout.data_ptr(), ga.data_ptr(), ptr(go), ptr(gparam), rows, N, pre, post,
                                           float(eps), _DT[a.dtype], ptr(ws), ws_bytes, _stream_ptr(a.device)))
        g_other = go if post == POST_SIGMOID_GATE else (gout if post == POST_RESIDUAL else None)
        gp = gparam
        g_w = gp[0] if ln_weight is not None else None
        g_b = gp[1] if ln_bias is not None else None
        g_g = gp[2] if (gamma is not None and post == POST_RESIDUAL) else None
        return ga, g_other, g_w, g_b, g_g, None, None, None


def _row_fuse_launch(a, other, ln_weight, ln_bias, gamma, pre, post, eps):
    out = torch.empty_like(a)
    N = a.shape[-1]
    ptr = lambda t: t.data_ptr() if t is not None else None
    with _on(a.device):
        _lib.check(_lib.lib().vrwkv_rowfuse(a.data_ptr(), ptr(other), ptr(ln_weight), ptr(ln_bias), ptr(gamma), out.data_ptr(),
                                            a.numel() // N, N, pre, post, float(eps), _DT[a.dtype], _stream_ptr(a.device)))
    return out


def row_fuse(a, other=None, ln_weight=None, ln_bias=None, gamma=None, pre=PRE_NONE, post=POST_NONE, eps=1e-5):
    """One HIP kernel per row-wise epilogue of a block: out = post(LayerNorm(pre(a))) with pre = identity / relu^2,
    LayerNorm optional, post = identity / sigmoid(other) * y / other + gamma * y; under autograd one backward kernel
    (rows of at most 1024 channels when LayerNorm or gamma take part).  Where the kernels do not apply (not on the
    GPU, row length, alignment) the tensor ops are used instead."""
    tensors = [t for t in (a, other, ln_weight, ln_bias, gamma) if t is not None]
    N = a.shape[-1]
    vec = 4 if a.dtype == torch.float32 else 8
    need_grad = torch.is_grad_enabled() and any(t.requires_grad for t in tensors)
    sums = ln_weight is not None or (post == POST_RESIDUAL and gamma is not None)
    fits = (ROW_FUSE_ENABLED and not _forward_mode() and a.is_cuda and a.dtype in _DT and N % vec == 0 and N // vec <= 1024 and a.numel() > 0
            and (other is None or (other.shape == a.shape and other.dtype == a.dtype))
            and not (need_grad and sums and N > 1024))
    if not fits:
        return row_fuse_tensor_ops(a, other, ln_weight, ln_bias, gamma, pre, post, eps)
    if need_grad:
        ac = a.contiguous()
        oc = other.contiguous() if other is not None else None
        par = [p.reshape(-1).to(a.dtype).contiguous() if p is not None else None for p in (ln_weight, ln_bias, gamma)]
        if post != POST_RESIDUAL:
            par[2] = None
        if not _vec_ok(ac, oc, *par) or any(p is not None and p.numel() != N for p in par):
            return row_fuse_tensor_ops(a, other, ln_weight, ln_bias, gamma, pre, post, eps)
        return _RowFuse.apply(ac, oc, par[0], par[1], par[2], pre, post, float(eps))
    a = a.contiguous()
    other = other.contiguous() if other is not None else None
    par = [p.detach().reshape(-1).to(a.dtype).contiguous() if p is not None else None for p in (ln_weight, ln_bias, gamma)]
    if not _vec_ok(a, other, *par):
        return row_fuse_tensor_ops(a, other, ln_weight, ln_bias, gamma, pre, post, eps)
    for p in par:
        if p is not None and p.numel() != N:
            raise RuntimeError("LayerNorm weight, bias and gamma must have one element per channel")
    return _row_fuse_launch(a, other, par[0], par[1], par[2], pre, post, eps)


def maa_mix_tensor_ops(x, sx, m, maas):
    """vrwkv6.py:180, 190-194 as the reference writes them: xx = sx - x; x + xx * (maa_i + m_i)."""
    xx = sx - x
    return [x + xx * (maa + mi) for maa, mi in zip(maas, m.unbind(0))]


class _MaaMix(torch.autograd.Function):
    """maa_mix with a hand-written backward (vrwkv_maa_mix / vrwkv_maa_mix_bwd); the five vectors enter as one (5, C)
    fp32 table built by differentiable tensor ops outside."""

    @staticmethod
    def forward(ctx, x, sx, m, table):
        ctx.save_for_backward(x, sx, m, table)
        return tuple(_maa_mix_launch(x, sx, m, table))

    @staticmethod
    def backward(ctx, *gouts):
        x, sx, m, table = _saved(ctx)
        C = x.shape[-1]
        rows = x.numel() // C
        gs = [g.to(x.dtype).contiguous() for g in gouts]
        gx, gsx, gm = torch.empty_like(x), torch.empty_like(x), torch.empty_like(m)
        gmaa = torch.empty_like(table)
        L = _lib.lib()
        ws_bytes = L.vrwkv_maa_mix_bwd_workspace_bytes(rows, C)
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=x.device)
        ptrs = (ctypes.c_void_p * 5)(*[g.data_ptr() for g in gs])
        with _on(x.device):
            _lib.check(L.vrwkv_maa_mix_bwd(x.data_ptr(), sx.data_ptr(), m.data_ptr(), table.data_ptr(), ptrs, gx.data_ptr(),
                                           gsx.data_ptr(), gm.data_ptr(), gmaa.data_ptr(), rows, C, _DT[x.dtype],
                                           ws.data_ptr(), ws_bytes, _stream_ptr(x.device)))
        return gx, gsx, gm, gmaa


def _maa_mix_launch(x, sx, m, table):
    C = x.shape[-1]
    outs = [torch.empty_like(x) for _ in range(5)]
    ptrs = (ctypes.c_void_p * 5)(*[o.data_ptr() for o in outs])
    with _on(x.device):
        _lib.check(_lib.lib().vrwkv_maa_mix(x.data_ptr(), sx.data_ptr(), m.data_ptr(), table.data_ptr(), ptrs,
                                            x.numel() // C, C, _DT[x.dtype], _stream_ptr(x.device)))
    return outs


def maa_mix(x, sx, m, maas, maa_table=None):
    """The five data-dependent token mixes of VRWKV6 (vrwkv6.py:190-194) in one HIP kernel: x, sx (the shifted x):
    (B,T,C); m: (5,B,T,C); maas: the five (C,) vectors time_maa_w, _k, _v, _r, _g (or their stacked fp32 table).
    Under autograd one backward kernel; tensor ops when the kernels do not apply."""
    C = x.shape[-1]
    vec = 4 if x.dtype == torch.float32 else 8
    tensors = [x, sx, m] + list(maas)
    need_grad = torch.is_grad_enabled() and any(t.requires_grad for t in tensors)
    fits = (ROW_FUSE_ENABLED and not _forward_mode() and x.is_cuda and x.dtype in _DT and C % vec == 0 and x.numel() > 0
            and sx.shape == x.shape and sx.dtype == x.dtype and m.dtype == x.dtype and tuple(m.shape) == (5,) + tuple(x.shape)
            and not (need_grad and x.numel() // C > 65535 * 32))
    if not fits:
        return maa_mix_tensor_ops(x, sx, m, maas)
    xc, sxc, mc = x.contiguous(), sx.contiguous(), m.contiguous()
    if not _vec_ok(xc, sxc, mc):
        return maa_mix_tensor_ops(x, sx, m, maas)
    if need_grad:
        table = torch.stack([a.reshape(-1) for a in maas]).float()      # differentiable; one cast for the five vectors
        return list(_MaaMix.apply(xc, sxc, mc, table))
    table = maa_table if maa_table is not None else stack_mixes(maas, x.device)
    if tuple(table.shape) != (5, C) or table.dtype != torch.float32 or not table.is_contiguous():
        raise RuntimeError("maa table must be a contiguous float32 (5, C) tensor")
    return _maa_mix_launch(xc, sxc, mc, table)


class _MaaLoraMix(torch.autograd.Function):
    """The five mixes with their low-rank products inside (vrwkv_maa_lora_mix and its backward, which forms the products again); lo (M, 160),
    w2 (5, 32, C), table as for _MaaMix."""

    @staticmethod
    def forward(ctx, x, sx, lo, w2, table, token_product):
        ctx.save_for_backward(x, sx, lo, w2, table)
        ctx.token_product = token_product
        return tuple(_maa_lora_launch(x, sx, lo, w2, table))

    @staticmethod
    def backward(ctx, *gouts):
        x, sx, lo, w2, table = ctx.saved_tensors
        C = x.shape[-1]
        rows = x.numel() // C
        stack = lo.reshape(rows, 5, -1).transpose(0, 1)
        gs = [g.to(x.dtype) for g in gouts]
        if torch.is_grad_enabled() or batched_cotangent(*gs) or _transformed():
            f = [t + m.view(x.shape) for t, m in zip(table.to(x.dtype), torch.bmm(stack, w2))]
            gx, gsx = sum(g * (1 - t) for g, t in zip(gs, f)), sum(g * t for g, t in zip(gs, f))
            gm = torch.stack([(g * (sx - x)).reshape(rows, C) for g in gs])
            gtable = gm.float().sum(1)
        else:
            x, sx, lo, w2, table, *gs = (_dense(t) for t in (x, sx, lo, w2, table, *gs))
            gx, gsx, gtable = torch.empty_like(x), torch.empty_like(x), torch.empty_like(table)
            gm = torch.empty((5, rows, C), dtype=x.dtype, device=x.device)
            L = _lib.lib()
            ws_bytes = L.vrwkv_maa_lora_mix_bwd_workspace_bytes(rows, C)
            ws = torch.empty(ws_bytes, dtype=torch.uint8, device=x.device)
            with _on(x.device):
                _lib.check(L.vrwkv_maa_lora_mix_bwd(x.data_ptr(), sx.data_ptr(), lo.data_ptr(), w2.data_ptr(), table.data_ptr(),
                                                    (ctypes.c_void_p * 5)(*[g.data_ptr() for g in gs]), gx.data_ptr(), gsx.data_ptr(), gm.data_ptr(),
                                                    gtable.data_ptr(), rows, C, _DT[x.dtype], ws.data_ptr(), ws_bytes, _stream_ptr(x.device)))
        need = ctx.needs_input_grad
        glo = torch.bmm(gm, w2.transpose(1, 2).contiguous()).transpose(0, 1).reshape(lo.shape) if need[2] else None
        gw2 = ctx.token_product(stack, gm) if need[3] else None
        return gx, gsx, glo, gw2, gtable, None


def _maa_lora_launch(x, sx, lo, w2, table):
    C = x.shape[-1]
    outs = [torch.empty_like(x) for _ in range(5)]
    with _on(x.device):
        _lib.check(_lib.lib().vrwkv_maa_lora_mix(x.data_ptr(), sx.data_ptr(), lo.data_ptr(), w2.data_ptr(), table.data_ptr(),
                                                 (ctypes.c_void_p * 5)(*[o.data_ptr() for o in outs]), x.numel() // C, C, _DT[x.dtype],
                                                 _stream_ptr(x.device)))
    return outs


def maa_lora_mix(x, sx, lo, w2, maas, token_product, maa_table=None):
    """maa_mix(x, sx, m, maas) with m_i = lo_i w2_i formed inside (vrwkv6.py:183-194): lo (B*T, 160), w2 (5, 32, C), 16-bit tensors.  None where
    the kernels do not apply.  token_product(a, b): a^T b over the tokens, for the gradient of w2."""
    C = x.shape[-1]
    tensors = (x, sx, lo, w2, *maas)
    if not (ROW_FUSE_ENABLED and x.is_cuda and x.dtype in (torch.bfloat16, torch.float16) and x.dim() == 3 and x.numel() > 0 and C % 64 == 0 and C <= 65536
            and all(type(t) in (torch.Tensor, torch.nn.Parameter) and t.dtype == x.dtype and t.device == x.device for t in tensors)
            and sx.shape == x.shape and tuple(w2.shape) == (5, 32, C) and tuple(lo.shape) == (x.numel() // C, 160) and all(m.numel() == C for m in maas)
            and all(t.is_contiguous() for t in (x, sx, lo, w2)) and _vec_ok(x, sx, lo, w2) and x.numel() // C <= 65535 * 64
            and not torch.is_autocast_enabled("cuda") and not _transformed()):
        return None
    if torch.is_grad_enabled() and any(t.requires_grad for t in tensors):
        return list(_MaaLoraMix.apply(x, sx, lo, w2, torch.stack([a.reshape(-1) for a in maas]).float(), token_product))
    return _maa_lora_launch(x, sx, lo, w2, maa_table if maa_table is not None else stack_mixes(maas, x.device))


def groupnorm_gate_tensor_ops(y, gate, gn_weight, gn_bias, n_groups, eps=1e-5):
    """vrwkv6.py:205-211 and :199: ln_x on the (B*T, C) view, times silu(gate).  The group statistics are written out
    with mean / var instead of torch.nn.functional.group_norm: on a GPU that function's backward returns wrong weight
    and bias gradients for a 2-D input of more than 128 rows (PyTorch 2.10.0+rocm7.0, every dtype: measured against
    the sums written out in float64 and against the CPU), and this function is the path that autograd differentiates
    when the kernels do not apply.  Statistics in fp32 for 16-bit inputs, as the library computes them."""
    C = y.shape[-1]
    x = y.to(gate.dtype).reshape(-1, n_groups, C // n_groups)
    xs = x.float() if x.dtype in (torch.bfloat16, torch.float16) else x
    mean = xs.mean(-1, keepdim=True)
    var = xs.var(-1, unbiased=False, keepdim=True)
    xh = ((xs - mean) * torch.rsqrt(var + eps)).reshape(-1, C)
    yn = (xh * gn_weight + gn_bias).to(gate.dtype)
    return yn.view(gate.shape) * torch.nn.functional.silu(gate)


class _GroupNormGate(torch.autograd.Function):
    """groupnorm_gate with a hand-written backward (vrwkv_groupnorm_gate / vrwkv_groupnorm_gate_bwd)."""

    @staticmethod
    def forward(ctx, y, gate, w, b, group, eps):
        ctx.save_for_backward(y, gate, w, b)
        ctx.meta = (group, eps)
        return _groupnorm_gate_launch(y, gate, w, b, group, eps)

    @staticmethod
    def backward(ctx, gout):
        y, gate, w, b = _saved(ctx)
        group, eps = ctx.meta
        C = y.shape[-1]
        rows = y.numel() // C
        gout = gout.to(gate.dtype).contiguous()
        gy, gg = torch.empty_like(y), torch.empty_like(gate)
        gparam = torch.empty(2, C, dtype=gate.dtype, device=y.device)
        L = _lib.lib()
        ws_bytes = L.vrwkv_groupnorm_gate_bwd_workspace_bytes(rows, C)
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=y.device)
        with _on(y.device):
            _lib.check(L.vrwkv_groupnorm_gate_bwd_like(y.data_ptr(), gate.data_ptr(), w.data_ptr(), b.data_ptr(), gout.data_ptr(),
                                                  gy.data_ptr(), gg.data_ptr(), gparam.data_ptr(), rows, C, group, float(eps),
                                                  _DT[y.dtype], _DT[gate.dtype], ws.data_ptr(), ws_bytes, _stream_ptr(y.device)))
        return gy, gg, gparam[0], gparam[1], None, None


def _groupnorm_gate_launch(y, gate, w, b, group, eps):
    C = y.shape[-1]
    out = torch.empty_like(gate)
    with _on(y.device):
        _lib.check(_lib.lib().vrwkv_groupnorm_gate(y.data_ptr(), gate.data_ptr(), w.data_ptr(), b.data_ptr(), out.data_ptr(),
                                                   y.numel() // C, C, group, float(eps), _DT[y.dtype], _DT[gate.dtype],
                                                   _stream_ptr(y.device)))
    return out


def groupnorm_gate(y, gate, gn_weight, gn_bias, n_groups, eps=1e-5):
    """GroupNorm(n_groups, C) of every token of y (fp32 as RUN_CUDA_RWKV6 returns it, or gate's dtype) times
    silu(gate), in one HIP kernel (vrwkv6.py:199, 205-211), and one backward kernel under autograd (C <= 1024);
    tensor ops for other shapes."""
    C = y.shape[-1]
    group = C // n_groups if n_groups > 0 and C % n_groups == 0 else 0
    tensors = [y, gate, gn_weight, gn_bias]
    need_grad = torch.is_grad_enabled() and any(t.requires_grad for t in tensors)
    fits = (ROW_FUSE_ENABLED and not _forward_mode() and y.is_cuda and gate.dtype in (torch.float32, torch.bfloat16, torch.float16) and y.shape == gate.shape
            and y.dtype in (torch.float32, gate.dtype) and group in (8, 16, 32, 64, 128) and y.numel() > 0
            and not (need_grad and C > 1024))
    if not fits:
        return groupnorm_gate_tensor_ops(y, gate, gn_weight, gn_bias, n_groups, eps)
    yc, gc = y.contiguous(), gate.contiguous()
    if need_grad:
        w, b = gn_weight.to(gate.dtype).contiguous(), gn_bias.to(gate.dtype).contiguous()
    else:
        w, b = gn_weight.detach().to(gate.dtype).contiguous(), gn_bias.detach().to(gate.dtype).contiguous()
    if not _vec_ok(yc, gc, w, b):
        return groupnorm_gate_tensor_ops(y, gate, gn_weight, gn_bias, n_groups, eps)
    if need_grad:
        return _GroupNormGate.apply(yc, gc, w, b, group, float(eps))
    return _groupnorm_gate_launch(yc, gc, w, b, group, eps)


class _QShiftMix(torch.autograd.Function):
    """q_shift + mix lerps with a hand-written backward (vrwkv_qshift_mix / vrwkv_qshift_mix_bwd_add); the mix vectors
    enter as one (n_mix, C) table of their own type, so whatever produced them (parameters, 1 - parameter, ...) is differentiated
    by autograd outside.  through: as many more results, each x itself: what uses x next to the mixes takes one of these, and the
    backward kernel adds its gradient where autograd would run a pass over the tokens."""

    @staticmethod
    def forward(ctx, x, table, shift_pixel, gamma, Hp, Wp, head_dim, through=0):
        x = x.contiguous()
        ctx.table_dtype = table.dtype
        table = table.float().contiguous()
        ctx.save_for_backward(x, table)
        ctx.meta = (shift_pixel, gamma, Hp, Wp, head_dim)
        ctx.set_materialize_grads(False)
        outs = q_shift_mix(x, [None] * table.shape[0], shift_pixel, gamma, (Hp, Wp), head_dim, mix_table=table)
        return (*outs, *(x.view_as(x) for _ in range(through)))

    @staticmethod
    def backward(ctx, *gouts):
        x, table = _saved(ctx)
        shift_pixel, gamma, Hp, Wp, head_dim = ctx.meta
        B, T, C = x.shape
        n_mix = table.shape[0]
        gs = [g.to(x.dtype).contiguous() if g is not None else torch.zeros_like(x) for g in gouts[:n_mix]]
        add, apart = [g for g in gouts[n_mix:] if g is not None], []
        if torch.is_grad_enabled():                              # to be differentiated again: what has a graph is added by tensor ops
            add, apart = [g for g in add if not g.requires_grad], [g for g in add if g.requires_grad]
        add = [g.to(x.dtype).contiguous() for g in add]
        gx = torch.empty_like(x)
        like = ctx.table_dtype == x.dtype                        # the table's gradient rounded by the kernel, or cast below
        gmix = torch.empty_like(table, dtype=x.dtype if like else torch.float32)
        L = _lib.lib()
        ws_bytes = L.vrwkv_qshift_mix_bwd_workspace_bytes(n_mix, B, T, C)
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=x.device)
        ptrs = (ctypes.c_void_p * n_mix)(*[g.data_ptr() for g in gs])
        adds = (ctypes.c_void_p * 2)(*[g.data_ptr() for g in add])
        g = head_dim // 4 if head_dim else int(C * gamma)
        with _on(x.device):
            _lib.check(L.vrwkv_qshift_mix_bwd_add(x.data_ptr(), table.data_ptr(), ptrs, n_mix, adds, len(add), gx.data_ptr(), gmix.data_ptr(),
                                                  _DT[gmix.dtype], B, T, C, Hp, Wp, shift_pixel, g, head_dim, _DT[x.dtype],
                                                  ws.data_ptr(), ws_bytes, _stream_ptr(x.device)))
        for a in apart:
            gx = gx + a
        return gx, gmix.to(ctx.table_dtype), None, None, None, None, None, None


def q_shift_mix_autograd(x, mixes, shift_pixel=1, gamma=1 / 4, patch_resolution=None, head_dim=0, through=0):
    """q_shift_mix for training: the same fused forward kernel, and one fused backward kernel in place of autograd
    through the slice copies and lerps.  `mixes` may be parameters or tensors derived from parameters.  through (0 to 2): so many
    more results, x for its other uses, whose gradients the backward kernel adds."""
    _check_input(x, "x")
    if x.dim() != 3 or x.dtype not in _DT:
        raise RuntimeError("x must be (B,T,C) float32 / bfloat16 / float16")
    table = torch.stack([m.reshape(-1) for m in mixes])
    Hp, Wp = patch_resolution
    if not _equal_quarters(x.shape[-1], gamma, head_dim):
        table = table.float()
        xx = q_shift(x, shift_pixel, gamma, patch_resolution)
        return [(x.float() * m + xx.float() * (1 - m)).to(x.dtype) for m in table] + [x] * through
    return list(_QShiftMix.apply(x, table, shift_pixel, gamma, Hp, Wp, head_dim, through))


class _TableResize(torch.autograd.Function):
    """Bicubic resampling of a (1, Hs*Ws, C) table, or its adjoint (vrwkv_pos_resize): linear maps, each the other's
    derivative, so gradients of any order and forward-mode tangents go through the same two kernels."""

    @staticmethod
    def forward(ctx, table, src, dst, adjoint):
        ctx.meta = (src, dst, adjoint)
        return _table_resize_launch(table, src, dst, adjoint)

    @staticmethod
    def backward(ctx, g):
        src, dst, adjoint = ctx.meta
        return _TableResize.of(g)(g, src, dst, not adjoint), None, None, None

    @staticmethod
    def jvp(ctx, t, *_):
        return _TableResize.of(t)(t, *ctx.meta)

    @staticmethod
    def of(t):
        """The map for a cotangent or tangent: tensor ops for a batch of them of either kind and wherever else t may not have
        memory of its own or a function of this class may not be applied."""
        return _table_resize_ops if batched_cotangent(t) or _transformed() else _TableResize.apply


def _table_resize_ops(table, src, dst, adjoint):
    """The same two maps as tensor ops, for tensors without memory of their own."""
    n, C = (dst if adjoint else src), table.shape[-1]
    t = table.float().reshape(1, n[0], n[1], C).permute(0, 3, 1, 2)
    if adjoint:
        t = torch.ops.aten.upsample_bicubic2d_backward(t, dst, (1, C) + src, False)
    else:
        t = torch.nn.functional.interpolate(t, size=dst, mode="bicubic", align_corners=False)
    return t.reshape(1, C, -1).transpose(1, 2).to(table.dtype)


def _table_resize_launch(table, src, dst, adjoint):
    table = table.contiguous()
    n, C = (src if adjoint else dst), table.shape[-1]
    out = torch.empty((1, n[0] * n[1], C), dtype=table.dtype, device=table.device)
    with _on(table.device):
        _lib.check(_lib.lib().vrwkv_pos_resize(table.data_ptr(), out.data_ptr(), src[0], src[1], dst[0], dst[1], C,
                                               1 if adjoint else 0, _DT[table.dtype], _stream_ptr(table.device)))
    return out


def batched_cotangent(*tensors):
    """True where a backward runs on a batch of cotangents (is_grads_batched): plain to Python, but without memory."""
    return any(torch._C._functorch.is_legacy_batchedtensor(t) for t in tensors)


def _forward_mode():
    """True inside a level of forward-mode differentiation: a kernel's result has no tangent, whatever its arguments carry."""
    return torch.autograd.forward_ad._current_level >= 0


def _transformed():
    """True inside torch.compile, jit tracing, a functorch transform, a level of forward-mode differentiation or a dispatch /
    function mode, which are to see the tensor ops."""
    return (torch.compiler.is_compiling() or torch.jit.is_tracing() or torch._C._functorch.peek_interpreter_stack() is not None
            or torch._C._len_torch_dispatch_stack() > 0 or torch._C._len_torch_function_stack() > 0 or _forward_mode())


def resize_table(table, src_shape, dst_shape):
    """A (1, Hs*Ws, C) position table resampled bicubically to the grid dst_shape in one HIP kernel (and one for its
    gradient): fp32 arithmetic, result of the table's type.  None where the kernel does not apply (off the GPU, other types
    of tensor, traced or transformed calls, empty grids)."""
    src, dst = tuple(int(n) for n in src_shape), tuple(int(n) for n in dst_shape)
    if (not table.is_cuda or table.dtype not in _DT or table.dim() != 3 or table.shape[0] != 1
            or type(table) not in (torch.Tensor, torch.nn.Parameter) or len(src) != 2 or len(dst) != 2
            or min(src + dst) <= 0 or table.shape[1] != src[0] * src[1] or table.shape[2] == 0
            or _transformed()):
        return None
    return _TableResize.apply(table, src, dst, False)


BLOCK_FUSE_ENABLED = True    # set False to make the blocks run operator by operator everywhere (for comparisons)


def block_takes(x):
    """True where vrwkv_block_fwd may stand in for a block's operators: no autograd, a plain contiguous GPU tensor
    outside every kind of transform."""
    return (not torch.is_grad_enabled() and BLOCK_FUSE_ENABLED and ROW_FUSE_ENABLED and type(x) is torch.Tensor and x.is_cuda
            and x.dtype in _DT and x.dim() == 3 and x.numel() > 0 and x.is_contiguous()
            and not torch.is_autocast_enabled("cuda") and not _transformed())


def block_weights_fit(x, weights):
    """True when every weight is a plain contiguous parameter of x's type and device."""
    return _lib.host().weights_fit(x, weights)


def block_forward(x, tensors, params=None, **scalars):
    """vrwkv_block_fwd on the current stream: tensors and scalars fill the like-named fields of vrwkv_block_args; with params
    (fields of vrwkv_block6_params) vrwkv_block6_fwd.  None when a tensor is not aligned for 16-byte accesses."""
    out = _lib.host().block_forward(x, tensors, params, scalars)
    if type(out) is int:
        _lib.check(out)
    return out


def _token_rows(t):
    """t (n, M, C) with every row in 16-byte pieces, copied where it is not laid out so."""
    sn, sm, sc = t.stride()
    if sc == 1 and sm >= t.shape[2] and not (sn | sm) & 7 and not t.data_ptr() & 15:
        return t
    return t.clone(memory_format=torch.contiguous_format)


def weight_grad(g, x):
    """sum over t of g[.., t, o] x[.., t, i] for token matrices g (M, O), x (M, I) or stacks (n, M, O), (n, M, I) of one 16-bit
    type, O and I multiples of 8: the gradient of a projection's weight (O, I), fp32 sums rounded once.  Rows may lie at any
    pitch of 16-byte pieces; other layouts are copied."""
    stack = g.dim() == 3
    g3, x3 = (_token_rows(g), _token_rows(x)) if stack else (_token_rows(g[None]), _token_rows(x[None]))
    n, M, O = g3.shape
    I = x3.shape[2]
    out = torch.empty((n, O, I) if stack else (O, I), dtype=g.dtype, device=g.device)
    if out.numel() == 0 or M == 0:
        return out.zero_()
    L = _lib.lib()
    ws_bytes = L.vrwkv_wgrad_workspace_bytes(n, M, O, I)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=g.device)
    gs, xs = g3.stride(), x3.stride()
    with _on(g.device):
        _lib.check(L.vrwkv_wgrad(g3.data_ptr(), x3.data_ptr(), out.data_ptr(), n, M, O, I, gs[1], xs[1], gs[0], xs[0],
                                 _DT[g.dtype], ws.data_ptr(), ws_bytes, _stream_ptr(g.device)))
    return out


def weight_grad_group(gs, xs):
    """[g^T x for g, x in zip(gs, xs)] over the rows of 1 to 5 pairs of token matrices g (M, O), x (M, I) of one 16-bit type, O and I
    multiples of 8: the gradients of several weights (O, I) in one launch (vrwkv_wgrad_group), fp32 sums rounded once."""
    gs, xs = [_token_rows(g[None])[0] for g in gs], [_token_rows(x[None])[0] for x in xs]
    n, M, dev = len(gs), gs[0].shape[0], gs[0].device
    outs = [torch.empty(g.shape[1], x.shape[1], dtype=g.dtype, device=dev) for g, x in zip(gs, xs)]
    P, I = ctypes.c_void_p * n, ctypes.c_int * n
    o, i = I(*[g.shape[1] for g in gs]), I(*[x.shape[1] for x in xs])
    L = _lib.lib()
    ws_bytes = L.vrwkv_wgrad_group_workspace_bytes(o, i, n, M)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
    with _on(dev):
        _lib.check(L.vrwkv_wgrad_group(P(*[t.data_ptr() for t in gs]), P(*[t.data_ptr() for t in xs]), P(*[t.data_ptr() for t in outs]), o, i,
                                       I(*[t.stride(0) for t in gs]), I(*[t.stride(0) for t in xs]), n, M, _DT[gs[0].dtype],
                                       ws.data_ptr(), ws_bytes, _stream_ptr(dev)))
    return outs


EPI_RELU_SQ, EPI_RELU_SQ_BWD, EPI_ROUND = 1, 8, 16


def linear_takes(x, weights, widths=None):
    """True where linear_group may stand in for x @ W^T on the GPU: 16-bit token matrices and weights of one type outside autocast and
    every kind of transform, sizes that the kernel of the large tiles takes, and the transpose that the backward makes of the weights
    (include/vrwkv_hip.h, csrc/linear_wide.hip), and that fill the chip with them: 70 tiles of 128 x 128.  widths: what each weight's input has for columns, x's by default; a weight that does not fit
    its input is left to the operators, which refuse it."""
    M, K = x.numel() // max(x.shape[-1], 1), x.shape[-1]
    if torch.compiler.is_compiling() or not (x.is_cuda and x.dtype in (torch.bfloat16, torch.float16) and M > 0):
        return False
    for w, width in zip(weights, widths if widths is not None else [K] * len(weights)):
        if w.dim() != 2 or w.shape[1] != width:
            return False
        N, k = w.shape
        if M * N < 70 * 128 * 128 or max(N, k) > 65536 or (M + 256) * max(N, k) >= 1 << 29 or (N + 256) * (k + 256) >= 1 << 29:
            return False
        if not (w.dtype == x.dtype and w.device == x.device and (N % 192 == k % 192 == 0 or N % 128 == k % 128 == 0)):
            return False
    return (not torch.is_autocast_enabled("cuda") and not _transformed()
            and all(w.is_contiguous() and w.data_ptr() % 16 == 0 for w in weights))        # (memory last: not every traced tensor has any)


def linear_group(problems):
    """vrwkv_linear_group: one launch of out = epilogue(a w^T) for 1 to 5 dicts of a (M, K), w (N, K) and, optional, gate, res (M, N), vec (N),
    epi, raw (True: the product itself is returned as well).  Returns the results (out, or (out, raw)) in order; no autograd."""
    M, dt, dev = problems[0]["a"].shape[0], problems[0]["a"].dtype, problems[0]["a"].device
    n = len(problems)
    structs, results, keep = (_lib.Linear * n)(), [], []
    for s, p in zip(structs, problems):
        a, w = p["a"], p["w"]
        if (w.dim() != 2 or a.shape != (M, w.shape[1]) or a.dtype != dt or w.dtype != dt or a.device != dev or w.device != dev
                or not w.is_contiguous()):
            raise RuntimeError(f"a {tuple(a.shape)} and a contiguous w {tuple(w.shape)} must be (M, K) and (N, K) of one dtype")
        a = a if a.stride(1) == 1 and a.stride(0) % 8 == 0 and a.stride(0) >= a.shape[1] and a.data_ptr() % 16 == 0 else a.clone(memory_format=torch.contiguous_format)
        keep.append(a)
        out = torch.empty((M, w.shape[0]), dtype=dt, device=dev)
        raw = torch.empty_like(out) if p.get("raw") else None
        s.a, s.w, s.out, s.N, s.K, s.lda, s.epi = a.data_ptr(), w.data_ptr(), out.data_ptr(), w.shape[0], w.shape[1], a.stride(0), p.get("epi", 0)
        for name in ("gate", "vec", "res"):
            t = p.get(name)
            if t is not None:
                if t.shape != (out.shape if name != "vec" else out.shape[1:]) or t.dtype != dt or t.device != dev or not t.is_contiguous():
                    raise RuntimeError(f"{name} must be contiguous, of the result's dtype and shape (vec: its columns)")
                setattr(s, name, t.data_ptr())
        if raw is not None:
            s.raw = raw.data_ptr()
        results.append(out if raw is None else (out, raw))
    with _on(dev):
        _lib.check(_lib.lib().vrwkv_linear_group(structs, n, M, _DT[dt], _stream_ptr(dev)))
    return results


def column_sums(x):
    """The sums of a contiguous (..., C) GPU tensor over all but the channels (vrwkv_column_sums): fp32, rounded once."""
    C = x.shape[-1]
    rows = x.numel() // C
    out = torch.empty(C, dtype=x.dtype, device=x.device)
    L = _lib.lib()
    ws_bytes = L.vrwkv_column_sums_workspace_bytes(rows, C)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=x.device)
    with _on(x.device):
        _lib.check(L.vrwkv_column_sums(x.data_ptr(), out.data_ptr(), rows, C, _DT[x.dtype], ws.data_ptr(), ws_bytes, _stream_ptr(x.device)))
    return out


class _AddToTokens(torch.autograd.Function):
    """vector + x for a vector (1, 1, C) and x (B, T, C) of its type, with the vector's gradient in column_sums."""

    @staticmethod
    def forward(ctx, vector, x):
        return vector + x

    @staticmethod
    def backward(ctx, g):
        if not ctx.needs_input_grad[0]:
            return None, g
        own = g.is_cuda and g.numel() > 0 and not torch.is_grad_enabled() and not batched_cotangent(g) and not _transformed()
        return (column_sums(g.contiguous()).view(1, 1, -1) if own else g.sum((0, 1), keepdim=True)), g


def add_to_tokens(vector, x):
    """vector + x, a vector (1, 1, C) added to every token of x (B, T, C)."""
    if (x.is_cuda and torch.is_grad_enabled() and vector.requires_grad and x.dtype in _DT and vector.dtype == x.dtype and x.dim() == 3
            and tuple(vector.shape) == (1, 1, x.shape[-1]) and vector.device == x.device and not torch.is_autocast_enabled("cuda") and not _transformed()):
        return _AddToTokens.apply(vector, x)
    return vector + x


def transposed(weights):
    """The transposes of 1 to 5 contiguous 16-bit matrices, one launch (vrwkv_transpose_group)."""
    n, dev = len(weights), weights[0].device
    outs = [torch.empty(w.shape[1], w.shape[0], dtype=w.dtype, device=dev) for w in weights]
    P, I = ctypes.c_void_p * n, ctypes.c_int * n
    with _on(dev):
        _lib.check(_lib.lib().vrwkv_transpose_group(P(*[w.data_ptr() for w in weights]), P(*[o.data_ptr() for o in outs]),
                                                    I(*[w.shape[0] for w in weights]), I(*[w.shape[1] for w in weights]), n, _stream_ptr(dev)))
    return outs


def sigmoid_gate_backward(y, r, g):
    """Gradients of sigmoid(r) * y for y and r (vrwkv_rowfuse_bwd); all contiguous token matrices of one type."""
    gy, gr = torch.empty_like(y), torch.empty_like(r)
    with _on(y.device):
        _lib.check(_lib.lib().vrwkv_rowfuse_bwd_like(y.data_ptr(), r.data_ptr(), None, None, None, g.data_ptr(), gy.data_ptr(), gr.data_ptr(), None,
                                                     y.numel() // y.shape[-1], y.shape[-1], PRE_NONE, POST_SIGMOID_GATE, 0.0, _DT[y.dtype],
                                                     None, 0, _stream_ptr(y.device)))
    return gy, gr
