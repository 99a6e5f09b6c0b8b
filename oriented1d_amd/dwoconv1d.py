"""Depthwise oriented 1D convolution operator module for MI355X.

Host-side mirror of the reference's operator module (models/dwoconv1d/dwoconv1d.py): same
class names, constructor, parameters (``weight [C,1,1,K]``, ``bias [C]``, ``theta``),
attributes and autograd contract, so ``models/convnext.py:115-127`` can construct it
unchanged.  All arithmetic happens in ``libdwoconv1d_hip.so`` through the C ABI declared
in ``include/dwoconv1d_hip.h``; tensors here only provide device memory and the stream.

Differences from the reference, all supersets:
* bf16/fp16 activations are computed (fp32 accumulate) instead of being reinterpreted as
  float (reference: kernels.cu:25 casts the pointer whatever the dtype).
* ``nhwc=True`` runs NHWC-native kernels; no transposed copies are made
  (reference: dwoconv1d.py:25-26,36-37,50-51,58-59).
* bias add is fused into fprop and the bias gradient into wgrad
  (reference: dwoconv1d.py:34-35,66-67).
* ``arbitrary_size=True`` needs no pad-to-power-of-two / crop round trip
  (reference: dwoconv1d.py:154-187); the kernels take any H, W and give
  ceil(H/stride) x ceil(W/stride) outputs, the same values that path produces.
"""
import ctypes
import weakref

import numpy as np
import torch
import torch.autograd.forward_ad as fwd
import torch.nn as nn

from . import _lib

__all__ = ["DepthwiseOrientedConv1d"]

_DTYPES = {torch.float32: _lib.F32, torch.bfloat16: _lib.BF16, torch.float16: _lib.F16}


def ordinary(*tensors):
    """True for ordinary tensors (None for an absent one) in ordinary execution: no compilation, tracing, torch.func
    transform, dispatch mode, forward-mode derivative or tensor subclass, all of which an autograd function around native
    code would hide a layer from."""
    if (torch.compiler.is_compiling() or torch.jit.is_tracing()
            or torch._C._are_functorch_transforms_active() or torch._C._len_torch_dispatch_stack()):
        return False
    dual = fwd._current_level >= 0
    for t in tensors:
        if t is not None and (type(t) not in _PLAIN or (dual and fwd.unpack_dual(t).tangent is not None)):
            return False
    return True


_PLAIN = (torch.Tensor, nn.Parameter)


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else None


def _check_activation(t, name):
    # models/dwoconv1d/kernels/kernels.cu:11-13,17-18
    if not t.is_cuda:
        raise RuntimeError("%s must be a CUDA tensor" % name)
    if not t.is_contiguous():
        raise RuntimeError("%s must be contiguous" % name)
    if t.dtype not in _DTYPES:
        raise RuntimeError("%s has unsupported dtype %s" % (name, t.dtype))
    if t.dim() != 4:
        raise RuntimeError("%s must be a 4-d tensor" % name)


def build_taps(theta, C, K):
    """Host tap table for ``theta`` ([C] or [C,1] radians) as a uint8 CPU tensor.

    The table is computed by the library on the host in fp32
    (models/dwoconv1d_reference/kernels/kernels.cpp:37,43-44)."""
    lib = _lib.load()
    th = theta.detach().to(device="cpu", dtype=torch.float32).reshape(-1).contiguous()
    if th.numel() != C:
        raise RuntimeError("theta must hold one angle per channel (%d), got %d" % (C, th.numel()))
    blob = torch.empty(lib.dwo_taps_bytes(C, K), dtype=torch.uint8)
    _lib.check(lib.dwo_build_taps(_ptr(th), C, K, _ptr(blob)), "dwo_build_taps")
    return blob


def taps_to_numpy(blob, C, K):
    """(dh, dw) int arrays [C,K] read back from a host tap blob (inspection / tests)."""
    lib = _lib.load()
    dh, dw = np.empty((C, K), np.int32), np.empty((C, K), np.int32)
    a, b = ctypes.c_int(), ctypes.c_int()
    for c in range(C):
        for s in range(K):
            _lib.check(lib.dwo_taps_get(_ptr(blob), c, s, ctypes.byref(a), ctypes.byref(b)),
                       "dwo_taps_get")
            dh[c, s], dw[c, s] = a.value, b.value
    return dh, dw


class _TapCache:
    """Device tap tables, one per (theta tensor, device, C, K), rebuilt when theta is modified
    or moved.  A module owns one (a single entry in practice); the five-function tuple of
    ``oriented_dwconv1d_get_module_from_params`` owns one that may serve several layers, so the
    few most recent tables are kept."""

    KEEP = 8

    def __init__(self):
        # (id(theta), device, C, K) -> (state key, weak ref, device blob, layouts by element size)
        self.entries = {}

    def get(self, theta, C, K, device):
        """The device tap table."""
        return self.lookup(theta, C, K, device)[0]

    def lookup(self, theta, C, K, device):
        """(device tap table, {element size: layout code of an NHWC call}): ``GROUPED`` is added
        where every 16 bytes of channels share an orientation."""
        slot = (id(theta), device, C, K)
        state = (theta.data_ptr(), theta._version)
        hit = self.entries.get(slot)
        if hit is None or hit[0] != state or hit[1]() is not theta:
            if len(self.entries) >= self.KEEP:
                self.entries.pop(next(iter(self.entries)))
            blob = build_taps(theta, C, K)
            grouped = _lib.load().dwo_taps_grouped
            layouts = {size: _lib.NHWC + (_lib.GROUPED if grouped(_ptr(blob), 16 // size) else 0)
                       for size in (2, 4)}
            hit = (state, weakref.ref(theta), blob.to(device), layouts)
            self.entries[slot] = hit
        return hit[2], hit[3]


def _dims(x, nhwc):
    if nhwc:
        N, H, W, C = x.shape
    else:
        N, C, H, W = x.shape
    return N, C, H, W


_F32_COPIES = {}  # id(parameter) -> (weak reference, state key, fp32 copy)


def f32_copy(p):
    """fp32 contiguous copy of a parameter, kept until the parameter is modified or moved (the
    library takes weights, biases and norm parameters as fp32; re-casting 16-bit parameters at
    every call costs a kernel launch each)."""
    if p.dtype == torch.float32 and p.is_contiguous():
        return p.detach()
    key = (p._version, p.data_ptr(), p.dtype, p.device)
    hit = _F32_COPIES.get(id(p))
    if hit is None or hit[0]() is not p or hit[1] != key:
        pid = id(p)
        ref = weakref.ref(p, lambda _, pid=pid: _F32_COPIES.pop(pid, None))
        hit = (ref, key, p.detach().to(torch.float32).contiguous())
        _F32_COPIES[pid] = hit
    return hit[2]


def fprop(x, w, taps, stride=1, bias=None, nhwc=False):
    """y = fprop(x, w, theta) (+ bias).  x: [N,C,H,W] or [N,H,W,C]; w: [C,1,1,K].  ``nhwc`` is a
    truth value or, here and below, a layout code of ``_TapCache.lookup``."""
    b = f32_copy(bias) if bias is not None else None
    return _lib.host(x.get_device()).fprop(x, w, taps, stride, b, int(nhwc))


def dgrad(dy, w, taps, in_hw, stride=1, nhwc=False):
    """dx = dgrad(dy, w, theta); ``in_hw`` is the (H, W) of the forward input."""
    H, W = in_hw
    return _lib.host(dy.get_device()).dgrad(dy, w, taps, H, W, stride, int(nhwc))


def wgrad(dy, x, taps, K, stride=1, nhwc=False, with_bias=False):
    """(dw [C,1,1,K] fp32, db [C] fp32 or None) = wgrad(dy, x, theta)."""
    return _lib.host(x.get_device()).wgrad(dy, x, taps, K, stride, int(nhwc), with_bias)


class KernelTuple(tuple):
    """The reference's five-function tuple ``(fprop, dgrad, wgrad, nhwc_to_nchw, nchw_to_nhwc)``
    (models/dwoconv1d/dwoconv1d.py:72-80) plus what the native path needs to run without the
    transposes: kernel size, stride, a tap-table cache, and whether extents that the stride does
    not divide are accepted."""

    def __new__(cls, functions, kernel_size, stride, arbitrary_size):
        self = super().__new__(cls, functions)
        self.kernel_size, self.stride = kernel_size, stride
        self.arbitrary_size = arbitrary_size
        self.taps = _TapCache()
        return self

    def __reduce__(self):
        # copies (copy.deepcopy of a model, e.g. for an averaged twin) and pickles are rebuilt
        # from the parameters; the tap cache starts empty
        return (oriented_dwconv1d_get_module_from_params,
                ("float", self.kernel_size, self.stride, self.kernel_size // 2,
                 4 if self.arbitrary_size else 1))


class _DepthwiseOrientedConv1d(torch.autograd.Function):
    """Autograd contract of models/dwoconv1d/dwoconv1d.py:18-69.

    ``apply(x, w, theta, bias, module, nhwc, resid)``.  ``module`` is what the reference passes
    in this slot, the tuple returned by ``oriented_dwconv1d_get_module_from_params`` (a
    ``KernelTuple`` here): the convolution then runs natively in the tensor's layout with the
    bias fused.  Any other 5-tuple of callables is driven exactly as the reference drives its
    own (transposes, separate bias add, ``dy.sum``), and the owning ``DepthwiseOrientedConv1d``
    is accepted as well.  backward returns (dx, dw, None, db, None, None, None): theta never
    receives a gradient (dwoconv1d.py:64)."""

    @staticmethod
    def forward(ctx, x, w, theta, bias, module, nhwc=False, resid=None):
        ctx.set_materialize_grads(False)
        if isinstance(module, DepthwiseOrientedConv1d):
            module = module.module_fp32_large if module.arbitrary_size else module.module_fp32
        ctx.plain = None
        if not isinstance(module, KernelTuple):
            return _DepthwiseOrientedConv1d._forward_plain(ctx, x, w, theta, bias, module, nhwc,
                                                           resid)
        stride = module.stride
        C = w.shape[0]
        K = w.shape[-1]
        if K != module.kernel_size:
            raise RuntimeError("weight has %d taps, the kernel tuple was made for %d"
                               % (K, module.kernel_size))
        w_eff = f32_copy(w)
        if resid is not None:
            w_eff = w_eff + resid.to(w_eff)
        x = x.contiguous()
        _check_activation(x, "x")
        _, Cx, H, W = _dims(x, nhwc)
        if Cx != C:
            raise RuntimeError("input has %d channels, weight has %d" % (Cx, C))
        if not module.arbitrary_size and (H % stride != 0 or W % stride != 0):
            # models/dwoconv1d/kernels/kernels.cu:20
            raise RuntimeError("Invalid input size: H,W not divisible by stride")
        taps, layouts = module.taps.lookup(theta, C, K, x.device)
        layout = layouts[x.element_size()] if nhwc else _lib.NCHW

        ctx.stride, ctx.nhwc, ctx.K = stride, layout, K
        ctx.with_bias = bias is not None
        ctx.w_dtype = w.dtype
        ctx.b_dtype = bias.dtype if bias is not None else None
        ctx.save_for_backward(x, w_eff, taps)
        return fprop(x, w_eff, taps, stride, bias=bias, nhwc=layout)

    @staticmethod
    def _forward_plain(ctx, x, w, theta, bias, module, nhwc, resid):
        # models/dwoconv1d/dwoconv1d.py:21-38, for a caller's own five functions
        f, _, _, nhwc_to_nchw, nchw_to_nhwc = module
        if resid is not None:
            w = w + resid
        x = x.contiguous()
        if nhwc:
            x = nhwc_to_nchw(x)
        ctx.plain, ctx.nhwc = module, nhwc
        ctx.save_for_backward(x, w, theta, bias)
        y = f(x, w, theta)
        if bias is not None:
            y = y + bias.to(y).view(1, -1, 1, 1)
        return nchw_to_nhwc(y) if nhwc else y

    @staticmethod
    def backward(ctx, dy):
        if dy is None:
            return None, None, None, None, None, None, None
        if ctx.plain is not None:
            # models/dwoconv1d/dwoconv1d.py:45-69
            _, d, g, nhwc_to_nchw, nchw_to_nhwc = ctx.plain
            x, w, theta, bias = ctx.saved_tensors
            dy = dy.contiguous()
            if ctx.nhwc:
                dy = nhwc_to_nchw(dy)
            dx = dw = db = None
            if ctx.needs_input_grad[0]:
                dx = d(dy, w, theta)
                if ctx.nhwc:
                    dx = nchw_to_nhwc(dx)
            if ctx.needs_input_grad[1]:
                dw = g(dy, x, theta)
            if bias is not None and ctx.needs_input_grad[3]:
                db = dy.sum(dim=[0, 2, 3])
            return dx, dw, None, db, None, None, None
        x, w_eff, taps = ctx.saved_tensors
        dy = dy.contiguous()
        if dy.dtype != x.dtype:
            dy = dy.to(x.dtype)
        N, C, H, W = _dims(x, ctx.nhwc)
        dx = dw = db = None
        if ctx.needs_input_grad[0]:
            dx = dgrad(dy, w_eff, taps, (H, W), ctx.stride, nhwc=ctx.nhwc)
        need_db = ctx.with_bias and ctx.needs_input_grad[3]
        if ctx.needs_input_grad[1]:
            dw, db32 = wgrad(dy, x, taps, ctx.K, ctx.stride, nhwc=ctx.nhwc, with_bias=need_db)
            if ctx.w_dtype != torch.float32:
                dw = dw.to(ctx.w_dtype)
            if need_db:
                db = db32 if ctx.b_dtype == torch.float32 else db32.to(ctx.b_dtype)
        elif need_db:
            red = [0, 1, 2] if ctx.nhwc else [0, 2, 3]
            db = dy.sum(dim=red, dtype=torch.float32).to(ctx.b_dtype)
        return dx, dw, None, db, None, None, None


def oriented_dwconv1d_get_module_from_params(ftype, kernel_size, stride, pad, Sb=None):
    """Five-function tuple in the reference's order (models/dwoconv1d/dwoconv1d.py:72-80):
    (fprop(x,w,theta), dgrad(dy,w,theta), wgrad(dy,x,theta), nhwc_to_nchw, nchw_to_nhwc),
    all on contiguous NCHW tensors; the result goes into slot 5 of
    ``_DepthwiseOrientedConv1d.apply`` as in the reference (dwoconv1d.py:189-198).
    ``ftype`` and ``pad`` are accepted for signature compatibility: there is nothing to compile
    per configuration and pad is always ``kernel_size // 2``.  The kernels need no filter
    partitioning; ``Sb=4`` is how the reference asks for its arbitrary-size variant
    (dwoconv1d.py:150-152), so such a tuple accepts extents the stride does not divide
    (output ceil(H/stride)), any other rejects them as kernels.cu:20 does."""
    K = int(kernel_size)
    stride = int(stride)
    arbitrary = Sb is not None and int(Sb) > 1

    def f(x, w, theta):
        if not arbitrary and (x.shape[2] % stride != 0 or x.shape[3] % stride != 0):
            raise RuntimeError("Invalid input size: H,W not divisible by stride")
        return fprop(x, w, kt.taps.get(theta, x.shape[1], K, x.device), stride)

    def d(dy, w, theta):
        hw = (dy.shape[2] * stride, dy.shape[3] * stride)
        return dgrad(dy, w, kt.taps.get(theta, dy.shape[1], K, dy.device), hw, stride)

    def g(dy, x, theta):
        return wgrad(dy, x, kt.taps.get(theta, x.shape[1], K, x.device), K, stride)[0].to(x.dtype)

    def nhwc_to_nchw(x):
        return x.permute(0, 3, 1, 2).contiguous()

    def nchw_to_nhwc(x):
        return x.permute(0, 2, 3, 1).contiguous()

    kt = KernelTuple((f, d, g, nhwc_to_nchw, nchw_to_nhwc), K, stride, arbitrary)
    return kt


def _is_f32(p):
    return p.dtype == torch.float32 and p.is_contiguous()


def _native_covers(x, w, theta, bias, resid, module, nhwc):
    """True for the calls that the native autograd node takes: ordinary tensors on one GPU whose sizes and types pass every check
    of the Python function (which reports the others)."""
    if not (x.is_cuda and x.dtype in _DTYPES and x.dim() == 4 and type(module) is KernelTuple
            and w.shape[-1] == module.kernel_size and x.device == w.device and w.is_floating_point()
            and (bias is None or bias.device == x.device) and (resid is None or resid.device == x.device)
            and ordinary(x, w, theta, bias, resid)):
        return False
    _, C, H, W = _dims(x, nhwc)
    return C == w.shape[0] and (module.arbitrary_size or (H % module.stride == 0 and W % module.stride == 0))


class DepthwiseOrientedConv1d(nn.Conv2d):
    """Drop-in for models/dwoconv1d/dwoconv1d.py:92-198.

    ``padding`` only shapes the parent ``nn.Conv2d``; the compute path always pads by
    ``kernel_size // 2`` (dwoconv1d.py:133)."""

    def __init__(
        self,
        in_channels,
        out_channels,
        kernel_size=3,
        *,
        groups=1,
        stride=1,
        padding=1,
        bias=True,
        angle=0,
        nhwc=False,
        resid=False,
        arbitrary_size=False,
    ):
        super().__init__(
            in_channels,
            out_channels,
            (1, kernel_size),
            groups=groups,
            stride=stride,
            padding=(0, padding),
            bias=bias,
        )
        assert (
            isinstance(kernel_size, int)
            and in_channels == out_channels
            and groups == in_channels
            and kernel_size % 2 == 1
        )
        assert self.stride[0] == self.stride[1]
        assert kernel_size <= 63 and self.stride[0] in (1, 2, 4)

        if isinstance(angle, (float, int)):
            angle = torch.zeros((in_channels, 1)) + angle
        self.theta = nn.Parameter(torch.as_tensor(angle, dtype=torch.float32).clone(),
                                  requires_grad=True)
        self.nhwc = nhwc
        self.arbitrary_size = arbitrary_size
        pad = kernel_size // 2
        if resid:
            onehot = torch.zeros_like(self.weight.detach())
            onehot[:, :, :, pad:pad + 1] = 1
            # follows .to()/.cuda() with the module, not part of the state_dict
            self.register_buffer("resid", onehot, persistent=False)
        else:
            self.resid = None
        # models/dwoconv1d/dwoconv1d.py:144-152: the tuples forward() hands to apply()
        self.module_fp32 = oriented_dwconv1d_get_module_from_params(
            "float", kernel_size, self.stride[0], pad, Sb=1)
        if arbitrary_size:
            self.module_fp32_large = oriented_dwconv1d_get_module_from_params(
                "float", kernel_size, self.stride[0], pad, Sb=4)

    def _apply(self, fn, recurse=True):
        """``.to()/.half()/.bfloat16()/.cuda()`` move and cast weight and bias, but the angles stay
        fp32: they are geometry, and their tap offsets (``(int)(cosf(theta) * k)``) change when
        theta is rounded to a 16-bit type (the reference supports fp32 only and would
        reinterpret the bits, kernels.cu:25)."""
        theta = self.theta.data
        super()._apply(fn, recurse)
        if self.theta.dtype != torch.float32:
            self.theta.data = theta.to(self.theta.device)
        return self

    @property
    def _taps(self):
        """Tap-table cache of the tuple forward() uses."""
        return (self.module_fp32_large if self.arbitrary_size else self.module_fp32).taps

    def forward_safe(self, x):
        """Arbitrary H, W (reference: dwoconv1d.py:154-187): no padding to a power of two, no
        crop and no permuted copies; the kernels produce ceil(H/stride) x ceil(W/stride)
        outputs in the tensor's own layout, the values that path returns."""
        return self._apply_operator(x, self.module_fp32_large)

    def forward(self, x):
        if self.arbitrary_size:  # the reference rebinds forward to forward_safe (:148-149)
            return self.forward_safe(x)
        return self._apply_operator(x, self.module_fp32)

    def _apply_operator(self, x, module):
        w, theta, bias, resid = self.weight, self.theta, self.bias, self.resid
        nhwc = bool(self.nhwc)
        if _native_covers(x, w, theta, bias, resid, module, nhwc):
            # the native node: the same checks, kernels and gradients without Python in the backward pass
            C, K = w.shape[0], w.shape[-1]
            taps, layouts = module.taps.lookup(theta, C, K, x.device)
            return _lib.host(x.get_device()).convolution(
                x, w, bias, None if _is_f32(w) else f32_copy(w),
                None if bias is None or _is_f32(bias) else f32_copy(bias), resid, taps, theta, module.stride,
                layouts[x.element_size()] if nhwc else _lib.NCHW)
        return _DepthwiseOrientedConv1d.apply(x, w, theta, bias, module, self.nhwc, resid)
