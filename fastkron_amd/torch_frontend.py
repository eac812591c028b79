"""PyTorch front end over libFastKron.so for tensors that live in HBM.

Mirrors the reference's `pyfastkron` interface (reference pyfastkron/fastkrontorch.py:404-465 `gemkm` /
`gekmm`, :340-401 the autograd functions `MKM` / `KMM`, pyfastkron/fastkronbase.py:104-518 the shape,
broadcast and batching rules):

* operands may carry leading batch dimensions, broadcast between X, the factors and Y the NumPy way; the
  batch dimensions become one strided-batched library call (stride 0 = shared operand) where one remains after neighbours
  that all operands have alike are merged, or two of which the factors have one; further ones a host loop; a batch of X
  against shared factors (MKM) is folded into the row count instead;
* a tensor whose last two dimensions are a transposed view of a row-major buffer is passed as that buffer
  with `fastKronOp_T` instead of being copied (reference fastkrontorch.py:66-76);
* 1-D X is a single row (MKM) or column (KMM);
* with gradients of factors required, the library's gradient functions (include/fastkron_ext.h) run the forward
  pass keeping every step's input and the backward pass through the steps (reference fastkrontorch.py:160-217);
  when only X needs a gradient the backward pass is one fused library call with the transposed factors.

PyTorch supplies memory and streams; the arithmetic of both passes is the library's HIP kernels, but for two parts: the
gradient of the input of a step with a wide factor is PyTorch's product (`wideStep` in csrc/frontend.cpp has the rule and
the measurements), and a backward pass that is itself differentiated (create_graph=True) or takes a batch of gradients
(is_grads_batched) is composed of PyTorch operations.  CPU tensors and dtypes other than
float32 / float64 are errors: there is no fallback path (the reference falls back to a shuffle algorithm
built from `torch.matmul`, fastkronbase.py:478-518).
"""
import ctypes
import importlib.machinery
import importlib.util
import math
import os

import torch

import fastkron_amd
from . import capi

__all__ = ["gemkm", "gekmm", "MKM", "KMM"]


def _load_native():
    """The host path in native code (csrc/frontend.cpp), bound to the library that capi has loaded."""
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "lib", "_frontend.so")
    if not os.path.exists(path):
        raise RuntimeError(f"{path} is missing: build it with fastkron_amd/csrc/build.sh (or __graft_entry__.build())")
    loader = importlib.machinery.ExtensionFileLoader("_frontend", path)
    m = importlib.util.module_from_spec(importlib.util.spec_from_loader("_frontend", loader))
    loader.exec_module(m)
    lib = capi.load()
    names = ["sgemkm", "dgemkm", "sgekmm", "dgekmm", "sgemkmStridedBatched", "dgemkmStridedBatched", "sgekmmStridedBatched",
             "dgekmmStridedBatched", "gekmmSizes", "fastKronSetStream", "fastKronProductOuter", "fastKronGradSizes", "fastKronGradForward",
             "fastKronGradBackwardSteps"]                 # the order of csrc/frontend.cpp
    m.use(tuple(ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in names))
    return m


_native = _load_native()


def _prod(v):
    return int(math.prod(v)) if len(v) else 1


def _validate(mm, x, fs, y):
    if not isinstance(x, torch.Tensor):
        raise ValueError("Input 'x' should be a Tensor")
    if not isinstance(fs, (list, tuple)) or len(fs) == 0:
        raise ValueError("Input 'fs' should be a list of Tensor")
    for i, f in enumerate(fs):
        if not isinstance(f, torch.Tensor):
            raise ValueError(f"Input fs[{i}] should be a Tensor")
        if f.ndim < 2:
            raise ValueError(f"Input fs[{i}] should have at least two dimensions")
    if y is not None and not isinstance(y, torch.Tensor):
        raise ValueError("Input 'y' should be a Tensor")
    tensors = [x] + list(fs) + ([y] if y is not None else [])
    devices = {t.device for t in tensors}
    if len(devices) != 1:
        raise RuntimeError(f"Expected all tensors to be on the same device, but found {sorted(str(d) for d in devices)}")
    if not x.is_cuda:
        raise RuntimeError("fastkron_amd runs on HBM-resident tensors only: there is no CPU path")
    if x.dtype not in (torch.float32, torch.float64):
        raise TypeError(f"float32 and float64 only, got {x.dtype}")
    if any(t.dtype != x.dtype for t in tensors):
        raise ValueError(f"Operand types mismatch: {[t.dtype for t in tensors]}")
    for f in fs[1:]:
        if f.shape[:-2] != fs[0].shape[:-2]:
            raise ValueError(f"Batched dims of factors do not match: {fs[0].shape[:-2]} != {f.shape[:-2]}")


def _refused(mm, x, fs, beta, y, where):
    """Raises for operands that the native path did not take."""
    _validate(mm, x, fs, y)
    if beta != 0.0 and y is None:
        raise ValueError(f"When beta != 0 ({beta}) then y should not be None")
    is_vec = x.ndim == 1
    if is_vec:
        x = x.reshape(1, -1) if mm == "mkm" else x.reshape(-1, 1)
    if mm == "mkm":
        M, K = x.shape[-2], x.shape[-1]
        Ps, Qs = [f.shape[-2] for f in fs], [f.shape[-1] for f in fs]
    else:
        K, M = x.shape[-2], x.shape[-1]
        Ps, Qs = [f.shape[-1] for f in fs], [f.shape[-2] for f in fs]
    if K != _prod(Ps):
        raise ValueError(f"Input operand x has a mismatch with its dimension ('{K}') with the rows of the "
                         f"Kronecker product of fs ('{_prod(Ps)}')")
    xbatch, fbatch = tuple(x.shape[:-2]), tuple(fs[0].shape[:-2])
    try:
        zbatch = tuple(torch.broadcast_shapes(xbatch, fbatch))
    except RuntimeError:
        raise ValueError(f"Shape {xbatch} of x and {fbatch} of fs are not broadcastable")
    zshape = zbatch + ((M, _prod(Qs)) if mm == "mkm" else (_prod(Qs), M))
    if y is not None:
        if is_vec and y.ndim == 1:
            y = y.reshape(1, -1) if mm == "mkm" else y.reshape(-1, 1)
        if tuple(y.shape[-2:]) != zshape[-2:]:
            raise ValueError(f"Input operand 'y' shape {tuple(y.shape)} mismatch with output {zshape}")
        try:
            ok = tuple(torch.broadcast_shapes(tuple(y.shape[:-2]), zbatch)) == zbatch
        except RuntimeError:
            ok = False
        if not ok:
            raise ValueError(f"Input operand 'y' shape {tuple(y.shape)} cannot be broadcasted to output {zshape}")
    raise fastkron_amd.FastKronError(capi.INVALID_KMM_PROBLEM, where)        # more factors than the library takes, or empty ones


def _handle():
    """(handle, current stream) as whole numbers"""
    h = fastkron_amd.default_handle()
    return h.h.value, torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


def _result(r, mm, x, fs, beta, y, where):
    if r is None:
        _refused(mm, x, fs, beta, y, where)
    if r.__class__ is int:
        raise fastkron_amd.FastKronError(r, where)
    return r


def _run(mm, x, fs, alpha, beta, y):
    """The product, or False when the call is to be recorded for gradients."""
    if fastkron_amd._default is None:
        _validate(mm, x, fs, y)                            # (before a handle is made, which needs a GPU)
    h, stream = _handle()
    return _result(_native.product(h, stream, mm == "mkm", x, fs, alpha, beta, y), mm, x, fs, beta, y, "gemkm" if mm == "mkm" else "gekmm")


def _sum_to(g, shape):
    """Reduce a gradient over the dimensions that were broadcast in the forward pass."""
    return g.sum_to_size(shape) if tuple(g.shape) != tuple(shape) else g


def _matrix(mm, v):
    """Vectors as matrices of one row (MKM) or column (KMM)."""
    return v.unsqueeze(-2 if mm == "mkm" else -1)


def _differentiable_backward(grad_z, x, fs, need_x, need_f):
    """Gradients of Z = X (F_0 (x) ... (x) F_{N-1}) from PyTorch operations, for backward passes that are themselves
    differentiated (create_graph) or take a batch of gradients at once (vmap).  Step of factor i maps rows (m, s) of its input, reshaped (M*S, P_i), through F_i and
    stores column q at q*S + s; its backward un-shuffles the output gradient to (M*S, Q_i) first."""
    M = x.shape[-2]
    inputs = [x]                                          # of the steps, last factor first
    for f in reversed(fs[1:] if any(need_f) else ()):
        P, Q = f.shape[-2:]
        t = inputs[-1]
        S = t.shape[-1] // P
        o = t.reshape(t.shape[:-2] + (M * S, P)) @ f
        inputs.append(o.reshape(o.shape[:-2] + (M, S, Q)).transpose(-1, -2).reshape(o.shape[:-2] + (M, S * Q)))
    inputs.reverse()
    g = grad_z
    grad_fs = []
    for i, f in enumerate(fs):
        P, Q = f.shape[-2], f.shape[-1]
        S = g.shape[-1] // Q
        a = g.reshape(g.shape[:-2] + (M, Q, S)).transpose(-1, -2).reshape(g.shape[:-2] + (M * S, Q))
        if need_f[i]:
            inp = inputs[i].reshape(inputs[i].shape[:-2] + (M * S, P))
            grad_fs.append(_sum_to((inp.mT.contiguous() @ a), f.shape))
        else:
            grad_fs.append(None)
        if i + 1 < len(fs) or need_x:
            g = (a @ f.mT.contiguous()).reshape(a.shape[:-2] + (M, S * P))
    return (_sum_to(g, x.shape) if need_x else None), grad_fs


def _forward(mm, ctx, x, fs):
    ctx.nf, ctx.kept = len(fs), any(f.requires_grad for f in fs)
    if ctx.kept:
        h, stream = _handle()
        z, save, ctx.opX, ctx.opF = _result(_native.grad_forward(h, stream, mm == "mkm", x, fs), mm, x, fs, 0.0, None, "fastKronGradForward")
        ctx.save_for_backward(x, *fs, save)
    else:
        z = _run(mm, x, fs, 1.0, 0.0, None)
        ctx.save_for_backward(x, *fs)
    return z


def _backward(mm, ctx, grad_z):
    saved = ctx.saved_tensors
    x, fs = saved[0], saved[1:ctx.nf + 1]
    need_x, need_f = ctx.needs_input_grad[0], ctx.needs_input_grad[1:ctx.nf + 1]
    batched = _native.batched(grad_z)                      # is_grads_batched, jacobian(vectorize=True)
    if not any(need_f) and not batched:
        # one fused library call on the transposed views: dX = dZ (F_0^T (x) ...) for MKM, (F_0^T (x) ...) dZ for KMM
        # (itself recorded where the backward pass is differentiated)
        if not need_x:
            return (None,) * (ctx.nf + 1)
        # (a vector against a batch of factors has one result per entry: each a matrix of one row / column)
        vec = x.ndim == 1 and grad_z.ndim > 1
        gz, fts = _matrix(mm, grad_z) if vec else grad_z, [f.mT for f in fs]
        gx = gemkm(gz, fts) if mm == "mkm" else gekmm(fts, gz)
        return (_sum_to(gx, _matrix(mm, x).shape).reshape(x.shape) if vec else _sum_to(gx, x.shape),) + (None,) * ctx.nf
    if not torch.is_grad_enabled() and not batched:
        h, stream = _handle()
        return _result(_native.grad_backward(h, stream, mm == "mkm", x, fs, ctx.opX, ctx.opF, grad_z, saved[-1], need_x, need_f), mm, x, fs,
                       0.0, None, "fastKronGradBackward")
    matrix = lambda t: _matrix(mm, t) if x.ndim == 1 else t
    if mm == "mkm":
        gx, gfs = _differentiable_backward(matrix(grad_z), matrix(x), fs, need_x, need_f)
        return (gx.reshape(x.shape) if gx is not None else None,) + tuple(gfs)
    # Z^T = X^T (F_0^T (x) ...): the MKM rule on the transposed tensors
    gx, gfs = _differentiable_backward(matrix(grad_z).mT, matrix(x).mT, [f.mT for f in fs], need_x, need_f)
    return (gx.mT.reshape(x.shape) if gx is not None else None,) + tuple(g.mT if g is not None else None for g in gfs)


class MKM(torch.autograd.Function):
    """Z = X (F_0 (x) ... (x) F_{N-1}) with gradients (reference fastkrontorch.py:340-357)."""

    @staticmethod
    def forward(ctx, x, *fs):
        return _forward("mkm", ctx, x, fs)

    @staticmethod
    def backward(ctx, grad_z):
        return _backward("mkm", ctx, grad_z)


class KMM(torch.autograd.Function):
    """Z = (F_0 (x) ... (x) F_{N-1}) X with gradients (reference fastkrontorch.py:360-378); the arguments
    are (x, *fs) as in the reference."""

    @staticmethod
    def forward(ctx, x, *fs):
        return _forward("kmm", ctx, x, fs)

    @staticmethod
    def backward(ctx, grad_z):
        return _backward("kmm", ctx, grad_z)


def _no_epilogue_with_grad(mm, x, fs, alpha, beta, y):
    if y is not None:
        _validate(mm, x, fs, y)
    if alpha != 1:
        raise ValueError(f"When requires_grad is True alpha should be 1 but is {alpha}")
    if beta != 0:
        raise ValueError(f"When requires_grad is True beta should be 0 but is {beta}")
    if y is not None:
        raise ValueError("When requires_grad is True y should be None")


def gemkm(x, fs, alpha=1.0, beta=0.0, y=None):
    """Z = alpha * X (F_0 (x) ... (x) F_{N-1}) + beta * Y.  X is (.., M, prod P) or a vector of prod P elements,
    fs[i] is (.., P_i, Q_i), Y broadcastable to Z (reference fastkrontorch.py:404-434)."""
    z = _run("mkm", x, fs, float(alpha), float(beta), y)
    if z is False:
        _no_epilogue_with_grad("mkm", x, fs, alpha, beta, y)
        return MKM.apply(x, *fs)
    return z


def gekmm(fs, x, alpha=1.0, beta=0.0, y=None):
    """Z = alpha * (F_0 (x) ... (x) F_{N-1}) X + beta * Y.  X is (.., prod P, M) or a vector, fs[i] is
    (.., Q_i, P_i) (reference fastkrontorch.py:437-465)."""
    z = _run("kmm", x, fs, float(alpha), float(beta), y)
    if z is False:
        _no_epilogue_with_grad("kmm", x, fs, alpha, beta, y)
        return KMM.apply(x, *fs)
    return z
