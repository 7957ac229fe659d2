"""The two passes a WTConvNeXt block makes around its WTConv layer, each as one HIP kernel
(`wtconv_channel_norm`, `wtconv_block_residual` of the C ABI), GPU only; with their backward kernels
(`wtconv_channel_norm_backward`, `wtconv_block_residual_backward`) behind autograd functions for training.

Reference semantics: `x.permute(0, 2, 3, 1)` + `nn.LayerNorm` after `conv_dw`
(wtconvnext/wtconvnext.py:132-133), `LayerNorm2d` of the stem and downsample layers (:171, :296), and
`permute(0, 3, 1, 2)` + `mul(gamma)` + shortcut add at the end of the block (:135-140)."""
import ctypes

import torch
from torch.autograd import forward_ad as _forward_ad
from torch.nn.modules import module as _nn
from torch.utils._device import DeviceContext

from . import _ext, _lib
from .modules import _param

_DT = {torch.float32: _lib.F32, torch.bfloat16: _lib.BF16}


def records(x, *params):
    """Whether autograd would record an operation on these tensors."""
    return torch.is_grad_enabled() and (x.requires_grad or any(p is not None and p.requires_grad for p in params))


def _tangents(*tensors):
    """Whether forward-mode differentiation follows any of these tensors."""
    return _forward_ad._current_level >= 0 and any(t is not None and _forward_ad.unpack_dual(t).tangent is not None for t in tensors)


def usable(x, *params, training=False):
    """Whether the kernels take this call: a contiguous fp32 / bf16 GPU tensor with an even channel count, parameters
    of one fp32 / bf16 dtype on the same device, no autocast, no forward-mode differentiation (the kernels have no tangents
    and raw pointers would lose them without a word), not under torch.compile.  With training=False also:
    nothing recorded for autograd (the plain functions below take raw pointers; the *_fn variants are the ones that
    autograd can differentiate)."""
    if not training and records(x, *params):
        return False
    if torch.compiler.is_compiling():
        return False
    if torch.is_autocast_enabled():      # autocast keeps LayerNorm outputs and the residual stream in fp32; the kernels return x.dtype
        return False
    if not x.is_cuda or x.dtype not in _DT or x.dim() != 4 or x.shape[1] % 2 or not x.is_contiguous():
        return False
    if _tangents(x, *params):
        return False
    pd = None
    for p in params:
        if p is None:
            continue
        if p.device != x.device or p.dtype not in _DT or not p.is_contiguous() or (pd is not None and p.dtype != pd):
            return False
        pd = p.dtype
    return True


def usable_nhwc(y, shortcut):
    """Whether the residual kernels take the MLP output `y` (B, H, W, C) for this shortcut: same dtype and device."""
    return y.dtype == shortcut.dtype and y.device == shortcut.device and y.dim() == 4 and not _tangents(y, shortcut)


def _watched(*modules):
    """Whether something expects to see these modules called, or the functions they call: hooks of the modules or of all
    modules, a `forward` put on a module itself, a dispatch or function mode (FLOP counters, tracers).  The function mode
    of a default device only looks at factory functions."""
    native = _ext.lookups()
    if native is not None:
        return native.watched(*modules)
    if _nn._global_forward_hooks or _nn._global_forward_pre_hooks or torch._C._len_torch_dispatch_stack():
        return True
    for m in modules:
        own = m.__dict__
        if own["_forward_hooks"] or own["_forward_pre_hooks"] or "forward" in own:
            return True
    for i in range(torch._C._len_torch_function_stack()):
        if type(torch._C._get_function_stack_at(i)) is not DeviceContext:
            return True
    return False


def _watched_backward(*modules):
    """Whether something expects to see gradients at the borders of these modules."""
    return bool(_nn._global_backward_hooks or _nn._global_backward_pre_hooks
                or any(m.__dict__["_backward_hooks"] or m.__dict__["_backward_pre_hooks"] for m in modules))


_PLAIN = (torch.Tensor, torch.nn.Parameter, type(None))


def block_mlp(x, shortcut, norm, mlp, gamma):
    """shortcut + gamma * fc2(gelu(fc1(norm(x)))) of a WTConvNeXt block, with x and shortcut (B, C, H, W), in one kernel;
    None where it does not apply: autograd records, another dtype than bfloat16, a channel count without a kernel, an
    activation other than the exact GELU, observers that expect to see the modules called, or tensors of a subclass
    (quantised or sharded weights bring their own product, and often no memory that a kernel could read)."""
    if torch.compiler.is_compiling() or torch.is_autocast_enabled():      # (first: loading the binding is not traceable)
        return None
    ext = _ext.get()
    if ext is None:
        return None
    native = _ext.lookups()
    args = (_mlp_args if native is None else native.mlp_args)(x, shortcut, norm, mlp, gamma)
    return None if args is None else ext.block_mlp(*args)


def _mlp_args(x, shortcut, norm, mlp, gamma):
    """What the binding's mlp_args() gives."""
    fc1, act, fc2 = mlp.fc1, mlp.act, mlp.fc2
    if (type(fc1) is not torch.nn.Linear or type(fc2) is not torch.nn.Linear or type(act) is not torch.nn.GELU
            or act.approximate != "none" or _watched(norm, mlp, fc1, act, fc2)):
        return None
    args = (x, shortcut, _param(norm), _param(norm, "bias"), norm.eps, _param(fc1), _param(fc1, "bias"), _param(fc2),
            _param(fc2, "bias"), gamma)
    if args[2] is None or args[3] is None or any(type(t) not in _PLAIN for t in args[:4] + args[5:]):
        return None
    return args


def patch_conv(x, seq, conv, norm, stem):
    """The stem (`conv` 4 x 4 with stride 4, then `norm` over the channels) or a downsample layer (`norm`, then `conv` 2 x 2
    with stride 2) of a WTConvNeXt, the two modules of `seq`, in one kernel; None where it does not apply: autograd records,
    another dtype than bfloat16, sizes without a kernel, another kind of convolution, observers that expect to see the
    modules called, or tensors of a subclass."""
    if torch.compiler.is_compiling() or torch.is_autocast_enabled():      # (first: loading the binding is not traceable)
        return None
    ext = _ext.get()
    if ext is None:
        return None
    size = (4, 4) if stem else (2, 2)
    if (type(conv) is not torch.nn.Conv2d or conv.kernel_size != size or conv.stride != size or conv.dilation != (1, 1)
            or conv.groups != 1 or conv.padding not in ((0, 0), "valid") or _watched(seq, conv, norm)):
        return None
    args = (_param(conv), _param(conv, "bias"), _param(norm), _param(norm, "bias"))
    for t in (x, *args):
        if t is None or type(t) not in _PLAIN:
            return None
    return ext.patch_conv(x, *args, norm.eps, stem)


def pool_norm(x, norm):
    """`norm` (a LayerNorm over the channels) of the mean of x (B, C, H, W) over its pixels, (B, C), as one kernel; None where
    it does not apply: autograd records, other dtypes than float32 and bfloat16, observers that expect to see the module
    called, or tensors of a subclass."""
    if torch.compiler.is_compiling() or torch.is_autocast_enabled():      # (first: loading the binding is not traceable)
        return None
    ext = _ext.get()
    if ext is None or _watched(norm):
        return None
    weight, bias = _param(norm), _param(norm, "bias")
    if weight is None or bias is None or not usable(x, weight, bias) or any(type(t) not in _PLAIN for t in (x, weight, bias)):
        return None
    return channel_norm(x, weight, bias, norm.eps, nhwc=False, pool=True).flatten(1)


def mlp_fn(x, mlp, twice=True):
    """A block's `mlp` (fc1, exact GELU, fc2) on x (B, H, W, C) where autograd records it, products, GELU and bias sums as
    kernels of this library; None where that does not apply (see block_mlp).  Second derivatives are PyTorch's; with
    `twice` False they are refused (for a caller whose upstream gradient comes without a history, so that an answer
    would lack what goes through it)."""
    if torch.compiler.is_compiling() or torch.is_autocast_enabled() or not torch.is_grad_enabled():
        return None
    ext = _ext.get()
    if ext is None:
        return None
    fc1, act, fc2 = mlp.fc1, mlp.act, mlp.fc2
    if (type(fc1) is not torch.nn.Linear or type(fc2) is not torch.nn.Linear or type(act) is not torch.nn.GELU
            or act.approximate != "none" or _watched(mlp, fc1, act, fc2) or _watched_backward(mlp, fc1, act, fc2)):
        return None
    args = (_param(fc1), _param(fc1, "bias"), _param(fc2), _param(fc2, "bias"))
    for t in (x, *args):
        if t is None or type(t) not in _PLAIN:
            return None
    return ext.mlp(x, *args, twice)


def _native(name, *args):
    """The function of the C++ binding: None where it is not built, does not take the arguments, or they are of a subclass."""
    ext = _ext.get()
    if ext is None:
        return None
    for t in args:
        if isinstance(t, torch.Tensor) and type(t) not in _PLAIN:
            return None
    return getattr(ext, name)(*args)


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def channel_norm(x, weight, bias, eps, nhwc, pool=False):
    """LayerNorm over the channels of x (B, C, H, W); returns (B, H, W, C) if `nhwc` else (B, C, H, W).  Not recorded.
    With `pool` (and without `nhwc`), of its mean over the pixels, (B, C, 1, 1)."""
    if pool:
        out = _native("pool_norm", x, weight, bias, eps)
        if out is not None:
            return out[:, :, None, None]
        x = x.mean(dim=(2, 3), keepdim=True)
    out = _native("channel_norm", x, weight, bias, eps, nhwc) if not records(x, weight, bias) else None
    if out is not None:
        return out
    lib = _lib.load()
    B, C, H, W = x.shape
    with torch.cuda.device(x.device):
        out = torch.empty((B, H, W, C) if nhwc else (B, C, H, W), dtype=x.dtype, device=x.device)
        rc = lib.wtconv_channel_norm(x.data_ptr(), out.data_ptr(), weight.data_ptr(), bias.data_ptr(), B, C, H * W,
                                     float(eps), _DT[x.dtype], _DT[weight.dtype], int(bool(nhwc)), _stream())
    if rc:
        _lib.check(rc, "wtconv_channel_norm")
    return out


def block_residual(y, shortcut, gamma):
    """shortcut (B, C, H, W) + gamma[c] * y, with y (B, H, W, C); gamma may be None.  Returns (B, C, H, W).  Not recorded."""
    out = _native("block_residual", y, shortcut, gamma) if not records(y, shortcut, gamma) else None
    if out is not None:
        return out
    lib = _lib.load()
    B, C, H, W = shortcut.shape
    if tuple(y.shape) != (B, H, W, C) or y.dtype != shortcut.dtype or not y.is_contiguous():
        raise ValueError(f"block_residual: y {tuple(y.shape)} {y.dtype} does not match shortcut {tuple(shortcut.shape)}")
    with torch.cuda.device(shortcut.device):
        out = torch.empty_like(shortcut)
        rc = lib.wtconv_block_residual(y.data_ptr(), shortcut.data_ptr(), gamma.data_ptr() if gamma is not None else None,
                                       out.data_ptr(), B, C, H * W, _DT[shortcut.dtype],
                                       _DT[gamma.dtype] if gamma is not None else _lib.F32, _stream())
    if rc:
        _lib.check(rc, "wtconv_block_residual")
    return out


def _workspace(x, B, C, HW):
    lib = _lib.load()
    n = lib.wtconv_block_workspace_bytes(B, C, HW, _DT[x.dtype])
    if n == 0:
        raise RuntimeError(f"block backward: no tile plan for C={C}, HW={HW}")
    return torch.empty(n, dtype=torch.uint8, device=x.device), n


def channel_norm_backward(x, dy, weight, eps, nhwc):
    """Gradients of channel_norm: dx (B, C, H, W) in x.dtype, dweight and dbias (C) in float32."""
    lib = _lib.load()
    B, C, H, W = x.shape
    with torch.cuda.device(x.device):
        dx = torch.empty_like(x)
        dwb = torch.empty(2, C, dtype=torch.float32, device=x.device)
        ws, n = _workspace(x, B, C, H * W)
        rc = lib.wtconv_channel_norm_backward(x.data_ptr(), dy.data_ptr(), weight.data_ptr(), dx.data_ptr(),
                                              dwb[0].data_ptr(), dwb[1].data_ptr(), B, C, H * W, float(eps),
                                              _DT[x.dtype], _DT[weight.dtype], int(bool(nhwc)), ws.data_ptr(), n, _stream())
    if rc:
        _lib.check(rc, "wtconv_channel_norm_backward")
    return dx, dwb[0], dwb[1]


def block_residual_backward(dout, y, gamma):
    """Gradients of block_residual with a layer scale: dy (B, H, W, C) in dout.dtype, dgamma (C) in float32."""
    lib = _lib.load()
    B, C, H, W = dout.shape
    with torch.cuda.device(dout.device):
        dy = torch.empty_like(y)
        dg = torch.empty(C, dtype=torch.float32, device=dout.device)
        ws, n = _workspace(dout, B, C, H * W)
        rc = lib.wtconv_block_residual_backward(dout.data_ptr(), y.data_ptr(), gamma.data_ptr(), dy.data_ptr(),
                                                dg.data_ptr(), B, C, H * W, _DT[dout.dtype], _DT[gamma.dtype],
                                                ws.data_ptr(), n, _stream())
    if rc:
        _lib.check(rc, "wtconv_block_residual_backward")
    return dy, dg


class _ChannelNormFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, bias, eps, nhwc):
        ctx.eps, ctx.nhwc = eps, nhwc
        ctx.save_for_backward(x, weight)
        return channel_norm(x, weight, bias, eps, nhwc)

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, dy):
        x, weight = ctx.saved_tensors
        if dy.dtype != x.dtype:
            dy = dy.to(x.dtype)
        dx, dw, db = channel_norm_backward(x, dy.contiguous(), weight, ctx.eps, ctx.nhwc)
        return dx, dw.to(weight.dtype), db.to(weight.dtype), None, None


class _BlockResidualFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, y, shortcut, gamma):
        ctx.save_for_backward(y, gamma)
        return block_residual(y, shortcut, gamma)

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, dout):
        y, gamma = ctx.saved_tensors
        if dout.dtype != y.dtype:
            dout = dout.to(y.dtype)
        dout = dout.contiguous()
        dy, dg = block_residual_backward(dout, y, gamma)
        return dy, dout, dg.to(gamma.dtype)


def channel_norm_fn(x, weight, bias, eps, nhwc):
    """channel_norm that autograd can differentiate (gradients of x, weight and bias from the backward kernel)."""
    out = _native("channel_norm", x, weight, bias, eps, nhwc)
    return out if out is not None else _ChannelNormFn.apply(x, weight, bias, eps, nhwc)


def block_residual_fn(y, shortcut, gamma):
    """block_residual (with a layer scale) that autograd can differentiate (gradients of y, shortcut and gamma)."""
    out = _native("block_residual", y, shortcut, gamma)
    return out if out is not None else _BlockResidualFn.apply(y, shortcut, gamma)
