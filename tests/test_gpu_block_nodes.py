"""The C++ autograd nodes of a block's two passes against the Python functions that run where they do not apply: the same
bits, whatever needs a gradient, and the same refusals."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _results(fn, tensors, g, mask):
    leaves = [t.detach().clone().requires_grad_(bool(mask >> i & 1)) for i, t in enumerate(tensors)]
    out = fn(*leaves)
    out.backward(g)
    return [out.detach()] + [t.grad for t in leaves]


@pytest.mark.parametrize("dtype,pdtype", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.float32, torch.float32),
                                          (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("shape", [(3, 96, 14, 14), (2, 64, 7, 5), (5, 384, 1, 1)])
@pytest.mark.parametrize("strided", [False, True])
def test_nodes_match_the_python_functions(hip_device, dtype, pdtype, shape, strided):
    from wtconv_amd import _ext, block_ops as ops
    B, C, H, W = shape
    gen = torch.Generator().manual_seed(C + H)
    r = lambda *s, t=dtype: torch.randn(*s, generator=gen).to(device=hip_device, dtype=t)
    grad = lambda *s: r(*s, 2)[..., 0] if strided else r(*s)
    x, y, w, b = r(*shape), r(B, H, W, C), r(C, t=pdtype), r(C, t=pdtype)
    ext = _ext.get()
    for nhwc in (False, True):
        g = grad(B, H, W, C) if nhwc else grad(*shape)
        for mask in range(1, 8):
            got = _results(lambda *a: ext.channel_norm(*a, 1e-6, nhwc), (x, w, b), g, mask)
            want = _results(lambda *a: ops._ChannelNormFn.apply(*a, 1e-6, nhwc), (x, w, b), g, mask)
            assert all(p is None and q is None or torch.equal(p, q) and p.dtype == q.dtype for p, q in zip(got, want))
    g = grad(*shape)
    for mask in range(1, 8):
        got = _results(ext.block_residual, (y, x, w), g, mask)
        want = _results(ops._BlockResidualFn.apply, (y, x, w), g, mask)
        assert all(p is None and q is None or torch.equal(p, q) and p.dtype == q.dtype for p, q in zip(got, want))


def test_what_the_nodes_refuse(hip_device):
    from wtconv_amd import _ext, block_ops as ops
    ext = _ext.get()
    r = lambda *s: torch.randn(*s, device=hip_device)
    x, y, w, b = r(2, 8, 4, 4).requires_grad_(), r(2, 4, 4, 8), r(8), r(8)
    assert ext.channel_norm(x.transpose(2, 3), w, b, 1e-6, True) is None and ext.channel_norm(x, w.half(), b, 1e-6, True) is None
    assert ext.channel_norm(x, w[:4], b, 1e-6, True) is None and ext.channel_norm(x.cpu(), w, b, 1e-6, True) is None
    assert ext.block_residual(y, x, None) is None                       # recorded, and no layer scale
    assert ext.block_residual(y[:, :2], x, w) is None
    with torch.no_grad():
        assert ext.block_residual(y, x, None) is not None
    out = ops.channel_norm_fn(x, w, b, 1e-6, True)
    assert out.requires_grad
    gx, = torch.autograd.grad(out, x, y, create_graph=True)
    with pytest.raises(RuntimeError, match="not differentiable"):
        gx.sum().backward()
    out = ops.block_residual_fn(y.requires_grad_(), x, w)
    gy, = torch.autograd.grad(out, y, r(2, 8, 4, 4), create_graph=True)
    with pytest.raises(RuntimeError, match="not differentiable"):
        gy.sum().backward()
    with torch.autograd.forward_ad.dual_level(), pytest.raises(RuntimeError):      # no tangents, as before
        ops.channel_norm_fn(torch.autograd.forward_ad.make_dual(x.detach(), r(2, 8, 4, 4)), w.requires_grad_(), b, 1e-6, True)


def test_upstream_gradient_keeps_its_own_history(hip_device):
    from wtconv_amd import block_ops as ops
    r = lambda *s: torch.randn(*s, device=hip_device)
    y, x, w = r(2, 4, 4, 8), r(2, 8, 4, 4).requires_grad_(), r(8)
    g = r(2, 8, 4, 4).requires_grad_()
    gx, = torch.autograd.grad(ops.block_residual_fn(y, x, w), x, g, create_graph=True)
    assert torch.equal(gx, g) and g.is_leaf and g.grad_fn is None      # the shortcut's gradient is g's values, not g
    with pytest.raises(RuntimeError, match="not differentiable"):
        gx.sum().backward()


def _spread(t):
    return torch.stack([t, torch.full_like(t, float("nan"))], -1)[..., 0] if t.is_floating_point() else t


def _shifted(t):
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    flat[1:] = t.reshape(-1)
    return flat[1:].view(t.shape)


@pytest.mark.parametrize("back", [_spread, _shifted])
@pytest.mark.parametrize("which", ["layer", "norm", "mlp", "residual"])
def test_saved_tensors_may_come_back_otherwise(hip_device, which, back):
    """Hooks on saved tensors that give them back with other strides or at an odd address: the same bits.  Another type, size or
    device is refused before anything is launched."""
    from wtconv import WTConv2d
    from wtconv_amd import _ext
    ext = _ext.get()
    gen = torch.Generator().manual_seed(0)
    r = lambda *s: torch.randn(*s, generator=gen).bfloat16().to(hip_device)
    B, C, H, W = 2, 96, 14, 14
    x, y, g = r(B, C, H, W), r(B, H, W, C), r(B, C, H, W)
    conv = WTConv2d(C, C, kernel_size=5, wt_levels=2).to(hip_device).bfloat16()
    params = [p for p in conv.parameters() if p.requires_grad]
    fn, tensors, g = {
        "layer": (lambda a, *p: torch.func.functional_call(conv, dict(zip(names, p)), (a,)), (x, *params), g),
        "norm": (lambda *a: ext.channel_norm(*a, 1e-6, True), (x, r(C), r(C)), y),
        "mlp": (ext.mlp, (y, r(4 * C, C), r(4 * C), r(C, 4 * C), r(C)), r(B, H, W, C)),
        "residual": (ext.block_residual, (y, x, r(C)), g)}[which]
    names = [n for n, p in conv.named_parameters() if p.requires_grad]

    def grads(unpack):
        leaves = [t.detach().clone().requires_grad_() for t in tensors]
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
            out = fn(*leaves)
        return torch.autograd.grad(out, leaves, g)

    for a, b in zip(grads(lambda t: t), grads(back)):
        assert torch.equal(a, b)
    for other in (lambda t: t.float(), lambda t: t.cpu(), lambda t: t.reshape(-1)[:-1]):
        with pytest.raises(RuntimeError, match="came back"):
            grads(other)
