"""GPU parity of the MLP's training kernels (wtconv_mlp_forward, wtconv_mlp_backward) against float64 on the same bfloat16
values, and of the block that calls them against its separate passes."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _inputs(dev, M, C, hidden, seed=0):
    gen = torch.Generator(device=dev).manual_seed(seed + C + M)
    r = lambda *s, k=1.0: (torch.randn(*s, generator=gen, device=dev) * k).bfloat16()
    return r(M, C), r(M, C), r(hidden, C, k=C ** -.5), r(hidden), r(C, hidden, k=hidden ** -.5), r(C)


def _call(x, dy, *params):
    from wtconv_amd import _ext
    leaves = [t.detach().clone().requires_grad_() for t in (x, *params)]
    y = _ext.get().mlp(*leaves)
    assert y is not None and y.dtype == torch.bfloat16 and y.shape == x.shape
    y.backward(dy)
    return [y.detach()] + [t.grad for t in leaves]


def _rel(a, b):
    return ((a.double() - b).norm() / b.norm()).item()


@pytest.mark.parametrize("M,C,hidden", [
    (1, 384, 1536),            # one pixel
    (63, 96, 384), (65, 96, 384), (80001, 96, 384),      # 96 channels: steps of 32, tiles of 96; a pixel more than whole stages
    (130, 128, 512), (33000, 128, 512),
    (200, 192, 768), (50176, 192, 768),                  # tiles of 64, then of 192 outputs
    (700, 384, 1536), (12544, 384, 1536), (12500, 384, 128),
    (49, 768, 3072), (3000, 768, 3072), (513, 1152, 256),
])
def test_mlp_against_fp64(hip_device, M, C, hidden):
    args = _inputs(hip_device, M, C, hidden)
    got = _call(*args)
    x, dy, w1, b1, w2, b2 = [t.double() for t in args]
    h = x @ w1.t() + b1
    y = F.gelu(h) @ w2.t() + b2
    phi = 0.5 * (1 + torch.erf(h * 0.5 ** 0.5))
    dh = (dy @ w2) * (phi + h * torch.exp(-0.5 * h * h) * (2 * torch.pi) ** -0.5)
    want = [y, dh @ w1, dh.t() @ x, dh.sum(0), dy.t() @ F.gelu(h), dy.sum(0)]
    for name, a, b in zip(("y", "dx", "dw1", "db1", "dw2", "db2"), got, want):
        # operands of the second product and results are rounded to bfloat16 (2^-9 relative at most, each)
        assert _rel(a, b) < 5e-3, name


def test_a_frozen_part_is_not_computed(hip_device):
    """Every subset of what may need a gradient: the full pass's gradients to rounding, None elsewhere."""
    from wtconv_amd import _ext
    x, dy, *params = _inputs(hip_device, 300, 192, 768)
    full = _call(x, dy, *params)[1:]
    for mask in range(1, 32):
        leaves = [t.detach().clone().requires_grad_(bool(mask >> i & 1)) for i, t in enumerate((x, *params))]
        _ext.get().mlp(*leaves).backward(dy)
        for t, want in zip(leaves, full):
            # (fewer products share the chip in other numbers of shares, whose sums round differently)
            assert t.grad is None if not t.requires_grad else _rel(t.grad, want.double()) < 4e-3


def test_bad_values_stay_where_they_belong(hip_device):
    x, dy, *params = _inputs(hip_device, 130, 128, 512)
    y0, dx0, dw10, db10, dw20, db20 = _call(x, dy, *params)
    xn = x.clone()
    xn[129, 3] = float("nan")                        # the last pixel, alone in its stage but one
    y, dx, dw1, db1, dw2, db2 = _call(xn, dy, *params)
    assert torch.isnan(y[129]).all() and torch.equal(y[:129], y0[:129]) and torch.equal(dx[:129], dx0[:129])
    assert torch.isnan(dx[129]).all() and torch.isnan(dw1).all() and torch.equal(db2, db20)
    g = dy.clone()
    g[129, 5] = float("inf")
    y, dx, dw1, db1, dw2, db2 = _call(x, g, *params)
    keep = torch.arange(128, device=x.device) != 5
    assert torch.equal(dw2[keep], dw20[keep]) and torch.equal(db2[keep], db20[keep]) and torch.isinf(db2[5])
    assert not torch.isfinite(dw2[5]).any() and torch.equal(dx[:129], dx0[:129])
    big = params[1].clone()
    big[:] = 1e30                                    # far out GELU is the identity
    got = _call(x, dy, params[0], big, *params[2:])
    assert all(torch.isfinite(t).all() for t in got[1:])


def test_calls_without_kernels_are_left_alone(hip_device):
    from wtconv_amd import _ext
    fn = _ext.get().mlp
    x, dy, w1, b1, w2, b2 = _inputs(hip_device, 64, 96, 384)
    r = lambda *s: torch.randn(*s, device=hip_device).bfloat16()
    assert fn(x, w1, b1, w2, b2) is None                                  # nothing to record
    x.requires_grad_()
    assert fn(x, w1, b1, w2, b2) is not None
    with torch.no_grad():
        assert fn(x, w1, b1, w2, b2) is None
    assert fn(x.float(), w1, b1, w2, b2) is None and fn(x, w1.float(), b1, w2, b2) is None
    assert fn(x.t().contiguous().t(), w1, b1, w2, b2) is None
    assert fn(r(96 * 64 + 1)[1:].view(64, 96).requires_grad_(), w1, b1, w2, b2) is None
    assert fn(r(64, 64).requires_grad_(), r(256, 64), r(256), r(64, 256), r(64)) is None
    assert fn(x, r(96, 96), r(96), r(96, 96), b2) is None
    assert fn(r(0, 96).requires_grad_(), w1, b1, w2, b2) is None
    y = fn(x, w1, b1, w2, b2)
    gx, = torch.autograd.grad(y, x, dy, create_graph=True)
    with pytest.raises(RuntimeError, match="not differentiable"):
        gx.float().sum().backward()


def test_second_derivatives_of_a_block_without_layer_scale(hip_device):
    """Those that do not lead through the gradients of the layer or the norm, against the separate passes (an observer)."""
    from wtconvnext.wtconvnext import WTConvNeXtBlock
    torch.manual_seed(0)
    blk = WTConvNeXtBlock(96, wt_levels=2, ls_init_value=None).to(hip_device).bfloat16()
    x = torch.randn(2, 96, 14, 14, device=hip_device).bfloat16()
    leaves = [blk.mlp.fc1.weight, blk.mlp.fc1.bias, blk.mlp.fc2.weight]

    def second():
        first = torch.autograd.grad(blk(x).float().square().sum(), leaves, create_graph=True)
        return torch.autograd.grad(sum(t.float().square().sum() for t in first), leaves)

    got = second()
    handle = blk.mlp.fc1.register_forward_hook(lambda m, i, o: None)
    want = second()
    handle.remove()
    for a, b in zip(got, want):      # products of bfloat16 values in another order, four deep
        assert _rel(a, b.double()) < 2e-2
    blk.gamma = torch.nn.Parameter(torch.ones(96, device=hip_device).bfloat16())
    with pytest.raises(RuntimeError):
        second()


@pytest.mark.parametrize("C,side", [(96, 14), (384, 14), (768, 7)])
def test_block_step_with_and_without_the_kernels(hip_device, C, side):
    """Observers make the block take the separate passes: the same gradients within bfloat16 rounding, strided upstream
    gradients included; and a captured step replays to the bits of an eager one."""
    from wtconvnext.wtconvnext import WTConvNeXtBlock
    torch.manual_seed(0)
    blk = WTConvNeXtBlock(C, wt_levels=2, ls_init_value=0.5).to(hip_device).bfloat16().train()
    x = torch.randn(4, C, side, side, device=hip_device).bfloat16().requires_grad_()
    g = torch.randn(4, C, side, 2 * side, device=hip_device).bfloat16()[..., ::2]
    params = list(blk.parameters())
    params = [p for p in params if p.requires_grad]

    def step():
        for t in (x, *params):
            t.grad = None
        out = blk(x)
        out.backward(g)
        return [out.detach().clone()] + [t.grad.clone() for t in (x, *params)]

    fused = step()
    seen = []
    for handle in (lambda: blk.mlp.fc1.register_forward_hook(lambda m, i, o: seen.append(1)),
                   lambda: blk.mlp.fc2.register_full_backward_hook(lambda m, i, o: seen.append(2)),
                   lambda: blk.mlp.act.register_full_backward_pre_hook(lambda m, o: seen.append(3))):
        h = handle()
        apart = step()
        h.remove()
        for a, b in zip(fused, apart):
            assert _rel(a, b.double()) < 2e-2
    assert seen == [1, 2, 3]
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for seed in range(3):
        with torch.no_grad():
            x.copy_(torch.randn(x.shape, generator=torch.Generator().manual_seed(seed)).bfloat16())
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in out]
        for a, b in zip(got, step()):
            assert torch.equal(a, b)
