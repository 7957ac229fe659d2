"""Parameter gradients written in the parameters' 16-bit type (the C++ node) against the same kernels' float results rounded
by PyTorch (the Python function): the same bits, for every kernel family that sums them."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,shape,K,L,dtype", [
    (2, (3, 24, 14, 14), 5, 3, torch.float32),       # plane-resident vector kernels
    (2, (3, 24, 14, 14), 5, 3, torch.bfloat16),      # matrix cores
    (2, (2, 8, 45, 37), 7, 2, torch.float16),        # kernel size 7
    (2, (1, 3, 200, 180), 3, 2, torch.bfloat16),     # one level at a time, a finishing launch
    (1, (2, 16, 1000), 5, 3, torch.float32),         # the whole backward pass in one kernel
    (1, (2, 16, 2011), 7, 5, torch.bfloat16),        # gradients in a kernel of their own
    (1, (2, 16, 100), 1, 2, torch.float16),          # kernel size 1
])
@pytest.mark.parametrize("pdtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("need_x", [True, False])
def test_typed_gradients_are_the_rounded_float_ones(hip_device, dims, shape, K, L, dtype, pdtype, need_x):
    from wtconv_amd import _ext, functional as Fn
    gen = torch.Generator().manual_seed(K + L)
    r = lambda *s: torch.randn(*s, generator=gen).to(device=hip_device, dtype=pdtype).requires_grad_()
    C, S, ones = shape[1], 2 ** dims, (1,) * dims
    params = [r(C, 1, *(K,) * dims), r(C), r(1, C, *ones)] + [r(S * C, 1, *(K,) * dims) for _ in range(L)] + [r(1, S * C, *ones) for _ in range(L)]
    x = torch.randn(shape, generator=gen).to(device=hip_device, dtype=dtype).requires_grad_(need_x)
    g = torch.randn(shape, generator=gen).to(device=hip_device, dtype=dtype)
    results = []
    for call in (lambda: _ext.get().layer(x, *params[:3], params[3:3 + L], params[3 + L:], dims, K, L),
                 lambda: Fn._WTConvFn.apply(x, *params[:3], dims, K, L, *params[3:])):
        for t in (x, *params):
            t.grad = None
        call().backward(g)
        results.append([t.grad for t in params])
    for a, b in zip(*results):
        assert a.dtype == b.dtype == pdtype and torch.equal(a, b)
