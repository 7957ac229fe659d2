"""Parameter gradients and results of the vector kernels at the shapes where their plans change: planes of which LDS holds one
pair of pyramids or two, K = 7 with one and with more planes an iteration, rows whose strips divide no thread count."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,K,L,dtype", [
    ((16, 24, 45, 37), 7, 2, torch.float16),      # three planes an iteration, one workgroup a CU
    ((5, 7, 40, 39), 7, 4, torch.float32),        # fewer workgroups than compute units: one plane
    ((33, 16, 11, 13), 7, 2, torch.float32),      # one iteration a workgroup, the last workgroup's not full
    ((40, 3, 6, 7), 7, 2, torch.float32),         # one iteration of as many planes as there are places
    ((53, 86, 20, 22), 7, 4, torch.float32),      # two workgroups a channel with several iterations each, the last one short
    ((37, 270, 8, 9), 7, 2, torch.float16),       # more channels than compute units
    ((9, 12, 30, 25), 7, 1, torch.bfloat16),      # one level: two workgroups a CU
    ((7, 6, 58, 66), 5, 3, torch.float32),        # one pair of pyramids takes more than half of the LDS
    ((3, 5, 75, 60), 5, 2, torch.float16),
    ((2, 4, 100, 85), 5, 1, torch.float32),
    ((4, 10, 33, 41), 5, 3, torch.float32),       # rows a little above a power of two
    ((3, 10, 35, 33), 5, 4, torch.float16),
    ((16, 9, 17, 19), 5, 1, torch.float16),       # rows of 5 strips or 10 over 64 threads: the last pass is not full
    ((6, 20, 12, 10), 7, 1, torch.float32),       # two strips a row, four planes a wave
    ((40, 9, 45, 50), 3, 2, torch.float32),       # K = 3: strips of two, odd rows a pass
    ((300, 1, 87, 66), 7, 1, torch.float32),      # 512 threads a plane, rows of 17 strips
    ((2, 130, 5, 77), 7, 2, torch.float32),       # three rows of 39 coefficients
    ((1, 7, 33, 36), 7, 1, torch.float32),        # few planes: 512 threads each, strips of one
    ((1, 5, 66, 58), 5, 3, torch.float16),        # and 1024
    ((4, 3, 99, 79), 3, 2, torch.float32),        # the same, K = 3
    ((300, 5, 6, 5), 7, 1, torch.float32),        # four planes a wave, strips of one
    ((209, 4, 13, 16), 7, 3, torch.float32),      # a wave a plane
    ((1, 2, 3, 130), 5, 1, torch.float32),        # two rows of 65 coefficients
    ((3, 4, 13, 255), 5, 2, torch.float32),       # parameter gradients: one row of 64 strips a wave
    ((4, 6, 30, 9), 3, 2, torch.float32),         # 21 rows of three strips
    ((5, 4, 21, 82), 7, 1, torch.float16),        # three rows of 21, one lane without
])
def test_layer_against_fp64(hip_device, shape, K, L, dtype):
    import wtconv
    from oracle import wtconv_ref as R
    torch.manual_seed(K + L)
    C = shape[1]
    ref = R.RefWTConv2d(C, C, K, wt_levels=L).double()
    mod = wtconv.WTConv2d(C, C, kernel_size=K, wt_levels=L).float()
    mod.load_state_dict({k: v.float() for k, v in ref.state_dict().items()})
    ref.load_state_dict({k: v.double() for k, v in mod.state_dict().items()})
    mod = mod.to(hip_device)
    x, g = torch.randn(shape).to(dtype), torch.randn(shape).to(dtype)
    out64, dx64, grads64 = R.layer_grads(ref, x.double(), g.double())
    xd = x.to(hip_device).requires_grad_()
    out = mod(xd)
    out.backward(g.to(hip_device))
    rel = lambda a, b: ((a.double().cpu() - b).norm() / b.norm()).item()
    # results are rounded to their type once; float sums of up to 1e5 products in float
    eps = {torch.float32: 2e-6, torch.float16: 4e-4, torch.bfloat16: 3e-3}[dtype]
    assert rel(out.detach(), out64) < eps and rel(xd.grad, dx64) < eps
    for n, p in mod.named_parameters():
        if p.grad is not None:
            assert rel(p.grad, grads64[n]) < 5e-6, n


@pytest.mark.parametrize("shape,K,L", [
    ((3, 5, 9, 33), 5, 2), ((2, 7, 10, 18), 5, 1), ((5, 3, 13, 43), 3, 3), ((4, 6, 12, 20), 5, 2),      # 1 to 7 columns past whole
    ((3, 4, 11, 29), 5, 3), ((2, 3, 7, 22), 5, 2), ((6, 5, 15, 15), 5, 3),                              # pairs of 4 x 4 blocks
    ((40, 3, 17, 17), 5, 4),      # eight tiles of level-1 blocks for four waves
    ((9, 2, 64, 40), 5, 5),       # as wide and deep as the kernel takes, five tiles
    ((37, 9, 4, 4), 1, 1), ((70, 4, 7, 7), 5, 2), ((1, 1, 5, 6), 3, 2),      # many planes a unit; one plane, the tensor's last
    ((26, 4, 14, 14), 5, 3),      # a compile-time plan, the last unit not full
    ((1, 5, 14, 14), 5, 3), ((5, 3, 14, 14), 5, 3), ((13, 4, 14, 14), 5, 2),      # and units of fewer planes than it has places for
    ((1, 3, 28, 28), 5, 4), ((3, 4, 28, 28), 5, 3), ((1, 9, 7, 7), 5, 2), ((17, 5, 7, 7), 5, 2), ((33, 2, 7, 7), 5, 2),
])
def test_matrix_core_layer_against_fp64(hip_device, shape, K, L):
    import wtconv
    from oracle import wtconv_ref as R
    torch.manual_seed(shape[3] + L)
    C = shape[1]
    mod = wtconv.WTConv2d(C, C, kernel_size=K, wt_levels=L).bfloat16()
    with torch.no_grad():
        for p in mod.parameters():
            if p.requires_grad:
                p.copy_(torch.randn(p.shape) * 0.4)
    ref = R.RefWTConv2d(C, C, K, wt_levels=L).double()
    ref.load_state_dict({k: v.double() for k, v in mod.state_dict().items()})
    mod = mod.to(hip_device)
    x, g = torch.randn(shape).bfloat16(), torch.randn(shape).bfloat16()
    out64, dx64, _ = R.layer_grads(ref, x.double(), g.double())
    xd = x.to(hip_device).requires_grad_()
    out = mod(xd)
    out.backward(g.to(hip_device))
    rel = lambda a, b: ((a.double().cpu() - b).norm() / b.norm()).item()
    # each product has a coefficient and a folded weight rounded to 8 bits (at most 2^-9 of them each), the result is once more
    assert rel(out.detach(), out64) < 3 * 2 ** -9 and rel(xd.grad, dx64) < 3 * 2 ** -9
