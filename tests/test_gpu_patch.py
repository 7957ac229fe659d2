"""GPU parity of the stem and downsample kernels (wtconv_patch_conv) against float64 on the same bfloat16 values, and of the
model that calls them against its separate passes."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _check(got, want):
    # one rounding of the normalised values (or none) and one of the result to bfloat16: 2^-9 relative each
    rel = ((got.double() - want).norm() / want.norm()).item()
    assert rel < 4e-3, rel
    rms = want.pow(2).mean().sqrt()
    assert ((got.double() - want).abs() / torch.maximum(want.abs(), rms)).max().item() < 4e-2


@pytest.mark.parametrize("shape,cout", [
    ((1, 96, 2, 2), 192),          # one output pixel
    ((1, 96, 14, 10), 32),         # 35 pixels: a remainder, images of odd size, the narrowest output
    ((3, 96, 56, 56), 192), ((4, 96, 56, 56), 192),      # the first split still, the second
    ((23, 96, 56, 54), 192),       # the third, with part of a tile
    ((66, 96, 6, 10), 224),        # many pixels, but not whole groups of output channels
    ((2, 128, 18, 14), 256), ((20, 128, 28, 28), 256), ((90, 128, 28, 28), 256),
    ((1, 192, 28, 28), 384), ((9, 192, 28, 26), 384), ((47, 192, 28, 26), 384),
    ((1, 256, 28, 28), 512), ((8, 256, 28, 28), 512), ((47, 256, 28, 28), 512),
    ((1, 384, 14, 14), 768), ((13, 384, 14, 14), 768), ((171, 384, 14, 14), 768), ((170, 384, 14, 14), 64),
    ((1, 512, 14, 14), 1024), ((13, 512, 14, 14), 1024), ((170, 512, 14, 14), 1024),
])
def test_downsample_against_fp64(hip_device, shape, cout):
    from wtconv_amd import _ext
    B, C, H, W = shape
    gen = torch.Generator(device=hip_device).manual_seed(C + B)
    r = lambda *s, k=1.0: (torch.randn(*s, generator=gen, device=hip_device) * k).bfloat16()
    x = r(B, C, H, W) + 3 * r(B, 1, H, W)                 # means away from zero
    cw, cb, nw, nb = r(cout, C, 2, 2, k=(4 * C) ** -.5), r(cout, k=.3), 1 + r(C, k=.2), r(C, k=.2)
    with torch.no_grad():
        got = _ext.get().patch_conv(x, cw, cb, nw, nb, 1e-6, False)
    assert got is not None and got.shape == (B, cout, H // 2, W // 2) and got.dtype == torch.bfloat16
    y = F.layer_norm(x.double().permute(0, 2, 3, 1), (C,), nw.double(), nb.double(), 1e-6)
    # the patches as rows, so that the product is a plain one
    y = y.reshape(B, H // 2, 2, W // 2, 2, C).permute(0, 1, 3, 5, 2, 4).reshape(-1, 4 * C)
    want = (y @ cw.double().reshape(cout, -1).t() + cb.double()).reshape(B, H // 2, W // 2, cout).permute(0, 3, 1, 2)
    _check(got, want)


@pytest.mark.parametrize("shape,cout", [
    ((1, 3, 4, 16), 96),           # four output pixels
    ((2, 3, 20, 48), 96),          # 120 pixels: a remainder
    ((1, 3, 224, 224), 96), ((64, 3, 160, 192), 96),      # one group of pixels a wave; many
    ((2, 3, 64, 80), 128), ((5, 4, 32, 32), 96), ((5, 1, 32, 32), 128), ((3, 2, 16, 16), 96),
])
def test_stem_against_fp64(hip_device, shape, cout):
    from wtconv_amd import _ext
    B, C, H, W = shape
    gen = torch.Generator(device=hip_device).manual_seed(C + B)
    r = lambda *s, k=1.0: (torch.randn(*s, generator=gen, device=hip_device) * k).bfloat16()
    x = r(B, C, H, W) + 2
    cw, cb, nw, nb = r(cout, C, 4, 4, k=.2), r(cout, k=.3), 1 + r(cout, k=.2), r(cout, k=.2)
    with torch.no_grad():
        got = _ext.get().patch_conv(x, cw, cb, nw, nb, 1e-6, True)
    assert got is not None and got.shape == (B, cout, H // 4, W // 4) and got.dtype == torch.bfloat16
    y = x.double().reshape(B, C, H // 4, 4, W // 4, 4).permute(0, 2, 4, 1, 3, 5).reshape(-1, 16 * C)
    y = (y @ cw.double().reshape(cout, -1).t() + cb.double()).reshape(B, H // 4, W // 4, cout)
    want = F.layer_norm(y, (cout,), nw.double(), nb.double(), 1e-6).permute(0, 3, 1, 2)
    _check(got, want)


def test_calls_without_a_kernel_are_left_alone(hip_device):
    """Sizes, strides, types and alignments that the kernels do not take, recording and tangents: None, and the model's own
    modules run."""
    from wtconv_amd import _ext
    fn = _ext.get().patch_conv
    r = lambda *s: torch.randn(*s, device=hip_device).bfloat16()
    cw, cb, nw, nb = r(192, 96, 2, 2), r(192), r(96), r(96)
    x = r(2, 96, 8, 8)
    with torch.no_grad():
        assert fn(x, cw, cb, nw, nb, 1e-6, False) is not None
        assert fn(r(2, 96, 8, 7), cw, cb, nw, nb, 1e-6, False) is None
        assert fn(r(2, 96, 7, 8), cw, cb, nw, nb, 1e-6, False) is None
        assert fn(r(2, 96, 8, 16)[..., ::2], cw, cb, nw, nb, 1e-6, False) is None
        assert fn(r(2 * 96 * 64 + 1)[1:].view(2, 96, 8, 8), cw, cb, nw, nb, 1e-6, False) is None
        assert fn(x.float(), cw, cb, nw, nb, 1e-6, False) is None
        assert fn(x, cw.float(), cb, nw, nb, 1e-6, False) is None
        assert fn(x, cw[:40], cb[:40], nw, nb, 1e-6, False) is None
        assert fn(r(0, 96, 8, 8), cw, cb, nw, nb, 1e-6, False) is None
        assert fn(r(2, 64, 8, 8), r(192, 64, 2, 2), cb, r(64), r(64), 1e-6, False) is None
        sw, sb = r(96, 3, 4, 4), r(96)
        assert fn(r(1, 3, 8, 32), sw, sb, nw, nb, 1e-6, True) is not None
        assert fn(r(1, 3, 8, 24), sw, sb, nw, nb, 1e-6, True) is None
        assert fn(r(1, 5, 8, 32), r(96, 5, 4, 4), sb, nw, nb, 1e-6, True) is None
        with torch.autograd.forward_ad.dual_level():
            dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
            assert fn(dual, cw, cb, nw, nb, 1e-6, False) is None
    assert fn(x.requires_grad_(), cw, cb, nw, nb, 1e-6, False) is None


def test_infinities_and_nans_keep_to_their_patches(hip_device):
    from wtconv_amd import _ext
    fn = _ext.get().patch_conv
    g = torch.Generator(device=hip_device).manual_seed(0)
    r = lambda *s: torch.randn(*s, generator=g, device=hip_device).bfloat16()
    for stem, x, args in ((False, r(2, 96, 8, 8), (r(192, 96, 2, 2), r(192), r(96), r(96))),
                          (True, r(2, 3, 16, 16), (r(96, 3, 4, 4), r(96), r(96), r(96)))):
        with torch.no_grad():
            clean = fn(x, *args, 1e-6, stem)
            for bad in (float("nan"), float("inf")):
                y = x.clone()
                y[1, 1, 5, 6] = bad
                got = fn(y, *args, 1e-6, stem)
                at = (1, slice(None), 1, 1) if stem else (1, slice(None), 2, 3)
                assert torch.isnan(got[at]).all()
                got[at] = clean[at]
                assert torch.equal(got, clean)


def test_model_with_and_without_the_kernels(hip_device):
    """A hook makes the model take the separate passes; the results agree, also replayed from a captured graph."""
    from wtconvnext.wtconvnext import WTConvNeXt
    torch.manual_seed(0)
    m = WTConvNeXt(depths=(1, 1, 1, 1), dims=(96, 192, 384, 768), wt_levels=(2, 2, 2, 1), num_classes=10,
                   ls_init_value=0.3).to(hip_device).bfloat16().eval()
    x = torch.randn(3, 3, 64, 64, device=hip_device).bfloat16()
    with torch.no_grad():
        fused = m(x)
        seen = []
        handles = [mod.register_forward_hook(lambda m, i, o: seen.append(m)) for mod in m.modules()
                   if isinstance(mod, torch.nn.Conv2d) and mod.groups == 1]
        apart = m(x)
        for h in handles:
            h.remove()
        assert len(seen) == 4
        assert (fused.float() - apart.float()).norm() < 2e-2 * apart.float().norm()
        static = x.clone()
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            m.forward_features(static)
        torch.cuda.current_stream().wait_stream(s)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = m.forward_features(static)
        for seed in range(3):
            static.copy_(torch.randn(x.shape, generator=torch.Generator().manual_seed(seed)).bfloat16())
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, m.forward_features(static))
