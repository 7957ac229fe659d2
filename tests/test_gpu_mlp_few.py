"""The one-image kernels of a block's MLP (few pixels, two launches) against float64 on the same bfloat16 values."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,hidden", [
    ((1, 96, 4, 8), 384), ((1, 96, 3, 11), 64), ((3, 96, 29, 38), 384),      # a tile; a tile and one; nearly the last number taken
    ((1, 128, 7, 7), 512), ((2, 192, 28, 28), 768), ((1, 256, 31, 40), 1024),
    ((1, 384, 14, 14), 1536), ((17, 384, 7, 7), 192), ((1, 384, 8, 8), 4096),
    ((1, 384, 17, 49), 2496), ((4, 192, 8, 16), 4096), ((2, 256, 23, 25), 1792),      # up to the most pixels times hidden units
    ((1, 512, 14, 14), 2048), ((1, 768, 7, 7), 3072), ((8, 768, 4, 13), 64), ((1, 1024, 7, 7), 4096), ((6, 1024, 4, 13), 1024),
])
@pytest.mark.parametrize("layer_scale", [True, False])
def test_few_pixels_against_fp64(hip_device, shape, hidden, layer_scale):
    from wtconv_amd import _ext
    B, C, H, W = shape
    gen = torch.Generator(device=hip_device).manual_seed(C + H)
    r = lambda *s, k=1.0: (torch.randn(*s, generator=gen, device=hip_device) * k).bfloat16()
    x, sc = r(B, C, H, W), r(B, C, H, W)
    x[0, :, 0, 0] *= 30                                  # large activations: GELU's far ends
    nw, nb, w1, b1 = 1 + r(C, k=.2), r(C, k=.2), r(hidden, C, k=C ** -.5), r(hidden, k=3.0)
    w2, b2, gm = r(C, hidden, k=hidden ** -.5), r(C, k=.3), r(C) if layer_scale else None
    with torch.no_grad():
        got = _ext.get().block_mlp(x, sc, nw, nb, 1e-6, w1, b1, w2, b2, gm)
    assert got is not None and got.shape == x.shape and got.dtype == torch.bfloat16
    d = lambda t: t.double()
    y = F.layer_norm(d(x).permute(0, 2, 3, 1), (C,), d(nw), d(nb), 1e-6)
    y = F.linear(F.gelu(F.linear(y, d(w1), d(b1))), d(w2), d(b2))
    want = d(sc) + (y if gm is None else y * d(gm)).permute(0, 3, 1, 2)
    # the normalised values, the hidden ones and the result are rounded to bfloat16 (2^-9 relative each)
    rel = ((d(got) - want).norm() / want.norm()).item()
    assert rel < 4e-3, rel
    rms = want.pow(2).mean().sqrt()
    assert ((d(got) - want).abs() / torch.maximum(want.abs(), rms)).max().item() < 6e-2


def test_nans_keep_to_their_pixels_and_large_maps_to_the_separate_passes(hip_device):
    from wtconv_amd import _ext
    r = lambda *s: torch.randn(*s, device=hip_device).bfloat16()
    C = 768
    x, sc = r(2, C, 5, 5), r(2, C, 5, 5)
    args = (1 + r(C), r(C), 1e-6, r(4 * C, C), r(4 * C), r(C, 4 * C), r(C), r(C))
    with torch.no_grad():
        clean = _ext.get().block_mlp(x, sc, *args)
        x[1, 5, 3, 2] = float("nan")
        got = _ext.get().block_mlp(x, sc, *args)
        assert torch.isnan(got[1, :, 3, 2]).all()
        got[1, :, 3, 2] = clean[1, :, 3, 2]
        assert torch.equal(got, clean)
        assert _ext.get().block_mlp(r(17, C, 5, 5), r(17, C, 5, 5), *args) is None
        assert _ext.get().block_mlp(x[:1], sc[:1], *args) is None
