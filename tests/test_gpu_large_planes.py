"""Planes beyond LDS, whose steps take rows of pixels over the lanes of a wave: widths around a wave's 64 lanes of four pixels
(one tile, two with a gap between the units, more with lanes of their own on either side), rows that are no whole lanes, planes
narrower than a lane, the fewest rows, and every kernel size and element type."""
import pytest
import torch

from parity_util import assert_bf16, assert_fp32, compare_all, copy_to_hip_module, hip_run, oracle_run, randomize_scales, seeded_case

pytestmark = pytest.mark.gpu


def _modules():
    from wtconv import WTConv2d
    return WTConv2d


def _assert_fp16(got, want, name):
    rms = want.double().pow(2).mean().sqrt().item()
    torch.testing.assert_close(got.double(), want.double(), rtol=2e-3, atol=2e-3 * max(rms, 1e-12), msg=lambda m: f"{name}: {m}")


def _assert_sums(got, want, name):
    # sums over all pixels of all images: float32 resolves their largest entry, not each of them
    torch.testing.assert_close(got.double(), want.double(), rtol=1e-5, atol=max(1e-4, 2e-6 * want.abs().max().item()),
                               msg=lambda m: f"{name}: {m}")


@pytest.mark.parametrize("shape,K,L", [
    ((3, 2, 120, 160), 5, 2),      # two tiles of 20 lanes, three units a wave
    ((2, 2, 101, 201), 5, 3),      # one tile more than half a wave wide, rows of a pixel over whole lanes
    ((1, 2, 130, 252), 5, 1),      # one tile of 63 lanes
    ((1, 2, 97, 258), 5, 2),       # two tiles a lane wider than a wave holds
    ((1, 1, 60, 1030), 5, 1),      # many tiles
    ((2, 2, 140, 143), 3, 2),      # K = 3, odd both ways
    ((2, 2, 150, 122), 7, 2),      # K = 7: windows two lanes wide
    ((1, 1, 90, 515), 7, 1),
    ((1, 2, 129, 160), 1, 1),      # K = 1: no window
    ((1, 2, 9000, 3), 5, 2),       # narrower than a lane
    ((1, 1, 20000, 1), 3, 1),
    ((1, 1, 3, 9001), 5, 1),       # fewer rows than a window
    ((70, 1, 128, 129), 5, 1),     # more units than a launch takes at once
])
def test_shapes_fp32(hip_device, shape, K, L):
    ref, x, g = seeded_case("2d", shape[1], K, L, shape)
    randomize_scales(ref)
    got = hip_run(copy_to_hip_module(ref, _modules(), "2d", K, L), x, g, hip_device)
    want = oracle_run(ref, x, g)
    assert_fp32(got[0], want[0], "out")
    assert_fp32(got[1], want[1], "grad_x")
    for n, w in want[2].items():
        if n in got[2]:
            _assert_sums(got[2][n], w, n)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape,K,L", [((2, 2, 131, 161), 5, 2), ((1, 2, 120, 254), 7, 1), ((2, 2, 150, 150), 3, 1)])
def test_shapes_16_bit(hip_device, dtype, shape, K, L):
    ref, x, g = seeded_case("2d", shape[1], K, L, shape)
    randomize_scales(ref)
    x, g = x.to(dtype).float(), g.to(dtype).float()
    got = hip_run(copy_to_hip_module(ref, _modules(), "2d", K, L), x, g, hip_device, dtype=dtype)
    want = oracle_run(ref, x, g)
    check = _assert_fp16 if dtype == torch.float16 else assert_bf16
    check(got[0], want[0], "out")
    check(got[1], want[1], "grad_x")
    for n, w in want[2].items():
        if n in got[2]:
            _assert_sums(got[2][n], w, n)


def test_infinities_stay_within_their_windows(hip_device):
    """A window that holds an infinity gives an infinity or NaN, every other one its finite result."""
    ref, x, g = seeded_case("2d", 2, 5, 1, (1, 2, 140, 160))
    x[0, 0, 70, 79] = float("inf")
    mod = copy_to_hip_module(ref, _modules(), "2d", 5, 1).to(hip_device)
    with torch.no_grad():
        got = mod(x.to(hip_device)).cpu()
        want = ref(x)
    # (the library convolution of the oracle spreads it no further than the windows' reach either)
    assert torch.equal(torch.isfinite(got), torch.isfinite(want))
    fin = torch.isfinite(want)
    assert_fp32(got[fin], want[fin], "finite outputs")


@pytest.mark.parametrize("row,col", [(70, 79), (70, 80), (70, 0), (139, 159), (0, 3)])
def test_infinities_stay_within_their_sums(hip_device, row, col):
    """An infinity of x makes those sums of the base filter's gradient infinite whose windows hold it, and no other: a lane
    beside its unit's own ones, or below the plane, adds nothing (an infinity times no gradient is not a number)."""
    H, W, K = 140, 160, 5
    ref, x, g = seeded_case("2d", 2, K, 1, (1, 2, H, W))
    x[0, 0, row, col] = float("inf")
    got = hip_run(copy_to_hip_module(ref, _modules(), "2d", K, 1), x, g, hip_device)[2]["base_conv.weight"].reshape(2, K, K)
    r = K // 2
    want = torch.tensor([[0 <= row - kh + r < H and 0 <= col - kw + r < W for kw in range(K)] for kh in range(K)])
    assert torch.equal(torch.isinf(got[0]).cpu(), want)
    assert torch.equal(torch.isfinite(got[0]).cpu(), ~want)
    assert torch.isfinite(got[1]).all()
