"""GPU parity of the block-epilogue kernels (wtconv_channel_norm, wtconv_block_residual) against
torch's own LayerNorm / permute / mul / add in float64 on the CPU, through the C ABI.  Floating-point
kernels: the reference here is the plain torch formulation of wtconvnext.py:132-140 of the reference."""
import pytest
import torch
import torch.nn.functional as F

import parity_util as U

pytestmark = pytest.mark.gpu

SHAPES = [(2, 96, 56, 56), (3, 192, 28, 28), (2, 384, 14, 14), (3, 768, 7, 7), (1, 6, 5, 3), (2, 2, 1, 1),
          (1, 1538, 3, 3), (2, 10, 9, 13)]


def _ref_norm(x, w, b, eps, nhwc):
    y = F.layer_norm(x.double().permute(0, 2, 3, 1), (x.shape[1],), w.double(), b.double(), eps)
    return y if nhwc else y.permute(0, 3, 1, 2)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype,pdtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16),
                                          (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("nhwc", [True, False])
def test_channel_norm(hip_device, shape, dtype, pdtype, nhwc):
    from wtconv_amd import block_ops
    B, C, H, W = shape
    gen = torch.Generator().manual_seed(B * 1000 + C)
    x = (torch.randn(shape, generator=gen) * 2 + 0.5).to(dtype)
    w = (torch.randn(C, generator=gen) * 0.5 + 1).to(pdtype)
    b = torch.randn(C, generator=gen).to(pdtype)
    assert block_ops.usable(x.to(hip_device), w.to(hip_device), b.to(hip_device))
    got = block_ops.channel_norm(x.to(hip_device), w.to(hip_device), b.to(hip_device), 1e-6, nhwc).float().cpu()
    want = _ref_norm(x.float(), w.float(), b.float(), 1e-6, nhwc)
    assert got.shape == want.shape
    (U.assert_fp32 if dtype == torch.float32 else U.assert_bf16)(got, want.float(), f"channel_norm {shape} nhwc={nhwc}")


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype,pdtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("with_gamma", [True, False])
def test_block_residual(hip_device, shape, dtype, pdtype, with_gamma):
    from wtconv_amd import block_ops
    B, C, H, W = shape
    gen = torch.Generator().manual_seed(B * 77 + C)
    y = torch.randn(B, H, W, C, generator=gen).to(dtype)
    sc = torch.randn(shape, generator=gen).to(dtype)
    gamma = (torch.randn(C, generator=gen) * 0.7).to(pdtype) if with_gamma else None
    got = block_ops.block_residual(y.to(hip_device), sc.to(hip_device),
                                   gamma.to(hip_device) if with_gamma else None).float().cpu()
    want = y.double().permute(0, 3, 1, 2)
    if with_gamma:
        want = want * gamma.double().reshape(1, -1, 1, 1)
    want = (want + sc.double()).float()
    (U.assert_fp32 if dtype == torch.float32 else U.assert_bf16)(got, want, f"block_residual {shape}")


def test_argument_checks(hip_device):
    from wtconv_amd import block_ops
    x = torch.randn(1, 3, 4, 4, device=hip_device)
    w = torch.ones(3, device=hip_device)
    assert not block_ops.usable(x, w, w)                      # odd channel count: the caller keeps the plain path
    with pytest.raises(RuntimeError, match="even"):
        block_ops.channel_norm(x, w, w, 1e-6, True)
    x = torch.randn(1, 4, 4, 4, device=hip_device)
    assert not block_ops.usable(x.requires_grad_(True))       # recorded by autograd: the plain functions are not differentiable ...
    assert block_ops.usable(x, training=True)                 # ... the *_fn variants are
    assert not block_ops.usable(torch.randn(1, 4, 4, 4))      # CPU tensor
    with pytest.raises(ValueError, match="does not match"):
        block_ops.block_residual(torch.randn(1, 4, 4, 3, device=hip_device), torch.randn(1, 4, 4, 4, device=hip_device), None)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_model_inference_fused_blocks_match_plain_blocks(hip_device, dtype, monkeypatch):
    """A small WTConvNeXt at inference with the fused block passes against the same model on the plain
    torch passes (what training runs), same WTConv kernels in both."""
    import wtconvnext
    from wtconv_amd import block_ops
    torch.manual_seed(0)
    m = wtconvnext.WTConvNeXt(depths=(1, 1, 2, 1), dims=(16, 32, 64, 128), num_classes=10, ls_init_value=0.5).to(hip_device).to(dtype).eval()
    x = torch.randn(3, 3, 64, 64, device=hip_device).to(dtype)
    calls = {"n": 0}
    real = block_ops.channel_norm

    def counting(*a, **k):
        calls["n"] += 1
        return real(*a, **k)
    monkeypatch.setattr(block_ops, "channel_norm", counting)
    with torch.no_grad():
        fused = m(x).float().cpu()
    assert calls["n"] == 5 + 4 + 1          # block norms, stem + 3 downsample norms, head norm
    monkeypatch.setattr(block_ops, "usable", lambda *a, **k: False)
    with torch.no_grad():
        plain = m(x).float().cpu()
    if dtype == torch.float32:
        torch.testing.assert_close(fused, plain, rtol=1e-4, atol=1e-4)
    else:
        U.assert_bf16(fused, plain, "model logits")


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype,pdtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16),
                                          (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("nhwc", [True, False])
def test_channel_norm_backward(hip_device, shape, dtype, pdtype, nhwc):
    """dx, dweight, dbias of the backward kernel against torch autograd through F.layer_norm in float64."""
    from wtconv_amd import block_ops
    B, C, H, W = shape
    gen = torch.Generator().manual_seed(B * 31 + C)
    x = (torch.randn(shape, generator=gen) * 2 + 0.5).to(dtype)
    w = (torch.randn(C, generator=gen) * 0.5 + 1).to(pdtype)
    b = torch.randn(C, generator=gen).to(pdtype)
    dy = torch.randn((B, H, W, C) if nhwc else shape, generator=gen).to(dtype)
    xr = x.double().requires_grad_(True)
    wr, br = w.double().requires_grad_(True), b.double().requires_grad_(True)
    _ref_norm(xr, wr, br, 1e-6, nhwc).backward(dy.double())
    xd = x.to(hip_device).requires_grad_(True)
    wd, bd = w.to(hip_device).requires_grad_(True), b.to(hip_device).requires_grad_(True)
    out = block_ops.channel_norm_fn(xd, wd, bd, 1e-6, nhwc)
    out.backward(dy.to(hip_device))
    torch.cuda.synchronize()
    # dx = rstd * (g - mean(g) - xh * mean(g * xh)) cancels (for two channels almost completely: xh is +-1 there), so the
    # absolute floor is set by the size of its terms, rstd * |dy * w|, not by the size of the result
    xf = x.double()
    rstd = 1.0 / torch.sqrt(xf.var(dim=1, unbiased=False, keepdim=True) + 1e-6)
    dyn = dy.double().permute(0, 3, 1, 2) if nhwc else dy.double()
    terms = (rstd * dyn * w.double().reshape(1, -1, 1, 1)).pow(2).mean().sqrt().item()
    tol_x = (U.FP32_RTOL, max(U.FP32_ATOL, 1e-6 * terms)) if dtype == torch.float32 else (U.BF16_RTOL, U.BF16_RTOL * terms)
    torch.testing.assert_close(xd.grad.double().cpu(), xr.grad, rtol=tol_x[0], atol=tol_x[1],
                               msg=lambda m: f"dx {shape} nhwc={nhwc}: {m}")
    # parameter gradients are fp32 sums of products of the (rounded) tensors; compared at the parameter dtype's bar
    pcheck = U.assert_fp32 if (dtype == torch.float32 and pdtype == torch.float32) else U.assert_bf16
    pcheck(wd.grad.float().cpu(), wr.grad.float(), f"dweight {shape}")
    pcheck(bd.grad.float().cpu(), br.grad.float(), f"dbias {shape}")


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype,pdtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16)])
def test_block_residual_backward(hip_device, shape, dtype, pdtype):
    """dy, dshortcut, dgamma against torch autograd through permute / mul / add in float64."""
    from wtconv_amd import block_ops
    B, C, H, W = shape
    gen = torch.Generator().manual_seed(B * 13 + C)
    y = torch.randn(B, H, W, C, generator=gen).to(dtype)
    sc = torch.randn(shape, generator=gen).to(dtype)
    gamma = (torch.randn(C, generator=gen) * 0.7).to(pdtype)
    dout = torch.randn(shape, generator=gen).to(dtype)
    yr, scr, gr = (t.double().requires_grad_(True) for t in (y, sc, gamma))
    (yr.permute(0, 3, 1, 2) * gr.reshape(1, -1, 1, 1) + scr).backward(dout.double())
    yd, scd, gd = (t.to(hip_device).requires_grad_(True) for t in (y, sc, gamma))
    block_ops.block_residual_fn(yd, scd, gd).backward(dout.to(hip_device))
    torch.cuda.synchronize()
    check = U.assert_fp32 if dtype == torch.float32 else U.assert_bf16
    check(yd.grad.float().cpu(), yr.grad.float(), f"dy {shape}")
    check(scd.grad.float().cpu(), scr.grad.float(), f"dshortcut {shape}")
    check(gd.grad.float().cpu(), gr.grad.float(), f"dgamma {shape}")


@pytest.mark.parametrize("shape", [(64, 96, 56, 56), (40, 192, 28, 28), (48, 768, 7, 7)])
def test_block_backward_many_records_reproducible(hip_device, shape):
    """Batches whose per-workgroup records fill every slice of the two-stage column sum (1 600 / 280 / 192 records):
    the parameter gradients against float64 sums computed on the GPU, and bit-identical on a second run (the slices are
    added in a fixed order; the ticket only decides which workgroup does the adding)."""
    from wtconv_amd import block_ops
    B, C, H, W = shape
    gen = torch.Generator().manual_seed(C)
    x = (torch.randn(shape, generator=gen) * 2 + 0.5).bfloat16().to(hip_device)
    dy = torch.randn(B, H, W, C, generator=gen).bfloat16().to(hip_device)
    w = (torch.randn(C, generator=gen) * 0.5 + 1).to(hip_device)
    runs = [block_ops.channel_norm_backward(x, dy, w, 1e-6, True) for _ in range(2)]
    xd = x.double()
    xh = (xd - xd.mean(1, keepdim=True)) / torch.sqrt(xd.var(1, unbiased=False, keepdim=True) + 1e-6)
    dyn = dy.double().permute(0, 3, 1, 2)
    U.assert_bf16(runs[0][1].cpu(), (dyn * xh).sum((0, 2, 3)).float().cpu(), f"dweight {shape}")
    U.assert_bf16(runs[0][2].cpu(), dyn.sum((0, 2, 3)).float().cpu(), f"dbias {shape}")
    for a, b in zip(runs[0], runs[1]):
        assert torch.equal(a, b)
    gamma = (torch.randn(C, generator=gen) * 0.7).to(hip_device)
    y = torch.randn(B, H, W, C, generator=gen).bfloat16().to(hip_device)
    res = [block_ops.block_residual_backward(x, y, gamma) for _ in range(2)]
    U.assert_bf16(res[0][1].cpu(), (xd * y.double().permute(0, 3, 1, 2)).sum((0, 2, 3)).float().cpu(), f"dgamma {shape}")
    for a, b in zip(res[0], res[1]):
        assert torch.equal(a, b)


def test_model_training_fused_blocks_match_plain_blocks(hip_device, monkeypatch):
    """One training step of a small WTConvNeXt (fp32): loss and every parameter gradient with the fused block passes
    (forward and backward kernels) against the same model on the plain torch passes."""
    import wtconvnext
    from wtconv_amd import block_ops
    torch.manual_seed(0)
    m = wtconvnext.WTConvNeXt(depths=(1, 1, 2, 1), dims=(16, 32, 64, 128), num_classes=10, ls_init_value=0.5).to(hip_device).train()
    x = torch.randn(3, 3, 64, 64, device=hip_device)
    tgt = torch.randint(0, 10, (3,), device=hip_device)
    calls = {"n": 0}
    real = block_ops.channel_norm_fn

    def counting(*a, **k):
        calls["n"] += 1
        return real(*a, **k)
    monkeypatch.setattr(block_ops, "channel_norm_fn", counting)

    def step():
        for p in m.parameters():
            p.grad = None
        loss = torch.nn.functional.cross_entropy(m(x), tgt)
        loss.backward()
        torch.cuda.synchronize()
        return loss.item(), {n: p.grad.clone() for n, p in m.named_parameters() if p.grad is not None}
    lf, gf = step()
    assert calls["n"] == 5 + 4 + 1          # block norms, stem + 3 downsample norms, head norm
    monkeypatch.setattr(block_ops, "usable", lambda *a, **k: False)
    lp, gp = step()
    assert abs(lf - lp) <= 1e-5 * max(abs(lp), 1.0)
    assert set(gf) == set(gp)
    for n in gp:
        scale = gp[n].abs().max().item()
        torch.testing.assert_close(gf[n], gp[n], rtol=1e-3, atol=1e-5 + 1e-4 * scale, msg=lambda s, n=n: f"{n}: {s}")


def test_block_training_step_graph_replay_matches_eager(hip_device):
    """A training step of a whole WTConvNeXt block (WTConv layer, channel norm, MLP, residual; forward and backward)
    captured in a HIP graph: the library's block passes clear their tickets with kernels, never with memset nodes, so
    every replay -- with new inputs and eager work of the same block in between -- must equal the eager result bit
    for bit: the block's output, the input gradient (which passes through every backward kernel of the block) and the
    gradients of the layer's, the norm's and the layer scale's parameters."""
    import wtconvnext.wtconvnext as M
    torch.manual_seed(3)
    blk = M.WTConvNeXtBlock(32, kernel_size=5, wt_levels=2, ls_init_value=0.5).to(hip_device).train()
    params = [(n, p) for n, p in blk.named_parameters() if p.requires_grad]
    shape = (20, 32, 28, 28)            # 20 * 7 tiles = 140 records: several slices of the two-stage column sum
    xs = torch.randn(*shape, device=hip_device, requires_grad=True)
    gs = torch.randn(*shape, device=hip_device)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            xs.grad = None
            for _, p in params:
                p.grad = None
            blk(xs).backward(gs)
        xs.grad = None
        for _, p in params:
            p.grad = None
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            out = blk(xs)
            out.backward(gs)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    gen = torch.Generator().manual_seed(11)
    for it in range(3):
        xn, gn = torch.randn(*shape, generator=gen), torch.randn(*shape, generator=gen)
        with torch.no_grad():
            xs.copy_(xn.to(hip_device))
            gs.copy_(gn.to(hip_device))
        graph.replay()
        torch.cuda.synchronize()
        got_out, got_dx = out.detach().clone(), xs.grad.clone()
        got = {n: p.grad.clone() for n, p in params}
        held = {n: p.grad for n, p in params}
        for _, p in params:
            p.grad = None
        xe = xn.to(hip_device).requires_grad_(True)
        oe = blk(xe)                                  # eager work between the replays
        oe.backward(gn.to(hip_device))
        torch.cuda.synchronize()
        # (the MLP's bias gradients are torch's own multi-block `sum`, whose captured form holds a memset node and does
        # not replay reliably on this platform: they are not this library's and are left out)
        bad = [n for n, p in params if not n.startswith("mlp.") and not torch.equal(got[n], p.grad)]
        diffs = {n: float((got[n] - dict(params)[n].grad).abs().max()) for n in bad}
        assert torch.equal(got_out, oe.detach()) and torch.equal(got_dx, xe.grad) and not bad, (it, diffs)
        for n, p in params:
            p.grad = held[n]


def test_block_mlp_only_finetuning_keeps_the_mlp_gradients(hip_device):
    """Everything frozen but the MLP of a block, input without gradient: the MLP parameters must still receive their
    gradients (the residual pass goes through the differentiable function, not through raw pointers)."""
    import wtconvnext
    torch.manual_seed(0)
    blk = wtconvnext.wtconvnext.WTConvNeXtBlock(16, wt_levels=2, ls_init_value=0.5).to(hip_device)
    for p in blk.parameters():
        p.requires_grad_(False)
    for p in blk.mlp.parameters():
        p.requires_grad_(True)
    x = torch.randn(2, 16, 14, 14, device=hip_device)
    blk(x).square().sum().backward()
    assert all(p.grad is not None and torch.isfinite(p.grad).all() and p.grad.abs().sum() > 0 for p in blk.mlp.parameters())
    ref = [p.grad.clone() for p in blk.mlp.parameters()]
    # the same through the plain torch passes
    from wtconv_amd import block_ops
    real = block_ops.usable
    block_ops.usable = lambda *a, **k: False
    try:
        for p in blk.mlp.parameters():
            p.grad = None
        blk(x).square().sum().backward()
    finally:
        block_ops.usable = real
    for a, p in zip(ref, blk.mlp.parameters()):
        torch.testing.assert_close(a, p.grad, rtol=1e-4, atol=1e-5)


def test_autocast_keeps_the_plain_passes(hip_device):
    """Under torch.autocast the fused passes step aside (autocast keeps LayerNorm and the residual stream in fp32)."""
    import wtconvnext
    torch.manual_seed(0)
    m = wtconvnext.WTConvNeXt(depths=(1, 1, 1, 1), dims=(16, 32, 64, 128), num_classes=10).to(hip_device).eval()
    x = torch.randn(2, 3, 64, 64, device=hip_device)
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        a = m(x)
        from wtconv_amd import block_ops
        real = block_ops.usable
        block_ops.usable = lambda *a_, **k: False
        try:
            b = m(x)
        finally:
            block_ops.usable = real
    assert a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.parametrize("shape,hidden", [
    ((2, 96, 8, 8), 384),        # (two kernels:) whole tiles, rows of whole 4-pixel vectors
    ((5, 96, 7, 9), 384),        # (two kernels:) odd pixel count: pixel by pixel, tile over several images, remainder
    ((3, 128, 6, 6), 512),       # one kernel: part of a tile, a slice of hidden units a workgroup, 4-pixel vectors
    ((1, 192, 11, 3), 768),      # (two kernels:) one pixel more than the smallest taken
    ((70, 192, 28, 28), 64),     # one kernel: a single slice of hidden units, many tiles
    ((2, 256, 14, 14), 1024),    # (two kernels)
    ((2, 384, 14, 14), 1536),
    ((168, 384, 14, 14), 1536),  # one kernel: enough tiles to go unsplit
    ((1, 384, 13, 11), 192),     # (two kernels)
    ((168, 384, 14, 14), 4096),  # one kernel: the bias of all hidden units ends where the LDS does
])
@pytest.mark.parametrize("layer_scale", [True, False])
def test_fused_block_against_fp64(hip_device, shape, hidden, layer_scale):
    """LayerNorm, MLP, layer scale and shortcut, in the one kernel or the two for few pixels, against float64 on the same
    bfloat16 values."""
    import torch.nn.functional as F
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
    rel = ((d(got) - want).norm() / want.norm()).item()
    assert rel < 4e-3, rel
    rms = want.pow(2).mean().sqrt()
    assert ((d(got) - want).abs() / torch.maximum(want.abs(), rms)).max().item() < 6e-2


@pytest.mark.parametrize("shape,hidden", [
    ((5, 96, 29, 31), 384), ((20, 128, 14, 14), 512), ((10, 192, 15, 13), 768), ((3, 256, 25, 27), 1024), ((8, 384, 14, 14), 1536),
    ((4, 384, 16, 24), 1536), ((7, 128, 16, 24), 512),      # 8-pixel vectors
    ((1, 96, 8, 24), 2048),                                 # a slice a workgroup
])
@pytest.mark.parametrize("layer_scale", [True, False])
def test_one_kernel_block_with_hidden_units_dealt_to_workgroups(hip_device, shape, hidden, layer_scale):
    """The sums of several workgroups meet in a second launch."""
    from wtconv_amd import _lib
    B, C, H, W = shape
    padded = (B * H * W + 127) // 128 * 128
    assert _lib.load().wtconv_block_mlp_workspace_bytes(B, C, H * W, hidden) in [4 * n * C * padded for n in range(2, hidden // 32 + 1)]
    test_fused_block_against_fp64(hip_device, shape, hidden, layer_scale)


def test_fused_block_keeps_infinities_and_nans_to_their_pixels(hip_device):
    from wtconv_amd import _ext
    C = 96
    g = torch.Generator(device=hip_device).manual_seed(0)
    r = lambda *s: torch.randn(*s, generator=g, device=hip_device).bfloat16()
    x, sc = r(2, C, 8, 8), r(2, C, 8, 8)
    args = (1 + r(C), r(C), 1e-6, r(4 * C, C), r(4 * C), r(C, 4 * C), r(C), r(C))
    with torch.no_grad():
        clean = _ext.get().block_mlp(x, sc, *args)
        x[1, 5, 3, 2] = float("nan")
        got = _ext.get().block_mlp(x, sc, *args)
        assert torch.isnan(got[1, :, 3, 2]).all()
        got[1, :, 3, 2] = clean[1, :, 3, 2]
        assert torch.equal(got, clean)
        big = torch.full((4 * C,), float("inf"), device=hip_device, dtype=torch.bfloat16)      # gelu(inf) is inf, not nan
        w2 = torch.ones(C, 4 * C, device=hip_device, dtype=torch.bfloat16)
        assert torch.isinf(_ext.get().block_mlp(clean, sc, *args[:4], big, w2, args[6], None)).all()


def test_fused_block_is_left_alone_where_modules_are_watched(hip_device):
    """Recording, hooks and other activations take the separate passes; the results agree."""
    from wtconvnext.wtconvnext import WTConvNeXtBlock
    torch.manual_seed(0)
    blk = WTConvNeXtBlock(96, wt_levels=2, ls_init_value=0.5).to(hip_device).bfloat16().eval()
    x = torch.randn(2, 96, 14, 14, device=hip_device).bfloat16()
    with torch.no_grad():
        fused = blk(x)
        seen = []
        handle = blk.mlp.fc1.register_forward_hook(lambda m, i, o: seen.append(o.shape))
        apart = blk(x)
        handle.remove()
    assert seen and (fused.float() - apart.float()).norm() < 1e-2 * apart.float().norm()
    blk(x).float().sum().backward()
    assert blk.mlp.fc1.weight.grad is not None


@pytest.mark.parametrize("B,C,H,W,dtype,pdtype", [
    (1, 768, 7, 7, torch.bfloat16, torch.bfloat16), (300, 768, 7, 7, torch.bfloat16, torch.float32),      # odd rows: pairs share a word
    (3, 2, 1, 1, torch.bfloat16, torch.bfloat16), (2, 6, 1, 3, torch.float32, torch.bfloat16), (5, 10, 8, 8, torch.bfloat16, torch.bfloat16),
    (2, 766, 5, 13, torch.float32, torch.float32), (2, 2048, 8, 8, torch.bfloat16, torch.bfloat16),       # a pass of pairs not full; as many as it takes
    (4, 770, 12, 14, torch.bfloat16, torch.bfloat16), (2, 130, 14, 14, torch.float32, torch.float32),     # several trips a channel
])
def test_pool_norm_matches_the_two_operators(hip_device, B, C, H, W, dtype, pdtype):
    from wtconv_amd import _ext
    torch.manual_seed(C + H)
    x = (torch.randn(B, C, H, W, device=hip_device) + 3.).to(dtype)
    w, b = torch.randn(C, device=hip_device).to(pdtype), torch.randn(C, device=hip_device).to(pdtype)
    with torch.no_grad():
        got = _ext.get().pool_norm(x, w, b, 1e-6)
        mean = x.double().mean(dim=(2, 3))
        rounded = mean.to(dtype).double()
        want = torch.nn.functional.layer_norm(rounded, (C,), w.double(), b.double(), 1e-6)
    assert got.shape == (B, C) and got.dtype == dtype
    # Float sums of H W values: the mean is off by up to H W 2^-24 of itself.  Where that moves a mean across a rounding
    # boundary of bfloat16, it is off by a unit, 2^-8 of its 3 + eps; divided by the deviation over the channels, that enters
    # one value and, through the statistics, all of an image a little.
    std = rounded.std(dim=1, unbiased=False, keepdim=True) + 1e-3
    unit = (2. ** -7 if dtype == torch.bfloat16 else H * W * 2. ** -24) * rounded.abs() / std * (w.double().abs() + 1e-3)
    err = (got.double() - want).abs()
    assert (err <= 2 * unit + (2. ** -8 if dtype == torch.bfloat16 else 1e-5) * (want.abs() + 1)).all()
    # nearly all means round alike
    assert (err <= (2. ** -8 if dtype == torch.bfloat16 else 1e-4) * (want.abs() + 1)).double().mean() > 0.97


def test_pool_norm_hands_on_what_is_not_finite_and_leaves_the_rest(hip_device):
    from wtconv_amd import _ext
    fn = _ext.get().pool_norm
    x, w, b = torch.randn(3, 20, 7, 7, device=hip_device), torch.ones(20, device=hip_device), torch.zeros(20, device=hip_device)
    x[1, 4, 6, 6] = float("inf")
    with torch.no_grad():
        got = fn(x, w, b, 1e-6)
        clean = fn(x[::2].contiguous(), w, b, 1e-6)
        assert torch.equal(got[::2], clean) and not got[1].isfinite().any()
        assert fn(x[:, :19].contiguous(), w[:19], b[:19], 1e-6) is None and fn(x.half(), w, b, 1e-6) is None
        assert fn(x.transpose(2, 3)[:, :, :5], w, b, 1e-6) is None and fn(x[:0], w, b, 1e-6) is None
        assert fn(x, w.double(), b, 1e-6) is None and fn(x, w, None, 1e-6) is None
        assert fn(torch.zeros(1, 2, 300, 300, device=hip_device), w[:2], b[:2], 1e-6) is None
    assert fn(x.requires_grad_(), w, b, 1e-6) is None


@pytest.mark.parametrize("kind,part", [("block", "input"), ("block", "norm.weight"), ("block", "mlp.fc1.weight"), ("block", "gamma"),
                                       ("head", "input"), ("head", "norm.bias")])
def test_tangents_take_pytorchs_own_passes(hip_device, kind, part):
    """Forward-mode differentiation at inference: no kernel here has tangents, and none may lose them.  On the CPU, where no
    kernel runs, the same module in double gives the tangent that is wanted."""
    import copy
    import torch.autograd.forward_ad as fwd
    from wtconvnext import wtconvnext as N
    torch.manual_seed(7)
    module = N.WTConvNeXtBlock(96, wt_levels=1, ls_init_value=0.5) if kind == "block" else N._Head(96, 10)
    if kind == "block":
        module.conv_dw = torch.nn.Identity()      # (the layer itself refuses tangents)
    x, step = torch.randn(2, 96, 8, 8), torch.randn(2, 96, 8, 8)

    def tangent(device, dtype):
        m = copy.deepcopy(module).to(device, dtype).requires_grad_(False)
        xin = x.to(device, dtype)
        with fwd.dual_level():
            if part == "input":
                xin = fwd.make_dual(xin, step.to(xin))
            else:
                owner, _, name = part.rpartition(".")
                owner = m.get_submodule(owner)
                p = getattr(owner, name).detach()
                delattr(owner, name)
                setattr(owner, name, fwd.make_dual(p, torch.linspace(-1, 2, p.numel()).square().view(p.shape).to(p)))
            return fwd.unpack_dual(m(xin)).tangent

    got, want = tangent(hip_device, torch.float32), tangent("cpu", torch.float64)
    assert got is not None, "the tangent was lost"
    torch.testing.assert_close(got.cpu().double(), want, rtol=1e-4, atol=1e-4 * want.abs().max().item())
