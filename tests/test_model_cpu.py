"""The WTConvNeXt harness reproduces the parameter counts the reference logs hold
(logs/val_tiny.out:4, val_small.out:4, val_base.out:4) -- the only known answers the
reference has for the model shell."""
import pytest
import torch


@pytest.mark.parametrize("name,count", [("wtconvnext_tiny", 30595624), ("wtconvnext_small", 54448936),
                                        ("wtconvnext_base", 94225128)])
def test_param_counts(name, count):
    import wtconvnext
    with torch.device("meta"):
        m = getattr(wtconvnext, name)()
    assert sum(p.numel() for p in m.parameters()) == count


def test_structure_and_init():
    import wtconvnext
    from oracle import wtconv_ref as R
    torch.manual_seed(0)
    m = wtconvnext.wtconvnext_tiny(depths=(1, 1, 1, 1), num_classes=10)
    levels = [s.blocks[0].conv_dw.wt_levels for s in m.stages]
    assert levels == [5, 4, 3, 2]
    blk = m.stages[0].blocks[0]
    # the model init re-draws the WTConv convolutions (trunc-normal 0.02) and zeroes biases
    w = torch.cat([c.weight.flatten() for c in blk.conv_dw.wavelet_convs])
    assert abs(w.std().item() - 0.02) < 2e-3 and w.abs().max() < 0.15
    assert torch.all(blk.conv_dw.base_conv.bias == 0)
    assert torch.all(blk.conv_dw.wavelet_scale[0].weight == 0.1)
    assert torch.all(blk.gamma == 1e-6)
    nwd = m.no_weight_decay()
    assert "stages.0.blocks.0.conv_dw.base_scale.weight" in nwd
    assert "stages.3.blocks.0.conv_dw.wavelet_scale.1.weight" in nwd
    keys = set(m.state_dict())
    assert {"stem.0.weight", "stem.1.weight", "stages.1.downsample.1.weight", "stages.2.blocks.0.mlp.fc1.weight",
            "stages.0.blocks.0.conv_dw.wavelet_convs.4.weight", "head.norm.weight", "head.fc.bias"} <= keys
    # the oracle class plugs into the same hook and yields the same state-dict keys
    torch.manual_seed(0)
    r = wtconvnext.wtconvnext_tiny(depths=(1, 1, 1, 1), num_classes=10, wtconv_class=R.RefWTConv2d)
    assert set(r.state_dict()) == keys
    out = r(torch.randn(1, 3, 64, 64))
    assert out.shape == (1, 10)


def test_drop_path_schedule_and_head_options():
    """drop_path_rate spreads linearly over all blocks (reference wtconvnext.py:309), is the identity
    in eval mode and keeps the expectation in training; head_init_scale scales the classifier
    (wtconvnext.py:483-493); reset_classifier / forward_head(pre_logits) follow the reference's API."""
    import wtconvnext
    from oracle import wtconv_ref as R
    torch.manual_seed(0)
    m = wtconvnext.wtconvnext_tiny(depths=(1, 2, 1, 1), num_classes=7, drop_path_rate=0.4, head_init_scale=0.5,
                                   wtconv_class=R.RefWTConv2d)
    rates = [getattr(b.drop_path, "drop_prob", 0.0) for s in m.stages for b in s.blocks]
    assert rates == pytest.approx([0.0, 0.1, 0.2, 0.3, 0.4])
    torch.manual_seed(0)
    ref = wtconvnext.wtconvnext_tiny(depths=(1, 2, 1, 1), num_classes=7, wtconv_class=R.RefWTConv2d)
    assert torch.allclose(m.head.fc.weight, 0.5 * ref.head.fc.weight)
    x = torch.randn(2, 3, 64, 64)
    m.eval()
    ref.eval()
    with torch.no_grad():
        ref.head.fc.load_state_dict(m.head.fc.state_dict())
        assert torch.equal(m(x), ref(x))                     # stochastic depth is off in eval mode
        feats = m.forward_features(x)
        assert m.forward_head(feats, pre_logits=True).shape == (2, 768)
    dp = wtconvnext.wtconvnext.DropPath(0.25).train()
    y = dp(torch.ones(4000, 3))
    kept = (y[:, 0] != 0).float().mean().item()
    assert abs(kept - 0.75) < 0.03 and torch.all((y == 0) | (y == 1 / 0.75))
    m.reset_classifier(3)
    assert m(x).shape == (2, 3) and m.num_classes == 3
    m.set_grad_checkpointing(True)
    m.train()
    m(x.requires_grad_(True)).sum().backward()
    assert x.grad is not None


class _Quantised(torch.Tensor):
    """A weight without memory of its own: whatever is done with it runs on `inner`."""

    @staticmethod
    def __new__(cls, inner):
        return torch.Tensor._make_wrapper_subclass(cls, inner.shape, dtype=inner.dtype, device=inner.device)

    def __init__(self, inner):
        self.inner = inner

    __torch_function__ = torch._C._disabled_torch_function_impl

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        inner = lambda t: t.inner if isinstance(t, cls) else t
        res = func(*torch.utils._pytree.tree_map(inner, args), **torch.utils._pytree.tree_map(inner, kwargs or {}))
        return cls(res) if func is torch.ops.aten.detach.default else res


@pytest.fixture
def one_kernel(monkeypatch):
    """block_mlp(...) of the C++ module replaced by one that takes everything; the calls it got."""
    from wtconv_amd import _ext
    calls = []

    class Ext:
        @staticmethod
        def block_mlp(x, *args):
            calls.append(args)
            return x
    monkeypatch.setattr(_ext, "get", lambda: Ext)
    return calls


def _behind_the_layer(dim=8):
    """A block whose first layer hands its input on."""
    from wtconvnext.wtconvnext import WTConvNeXtBlock
    return WTConvNeXtBlock(dim, wtconv_class=lambda *a, **k: torch.nn.Identity()).eval()


@pytest.mark.parametrize("name", ["fc1.weight", "fc1.bias", "fc2.weight", "fc2.bias"])
def test_one_kernel_block_leaves_tensor_subclasses_to_their_own_products(one_kernel, name):
    blk = _behind_the_layer()
    x = torch.randn(2, 8, 4, 4)
    with torch.no_grad():
        blk(x)
        assert len(one_kernel) == 1
        want = blk.mlp(x.permute(0, 2, 3, 1))
        mod = blk.mlp.get_submodule(name.split(".")[0])
        p = getattr(mod, name.split(".")[1])
        setattr(mod, name.split(".")[1], torch.nn.Parameter(_Quantised(p.detach()), requires_grad=False))
        blk(x)
        assert len(one_kernel) == 1
        assert torch.equal(blk.mlp(x.permute(0, 2, 3, 1)), want)


def _global_hook(pre):
    reg = torch.nn.modules.module
    return (reg.register_module_forward_pre_hook if pre else reg.register_module_forward_hook)(lambda *a: None)


class _FunctionMode(torch.overrides.TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("kind", ["hook", "pre-hook", "global hook", "global pre-hook", "forward", "flops", "function mode"])
def test_one_kernel_block_is_not_taken_while_its_modules_are_observed(one_kernel, kind):
    from torch.utils.flop_counter import FlopCounterMode
    blk, x = _behind_the_layer(), torch.randn(2, 8, 4, 4)
    with torch.no_grad():
        if kind == "flops":
            with FlopCounterMode(display=False) as mode:
                blk(x)
            assert mode.get_total_flops() == 2 * 2 * 32 * 8 * 32
        elif kind == "function mode":
            with _FunctionMode():
                blk(x)
        elif kind == "forward":
            plain = blk.mlp.fc1.forward
            blk.mlp.fc1.forward = lambda t: plain(t)
            blk(x)
            del blk.mlp.fc1.forward
        else:
            handle = (_global_hook("pre" in kind) if "global" in kind else
                      blk.mlp.fc1.register_forward_pre_hook(lambda *a: None) if "pre" in kind else
                      blk.mlp.fc1.register_forward_hook(lambda *a: None))
            blk(x)
            handle.remove()
        assert not one_kernel
        blk(x)
        with torch.device("cpu"):          # a default device is no observer
            blk(x)
    assert len(one_kernel) == 2


def test_compiling_comes_before_the_binding(monkeypatch):
    """While a model is being compiled the fused passes step aside before they ask for the C++ binding: loading it is not
    traceable, and a model may be compiled before its first call."""
    from wtconv_amd import block_ops
    from wtconvnext.wtconvnext import WTConvNeXt
    model = WTConvNeXt(depths=(1, 1, 1, 1), dims=(8, 16, 24, 32), num_classes=2)
    blk, x = model.stages[0].blocks[0], torch.zeros(1, 3, 8, 8)
    monkeypatch.setattr(block_ops._ext, "get", lambda: pytest.fail("asked for"))
    monkeypatch.setattr(torch.compiler, "is_compiling", lambda: True)
    assert block_ops.block_mlp(x, x, blk.norm, blk.mlp, blk.gamma) is None
    assert block_ops.patch_conv(x, model.stem, model.stem[0], model.stem[1], True) is None
    assert block_ops.mlp_fn(x, blk.mlp) is None


@pytest.mark.parametrize("kind", ["plain", "pruned", "parametrized", "weight norm", "no bias", "no affine", "approximate", "subclass",
                                  "no layer scale", "hook", "own forward"])
def test_lookups_of_the_binding_find_what_python_finds(kind):
    """The native look-ups of a block's modules against the Python ones, also where a name is no ordinary parameter."""
    from torch.nn.utils import parametrize, prune, weight_norm
    from wtconv_amd import _ext, block_ops, modules
    from wtconvnext.wtconvnext import WTConvNeXtBlock
    native = _ext.lookups()
    if native is None:
        pytest.skip("the binding is not built")
    blk = WTConvNeXtBlock(8, wt_levels=3, ls_init_value=None if kind == "no layer scale" else 1.)
    fc1, level = blk.mlp.fc1, blk.conv_dw.wavelet_convs[1]
    if kind == "pruned":
        for m in (fc1, level):
            prune.random_unstructured(m, "weight", amount=0.5)
    elif kind == "parametrized":
        for m in (fc1, level):
            parametrize.register_parametrization(m, "weight", torch.nn.Identity())
    elif kind == "weight norm":
        for m in (fc1, blk.conv_dw.base_conv):
            weight_norm(m)
    elif kind == "no bias":
        fc1.bias = blk.conv_dw.base_conv.bias = None
    elif kind == "no affine":
        blk.norm = torch.nn.LayerNorm(8, elementwise_affine=False)
    elif kind == "approximate":
        blk.mlp.act = torch.nn.GELU(approximate="tanh")
    elif kind == "subclass":
        fc1.weight = torch.nn.Parameter(_Quantised(fc1.weight.detach()), requires_grad=False)
    elif kind == "hook":
        blk.norm.register_forward_pre_hook(lambda *a: None)
    elif kind == "own forward":
        blk.mlp.act.forward = lambda t: t
    same = lambda a, b: a is b or (type(a) is type(b) and torch.equal(a, b))
    x, y = torch.zeros(2), torch.ones(2)
    got, want = (f(x, y, blk.norm, blk.mlp, blk.gamma) for f in (native.mlp_args, block_ops._mlp_args))
    assert (got is None) == (want is None) == (kind not in ("plain", "no bias", "no layer scale"))
    if got is not None:
        assert len(got) == len(want) and got[4] == want[4] and all(same(a, b) for i, (a, b) in enumerate(zip(got, want)) if i != 4)
    with pytest.MonkeyPatch.context() as patch:
        patch.setattr(_ext, "lookups", lambda: None)
        want = modules._layer_params(blk.conv_dw)
    got = native.layer_params(blk.conv_dw)
    assert all(same(a, b) for a, b in zip(got[:3], want[:3]))
    assert all(len(g) == len(w) == 3 and all(same(a, b) for a, b in zip(g, w)) for g, w in zip(got[3:], want[3:]))
    with pytest.raises(AttributeError):
        native.mlp_args(x, y, blk.norm, torch.nn.Identity(), None)


@pytest.mark.parametrize("where", ["base_conv", "base_scale", "wavelet_convs", "wavelet_scale"])
@pytest.mark.parametrize("replaced", ["base_conv", "base_scale", "wavelet_convs", "wavelet_scale"])
def test_lookups_of_the_binding_outlive_what_a_parametrization_replaces(where, replaced):
    """A parametrized weight runs Python code while a layer's parameters are looked up, and that code may put another module
    in the place of one that the look-up began with: the old one goes, and the answer is the one of Python's own look-up."""
    from torch.nn.utils import parametrize
    import wtconv
    from wtconv_amd import _ext, modules
    if _ext.lookups() is None:
        pytest.skip("the binding is not built")

    class Replaces(torch.nn.Module):
        def __init__(self, layer):
            super().__init__()
            self.layer, self.made = [layer], 0

        def forward(self, w):
            self.made += 1
            fresh = getattr(wtconv.WTConv2d(2, 2, kernel_size=3, wt_levels=2), replaced)
            for p in fresh.parameters():
                p.data.fill_(self.made)
            setattr(self.layer[0], replaced, fresh)
            return w + self.made

    def look_up():
        torch.manual_seed(0)
        layer = wtconv.WTConv2d(2, 2, kernel_size=3, wt_levels=2)
        part = getattr(layer, where)
        replaces = Replaces(layer)
        parametrize.register_parametrization(part if where.startswith("base") else part[0], "weight", replaces, unsafe=True)
        setattr(layer, where, part)      # (registering evaluates the parametrization)
        found = modules._layer_params(layer)
        for _ in range(50):      # (freed memory is not put to another use at once)
            modules._layer_params(layer)
        return [t for p in found for t in (p if isinstance(p, (list, tuple)) else [p])], replaces.made

    got, made = look_up()
    with pytest.MonkeyPatch.context() as patch:
        patch.setattr(_ext, "lookups", lambda: None)
        want, made_in_python = look_up()
    assert made == made_in_python and len(got) == len(want) == 7
    assert all(torch.equal(a, b) for a, b in zip(got, want))
