"""CPU-side checks of the C-ABI library and the host layer (no GPU compute): the library
loads, exports every symbol the header declares, validates arguments before touching the
device, and the Python modules keep the reference's constructor/state-dict surface."""
import ctypes
import os
import re
import subprocess
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib():
    from wtconv_amd import _build, _lib
    if _build.is_stale():
        _build.build_library()
    return _lib.load()


def test_header_symbols_are_exported(lib):
    from wtconv_amd import _lib
    hdr = open(os.path.join(ROOT, "include", "wtconv_hip.h")).read()
    hdr = re.sub(r"/\*.*?\*/", "", hdr, flags=re.S)
    declared = set(re.findall(r"\b(wtconv[0-9a-z_]*)\s*\(", hdr))
    assert declared == set(_lib.EXPORTS), (declared ^ set(_lib.EXPORTS))
    for name in declared:
        assert hasattr(lib, name), name
    assert lib.wtconv_abi_version() == _lib.ABI_VERSION == 6
    assert lib.wtconv_max_kernel_size() == 7


def _prototypes(header):
    """name -> (result, argument types) of a header's functions, as ctypes types; enums and pointers by their kind."""
    text = re.sub(r"/\*.*?\*/", "", open(os.path.join(ROOT, "include", header)).read(), flags=re.S)
    text = re.sub(r"typedef struct \{.*?\} \w+;", "", text, flags=re.S)
    scalar = {"int": ctypes.c_int, "long long": ctypes.c_longlong, "size_t": ctypes.c_size_t, "float": ctypes.c_float}

    def kind(t):
        return "pointer" if "*" in t else scalar[" ".join(t.split()[:-1]) if t.split()[-1] not in ("int", "long", "float", "size_t") else t]
    out = {}
    for res, name, args in re.findall(r"^(int|size_t|const char\*) (wtconv\w*)\(([^)]*)\);", text, flags=re.M):
        args = [a.strip() for a in args.split(",") if a.strip() not in ("", "void")]
        out[name] = ("pointer" if "*" in res else scalar[res], [kind(a) for a in args])
    return out


def test_second_header_is_exported_and_bound_as_declared(lib):
    from wtconv_amd import _lib
    of = lambda t: t if t in (ctypes.c_int, ctypes.c_longlong, ctypes.c_size_t, ctypes.c_float) else "pointer"
    for header, exports in (("wtconv_ops.h", _lib.OPS_EXPORTS), ("wtconv_hip.h", _lib.EXPORTS)):
        declared = _prototypes(header)
        assert set(declared) == set(exports), set(declared) ^ set(exports)
        for name, (res, args) in exports.items():
            assert hasattr(lib, name), name
            assert (of(res), [of(a) for a in args]) == declared[name], name
    define = re.search(r"#define WTCONV_OPS_VERSION (\d+)", open(os.path.join(ROOT, "include", "wtconv_ops.h")).read())
    assert lib.wtconv_ops_version() == _lib.OPS_VERSION == int(define.group(1))


def test_workspace_sizes(lib):
    C, K, L = 96, 5, 3
    fwd = lib.wtconv2d_workspace_bytes(128, C, 56, 56, K, L, 0)
    assert fwd >= 4 * (C * (1 + 4 * L) * K * K + C) and fwd % 256 == 0
    assert lib.wtconv2d_workspace_bytes(128, C, 56, 56, K, L, 1) == fwd
    par = lib.wtconv2d_workspace_bytes(128, C, 56, 56, K, L, 2)
    assert par >= 4 * C * ((1 + 4 * L) * K * K + 1)
    # the one-call backward pass shares one workspace between its two passes
    assert lib.wtconv2d_workspace_bytes(128, C, 56, 56, K, L, 3) == max(fwd, par)
    assert lib.wtconv1d_workspace_bytes(64, 64, 4096, K, 4, 3) == max(
        lib.wtconv1d_workspace_bytes(64, 64, 4096, K, 4, 1), lib.wtconv1d_workspace_bytes(64, 64, 4096, K, 4, 2))
    assert lib.wtconv1d_workspace_bytes(64, 64, 4096, 5, 4, 0) >= 4 * (64 * 9 * 5 + 64)
    assert lib.wtconv2d_workspace_bytes(0, C, 56, 56, K, L, 0) == 0
    assert lib.wtconv2d_workspace_bytes(1, 1, 20000, 20000, K, L, 0) == 0     # plane beyond 2^28 elements
    # planes whose pyramid exceeds LDS: the workspace also holds the fp32 pyramid(s)
    big = lib.wtconv2d_workspace_bytes(2, 4, 400, 400, K, L, 0)
    assert big >= 4 * 2 * 4 * (400 * 400 + 200 * 200 * 4 // 4)
    assert lib.wtconv2d_workspace_bytes(2, 4, 400, 400, K, L, 2) >= 2 * (big - fwd)


def _params(L=2):
    from wtconv_amd import _lib
    p = _lib.Params()
    p.base_weight = p.base_scale = 0x1000          # never dereferenced: validation fails first
    for i in range(L):
        p.wt_weight[i] = 0x1000
        p.wt_scale[i] = 0x1000
    return p


@pytest.mark.parametrize("kw,code,needle", [
    (dict(K=4), -1, "odd and positive"),
    (dict(K=9), -2, "largest built kernel"),
    (dict(L=6), -1, "wt_levels"),
    (dict(L=0), -1, "wt_levels"),
    (dict(B=0), -1, "positive"),
    (dict(H=0), -1, "spatial size"),
    (dict(dtype=7), -1, "dtype"),
    (dict(x=0), -1, "null"),
    (dict(H=400, W=400), -3, "workspace"),     # larger than LDS: the HBM pyramid needs a larger workspace
    (dict(ws_bytes=16), -3, "workspace"),
    (dict(H=20000, W=20000), -2, "2^28"),      # 32-bit offsets inside a plane
])
def test_forward_argument_validation(lib, kw, code, needle):
    """Bad arguments are rejected with a code and a message before any kernel launch."""
    a = dict(x=0x1000, out=0x2000, B=2, C=4, H=8, W=8, K=5, L=2, dtype=0, pdtype=0, ws=0x3000, ws_bytes=1 << 20)
    a.update(kw)
    p = _params(2)
    rc = lib.wtconv2d_forward(a["x"], a["out"], ctypes.byref(p), a["B"], a["C"], a["H"], a["W"], a["K"], a["L"],
                              a["dtype"], a["pdtype"], a["ws"], a["ws_bytes"], None)
    assert rc == code
    assert needle in lib.wtconv_last_error().decode()


def test_static_scratch_refuses_rows_longer_than_a_workgroup_takes(lib):
    """5000 pixels in a row are 1250 pieces of four: LDS would hold the plane, no workgroup walks its rows, and the step
    that takes it instead needs more than the static scratch."""
    rc = lib.wtconv2d_forward_static(0x1000, 0x2000, ctypes.byref(_params(1)), 2000, 64, 1, 5000, 1, 1, 0, 0, None)
    assert rc == -2 and "scratch" in lib.wtconv_last_error().decode()


def test_size_queries_answer_for_sizes_that_do_not_exist(lib):
    """0 for extents of zero and below, in every position, and an error code from the calls (in a process of their own: a
    division by zero would end it)."""
    code = """
import itertools
from wtconv_amd import _lib
lib = _lib.load()
for c in (0, -1, -96):
    assert lib.wtconv_block_mlp_supported(1, c, 196, 64) == 0 and lib.wtconv_block_mlp_workspace_bytes(1, c, 196, 64) == 0
    p = _lib.MlpParams(*[0x1000] * 7)
    assert lib.wtconv_block_mlp(0x1000, 0x2000, 0x3000, p, 1, c, 196, 64, 1e-6, 1, 1, 0x4000, 1 << 20, None) < 0
queries = [(lib.wtconv_block_mlp_supported, (1, 96, 196, 64)), (lib.wtconv_block_mlp_workspace_bytes, (1, 96, 196, 64)),
           (lib.wtconv_patch_conv_supported, (0, 1, 96, 8, 8, 192)), (lib.wtconv_patch_conv_workspace_bytes, (0, 1, 96, 8, 8, 192)),
           (lib.wtconv_patch_conv_supported, (1, 1, 3, 16, 16, 96)), (lib.wtconv_patch_conv_workspace_bytes, (1, 1, 3, 16, 16, 96)),
           (lib.wtconv_mlp_supported, (196, 96, 384)), (lib.wtconv_mlp_backward_workspace_bytes, (196, 96, 384, 7)),
           (lib.wtconv_block_workspace_bytes, (1, 96, 196, 1))]
for fn, sizes in queries:
    first = 1 if fn in (lib.wtconv_patch_conv_supported, lib.wtconv_patch_conv_workspace_bytes) else 0
    for i, bad in itertools.product(range(first, first + 3), (0, -1, -2 ** 31)):
        assert fn(*sizes[:i], bad, *sizes[i + 1:]) == 0, (fn.__name__, i, bad)
print("answered")
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=ROOT, timeout=300)
    assert r.returncode == 0 and "answered" in r.stdout, (r.returncode, r.stderr[-2000:])


def test_mlp_sizes_beyond_32_bit_indices_are_refused(lib):
    """Threads of a launch and values of a weight gradient are counted in 32 bits."""
    ws = lib.wtconv_mlp_backward_workspace_bytes
    assert ws(64, 65536, 65536, 7) == 0 and lib.wtconv_mlp_supported(64, 65536, 65536) == 0      # 2^31 threads add up the weight gradients
    assert ws(64, 32768, 65536, 7) > 2 ** 33
    assert ws(1 << 27, 384, 1536, 7) == 0 and ws(1 << 30, 96, 128, 7) == 0                       # 2^33 threads of a product
    assert ws(1 << 24, 384, 1536, 7) > 2 ** 35


@pytest.mark.parametrize("C,hidden,faster,slower", [
    (96, 384, (1, 401408), ()), (384, 1536, (1, 200704), ()), (512, 2048, (1, 100352), ()), (1024, 2048, (1, 100352), ()),
    (768, 3072, (1, 49, 12544, 25088), (50176, 200704)), (1536, 1536, (25088,), (50176,)),
    (896, 3584, (784, 6272), (12544, 50176)), (768, 4096, (784, 6272), (25088,)),
    (1024, 4096, (1, 784, 2048), (3136, 6272, 12544, 50176)), (2048, 2048, (1024,), (6272,)),
    (1536, 6144, (), (784, 12544)), (2048, 8192, (), (1, 200, 12544)), (4096, 4096, (), (200, 12544)),
])
def test_mlp_training_kernels_are_offered_where_they_are_faster(lib, C, hidden, faster, slower):
    """Sizes on both sides of the line (measured as faster or slower than the library's passes); the calls take all of them."""
    for pixels in faster + slower:
        assert lib.wtconv_mlp_supported(pixels, C, hidden) == (pixels in faster), pixels
        assert lib.wtconv_mlp_backward_workspace_bytes(pixels, C, hidden, 7) > 0


@pytest.mark.parametrize("C,two,one", [
    (96, ((32, 64), (3332, 384), (1664, 768), (488, 2048)), ((96, 2048), (64, 4096), (560, 2048), (1666, 4096))),
    (128, ((32, 64), (2340, 256), (256, 512), (1952, 512)), ((64, 512), (2500, 512), (192, 2048), (1120, 1024), (1250, 4096))),
    (192, ((32, 192), (1664, 768), (312, 4096)), ((833, 4096), (1666, 4096))),
    (256, ((32, 256), (1250, 1024), (244, 4096)), ((625, 4096),)),
    (384, ((196, 1536), (832, 1536), (312, 4096)), ((833, 4096), (834, 1536))),
    (512, ((624, 2048), (312, 4096)), ((625, 4096), (626, 64))), (768, ((49, 3072), (416, 3072)), ((416, 4096),)),
    (1024, ((49, 4096), (256, 4096), (312, 1024)), ((312, 4096),)),
])
def test_few_pixels_take_the_kernels_that_are_faster(lib, C, two, one):
    """Pixels x hidden units on both sides of the line between the two kernels for few pixels and the one kernel (from 512
    channels: the separate passes), each side measured.  The two kernels' workspace holds the hidden values of whole tiles."""
    for pixels, hidden in two + one:
        hid = 2 * ((pixels + 31) // 32 * 32) * hidden
        few = lib.wtconv_block_mlp_workspace_bytes(1, C, pixels, hidden) == hid
        if (pixels, hidden) in two or C < 512:
            assert few == ((pixels, hidden) in two), (pixels, hidden)
        assert lib.wtconv_block_mlp_supported(1, C, pixels, hidden) == (C < 512 or (pixels, hidden) in two)


@pytest.mark.parametrize("C,cout,faster,slower", [
    (96, 192, (1, 512), ()), (384, 768, (1, 64, 2048), ()), (512, 1024, (1, 64, 2048), ()), (512, 6144, (64, 512), ()),
    (96, 480, (1, 64, 512), (2048,)), (96, 992, (1, 64), (170, 512)), (128, 480, (170, 512), (2048,)),
    (192, 224, (64, 512, 2048), ()), (192, 480, (64,), (170, 512)), (256, 224, (512, 2048), ()), (256, 736, (), (64, 170)),
    (384, 224, (64, 170, 512), (2048,)), (384, 416, (16,), (64, 170)), (512, 224, (170, 512), (2048,)), (512, 544, (1, 16), (64, 256)),
    (256, 3200, (64, 512), ()), (384, 640, (64, 512), ()), (384, 2048, (16, 32), (64, 256)), (512, 640, (64, 512), (2048,)),
    (512, 896, (64, 170), (256, 2048)), (512, 1152, (32, 100), (256,)),
])
def test_downsample_kernels_are_offered_where_they_are_faster(lib, C, cout, faster, slower):
    """Images of 14 x 14 on both sides of the lines for output channels that the many-pixel split does not divide."""
    for images in faster + slower:
        assert lib.wtconv_patch_conv_supported(0, images, C, 14, 14, cout) == (images in faster), images


def test_null_parameter_pointer_rejected(lib):
    from wtconv_amd import _lib
    p = _lib.Params()
    rc = lib.wtconv1d_forward(0x1000, 0x2000, ctypes.byref(p), 1, 2, 64, 5, 2, 0, 0, 0x3000, 1 << 20, None)
    assert rc == -1 and "null parameter" in lib.wtconv_last_error().decode()
    g = _lib.ParamGrads()
    rc = lib.wtconv2d_backward_params(0x1000, 0x2000, ctypes.byref(_params(2)), ctypes.byref(g), 1, 2, 8, 8, 5, 2,
                                      0, 0, 0x3000, 1 << 20, None)
    assert rc == -1 and "gradient pointer" in lib.wtconv_last_error().decode()


def test_one_call_backward_validates_like_its_passes(lib):
    """wtconv2d_backward / wtconv1d_backward reject bad arguments before any launch, with the
    message of the pass that found them."""
    from wtconv_amd import _lib
    g = _lib.ParamGrads()
    rc = lib.wtconv2d_backward(0x1000, 0x2000, 0x3000, ctypes.byref(_params(2)), ctypes.byref(g), 2, 4, 8, 8, 4, 2,
                               0, 0, 0x4000, 1 << 20, None)
    assert rc == -1 and "odd and positive" in lib.wtconv_last_error().decode()
    rc = lib.wtconv1d_backward(0x1000, 0x2000, 0, ctypes.byref(_params(2)), ctypes.byref(g), 1, 2, 64, 5, 2,
                               0, 0, 0x4000, 1 << 20, None)
    assert rc == -1 and "null" in lib.wtconv_last_error().decode()
    rc = lib.wtconv2d_backward(0x1000, 0x2000, 0x3000, ctypes.byref(_params(2)), ctypes.byref(g), 2, 4, 8, 8, 5, 2,
                               0, 0, 0x4000, 16, None)
    assert rc == -3 and "workspace" in lib.wtconv_last_error().decode()


def test_check_raises_python_exceptions(lib):
    from wtconv_amd import _lib
    p = _params(2)
    rc = lib.wtconv2d_forward(0x1000, 0x2000, ctypes.byref(p), 2, 4, 8, 8, 4, 2, 0, 0, 0x3000, 1 << 20, None)
    with pytest.raises(ValueError, match="odd and positive"):
        _lib.check(rc, "forward")
    rc = lib.wtconv2d_forward(0x1000, 0x2000, ctypes.byref(p), 2, 4, 400, 400, 5, 2, 0, 0, 0x3000, 1 << 20, None)
    with pytest.raises(RuntimeError, match="workspace of"):
        _lib.check(rc, "forward")


# ------------------------------------------------------------------ module surface
def test_reference_module_surface_and_init(lib):
    import wtconv
    from wtconv.wtconv1d import WTConv1d
    from oracle import wtconv_ref as R
    torch.manual_seed(0)
    m = wtconv.WTConv2d(8, 8, kernel_size=5, stride=1, bias=True, wt_levels=3, wt_type='db1')
    torch.manual_seed(0)
    r = R.RefWTConv2d(8, 8, 5, wt_levels=3)
    assert list(m.state_dict().keys()) == list(r.state_dict().keys())
    for (k, a), (_, b) in zip(m.state_dict().items(), r.state_dict().items()):
        assert torch.equal(a, b), k
    assert (m.in_channels, m.wt_levels, m.stride, m.dilation) == (8, 3, 1, 1)
    assert sum(p.numel() for p in m.parameters()) == (59 + 104 * 3) * 8
    assert not m.wt_filter.requires_grad and not m.iwt_filter.requires_grad
    torch.manual_seed(1)
    m1 = WTConv1d(4, 4, 3, wt_levels=2)
    torch.manual_seed(1)
    r1 = R.RefWTConv1d(4, 4, 3, wt_levels=2)
    for (k, a), (_, b) in zip(m1.state_dict().items(), r1.state_dict().items()):
        assert torch.equal(a, b), k


def test_fast_twin_surface(lib):
    from fast_wtconv.wtconv_cuda import WTConv2d as Fast
    import fast_wtconv
    assert fast_wtconv.WTConv2d is Fast
    m = Fast(4, 4, 5, 1, 2, False)       # positional: kernel_size, stride, wt_levels, bias
    assert m.base_bias is None and m.wt_levels == 2 and m.kernel_size == 5 and m.stride == 1
    assert set(m.state_dict()) == {"base_weight", "base_scale", "wt_weights.0", "wt_weights.1",
                                   "wt_scales.0", "wt_scales.1"}
    assert m.wt_weights[0].shape == (16, 1, 5, 5) and torch.all(m.wt_scales[1] == 0.1)
    with pytest.raises(AssertionError):
        Fast(4, 8)
    with pytest.raises(AssertionError):
        Fast(4, 4, wt_levels=6)


class _Doubled(torch.nn.Module):
    def forward(self, w):
        return 2 * w


def _prune(m, name):
    from torch.nn.utils import prune
    prune.l1_unstructured(m, name, 0.5)


def _parametrize(m, name):
    torch.nn.utils.parametrize.register_parametrization(m, name, _Doubled())


@pytest.mark.parametrize("how", [_prune, _parametrize, torch.nn.utils.spectral_norm])
@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("names", [("base_weight",), ("wt_weights.0",), ("wt_weights.1", "wt_scales.1"), ("base_bias",)])
def test_fast_twin_calls_with_the_weights_its_attributes_have(lib, monkeypatch, names, bias, how):
    """Pruned, parametrized and spectrally normalised parameters: what the layer is called with is what a look at the
    attribute gives, for every parameter and every level."""
    from fast_wtconv.wtconv_cuda import WTConv2d as Fast
    from wtconv_amd import modules
    if names[0] == "base_bias" and (not bias or how is torch.nn.utils.spectral_norm):
        pytest.skip("no such parameter, or not a matrix")
    torch.manual_seed(0)
    m = Fast(4, 4, 3, 1, 2, bias)
    for full in names:
        owner, _, name = full.rpartition(".")
        how(m.get_submodule(owner), name)
    m.eval()          # (spectral_norm: no further power iteration, so that two looks see the same tensor)
    seen = []
    monkeypatch.setattr(modules.Fn, "wtconv2d", lambda x, *a, **kw: seen.append(a) or x)
    m(torch.zeros(1, 4, 8, 8))
    bw, bb, bs, ws, ss = seen[0]
    assert torch.equal(bw, m.base_weight) and torch.equal(bs, m.base_scale)
    assert torch.equal(bb, m.base_bias) if bias else bb is None
    assert len(ws) == len(ss) == 2
    for i in range(2):
        assert torch.equal(ws[i], m.wt_weights[i]) and torch.equal(ss[i], m.wt_scales[i])
    changed = getattr(m.get_submodule(names[0].rpartition(".")[0]), names[0].rpartition(".")[2])
    assert not isinstance(changed, torch.nn.Parameter)       # the effective tensor, not a stored one


def test_constructor_errors(lib):
    import wtconv
    with pytest.raises(AssertionError):
        wtconv.WTConv2d(4, 8)
    with pytest.raises(NotImplementedError, match="db1"):
        wtconv.WTConv2d(4, 4, wt_type='db2')
    with pytest.raises(ValueError, match="odd and positive"):
        wtconv.WTConv2d(4, 4, kernel_size=4)
    with pytest.raises(ValueError, match="largest built kernel"):
        wtconv.WTConv2d(4, 4, kernel_size=9)


def test_cpu_tensor_is_refused_loudly(lib):
    """No CPU fallback: a CPU tensor is an error, not a silent slow path."""
    import wtconv
    m = wtconv.WTConv2d(4, 4, 3, wt_levels=1)
    with pytest.raises(RuntimeError, match="GPU only"):
        m(torch.randn(1, 4, 8, 8))


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    from wtconv_amd import _lib
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setenv("WTCONV_HIP_LIB", str(tmp_path / "nope.so"))
    with pytest.raises(_lib.WTConvLibraryError, match="no fallback"):
        _lib.load()


def test_library_of_another_version_is_refused_with_a_message(monkeypatch, tmp_path):
    """Also one that lacks entry points of this version."""
    import subprocess
    from wtconv_amd import _lib
    hdr = open(os.path.join(ROOT, "include", "wtconv_hip.h")).read()
    assert int(re.search(r"#define WTCONV_ABI_VERSION (\d+)", hdr).group(1)) == _lib.ABI_VERSION
    old = tmp_path / "old.so"
    src = f"int wtconv_abi_version(void) {{ return {_lib.ABI_VERSION - 1}; }}"
    subprocess.run(["gcc", "-shared", "-fPIC", "-x", "c", "-", "-o", str(old)], input=src, text=True, check=True)
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setenv("WTCONV_HIP_LIB", str(old))
    with pytest.raises(_lib.WTConvLibraryError, match="ABI version"):
        _lib.load()


def test_cpp_autograd_node_builds_loads_and_declines_host_tensors(lib):
    """The C++ autograd node (host code only) compiles against the installed PyTorch, takes the library's entry
    points by address, and hands anything that is not a GPU tensor in a kernel dtype back to the Python path."""
    from wtconv_amd import _build, _ext
    if (not os.path.exists(_build.BINDING_PATH)
            or os.path.getmtime(_build.BINDING_PATH) < os.path.getmtime(_build.BINDING_SRC)):
        _build.build_binding()
        _ext._tried, _ext._mod = False, None
    ext = _ext.get()
    assert ext is not None
    C, K = 4, 3
    x = torch.randn(1, C, 8, 8)
    args = (torch.randn(C, 1, K, K), torch.randn(C), torch.randn(1, C, 1, 1), [torch.randn(4 * C, 1, K, K)],
            [torch.randn(1, 4 * C, 1, 1)])
    assert ext.layer(x, *args, 2, K, 1) is None
    assert ext.layer(x, args[0], None, *args[2:], 2, K, 1) is None


def test_planes_of_one_round_stay_in_one_round(lib):
    """K = 7 runs one workgroup a CU: up to 128 channels their chunks make no more workgroups than there are compute units (a
    few more take a second round), and at least two thirds of that where there are planes enough."""
    for B, C, H, W, L in [(52, 86, 20, 22, 4), (45, 102, 24, 19, 2), (132, 55, 12, 10, 2), (256, 96, 11, 10, 2), (20, 56, 63, 47, 5),
                          (45, 50, 15, 12, 2), (16, 72, 45, 37, 2), (128, 116, 15, 16, 2)]:
        records = lib.wtconv2d_workspace_bytes(B, C, H, W, 7, L, 2) // 4 - C
        assert 170 <= records // ((1 + 4 * L) * 49 + 1) <= 256, (B, C, H, W, L)
