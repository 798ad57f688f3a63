"""The operators' calls in native code (csrc/host/mnb_calls.cc): what they decline, and that they give what the Python path gives."""
import ctypes
import gc
import importlib.util
import sys
import sysconfig
import threading
import weakref
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from onnxruntime_amd import MatMulNBits, MatMulNBitsMlp, MatMulNBitsQkv, MnbError, _lib, matmul_nbits
from onnxruntime_amd.synthetic import make_case

gpu = pytest.mark.gpu
NAMES = ("linear", "variant", "mlp", "qkv", "quantize")


def test_declines_what_is_no_plain_tensor_of_the_gpu():
    _lib.load()
    entry, a = _lib.ADDRESS, torch.zeros(2, 128, dtype=torch.float16)
    linear = lambda *args: _lib.calls().linear(entry["MnbGemm"], entry["MnbGemmWorkspaceSize"], 16, 128, 4, 32, 0, *args)  # noqa: E731
    assert linear(_lib.DTYPE_FLOAT16, a, a, None, None) is None
    assert linear(_lib.DTYPE_FLOAT16, [1.0], a, None, None) is None
    assert linear(99, a, a, None, None) is None
    for name in NAMES:
        with pytest.raises(TypeError, match="arguments expected"):
            getattr(_lib.calls(), name)(1, 2)
    with pytest.raises(TypeError):
        linear("ten", a, a, None, None)


def test_a_call_holds_the_plan_that_it_was_given(monkeypatch):
    """PrePack of another thread replaces op.plan while a call asks for its scratch or launches: the plan stays until it is over."""
    op = MatMulNBits(256, 32, 4, 32, dtype=torch.bfloat16)
    op.packed, op.plan = torch.zeros(1), _lib.MnbVariantPlan()
    plan, result = weakref.ref(op.plan), object()

    def variant(*args):
        op.plan = _lib.MnbVariantPlan()
        gc.collect()
        assert plan() is not None and any(x is plan() for x in args)
        return result
    monkeypatch.setattr(matmul_nbits, "_calls", SimpleNamespace(variant=variant))
    assert op.Compute(torch.zeros(1, 256, dtype=torch.bfloat16)) is result


def test_a_plan_is_an_object_of_its_size():
    _lib.load()
    entry, a = _lib.ADDRESS, torch.zeros(2, 128, dtype=torch.float16)
    call = lambda plan: _lib.calls().variant(entry["MnbVariantGemm"], entry["MnbVariantGemmWorkspaceSize"], plan, 16, 128,  # noqa: E731
                                             _lib.DTYPE_FLOAT16, a, a, None, None)
    plan = _lib.MnbVariantPlan()
    assert call(plan) is None
    for bad in (ctypes.addressof(plan), None, bytes(8)):
        with pytest.raises(TypeError):
            call(bad)


@pytest.mark.filterwarnings("error")
@pytest.mark.parametrize("zp", [np.True_, np.False_, 1.0, 1, True, False])
def test_zero_points_are_a_truth_value_of_any_type(zp):
    """The presence of zero points has always been put through int(): numpy's truth values, and 1.0, are taken without a warning."""
    _lib.load()
    entry, a = _lib.ADDRESS, torch.zeros(2, 128, dtype=torch.float16)
    assert _lib.calls().linear(entry["MnbGemm"], entry["MnbGemmWorkspaceSize"], 16, 128, 4, 32, zp, _lib.DTYPE_FLOAT16, a, a, None, None) is None


def test_the_package_is_imported_without_the_extension(monkeypatch):
    """As without the library itself: what needs it says how to build it."""
    import onnxruntime_amd
    monkeypatch.setitem(sys.modules, "onnxruntime_amd._calls", None)
    monkeypatch.delattr(onnxruntime_amd, "_calls", raising=False)
    spec = importlib.util.spec_from_file_location("onnxruntime_amd.imported_again", matmul_nbits.__file__)
    again = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(again)
    for needs_it in (lambda: again.MatMulNBits(128, 16, 4, 32), lambda: again.MatMulNBitsMlp(128, 16, 4, 32),
                     lambda: again.quantize_blockwise(torch.zeros(32, 16), 4, 32, True)):
        with pytest.raises(RuntimeError, match="onnxruntime_amd.build"):
            needs_it()


def test_the_extension_is_that_of_this_python_and_torch(monkeypatch):
    """It reads the structures of both: another Python does not find it, and another torch is told to build it again."""
    assert _lib.calls().__file__.endswith("_calls" + sysconfig.get_config_var("EXT_SUFFIX"))
    monkeypatch.setattr(torch, "__version__", "1.13.1+rocm5.2")
    with pytest.raises(RuntimeError, match="onnxruntime_amd.build"):
        _lib.calls()


def dev(x):
    return None if x is None else torch.from_numpy(np.ascontiguousarray(x)).cuda()


class Paths:
    """Both ways of a call: as it is, and with the native calls declining everything.  `taken` counts native results."""

    def __init__(self, monkeypatch):
        self.native, self.taken = matmul_nbits._calls, 0
        self.patch = monkeypatch

        def count(name):
            def call(*args):
                y = getattr(self.native, name)(*args)
                self.taken += y is not None
                return y
            return call
        self.counting = SimpleNamespace(**{n: count(n) for n in NAMES})
        self.declining = SimpleNamespace(**{n: lambda *args: None for n in NAMES})

    def both(self, call, native=True):
        before = self.taken
        self.patch.setattr(matmul_nbits, "_calls", self.counting)
        got = call()
        assert (self.taken > before) == native
        self.patch.setattr(matmul_nbits, "_calls", self.declining)
        want = call()
        self.patch.setattr(matmul_nbits, "_calls", self.counting)
        got, want = (t if isinstance(t, tuple) else (t,) for t in (got, want))
        assert len(got) == len(want)
        for g, w in zip(got, want):
            if g is None:
                assert w is None
                continue
            assert g.shape == w.shape and g.dtype == w.dtype and g.device == w.device and g.stride() == w.stride()
            assert not g.requires_grad and torch.equal(g, w)
        return got


@pytest.fixture
def paths(monkeypatch):
    return Paths(monkeypatch)


@gpu
@pytest.mark.parametrize("dtype,bits,zp,g_idx", [(torch.float16, 4, True, False), (torch.float16, 8, False, False),
                                                 (torch.float32, 4, True, False), (torch.bfloat16, 4, False, False),
                                                 (torch.float16, 4, True, True)])
def test_products_of_every_form(paths, dtype, bits, zp, g_idx):
    K, N = 328, 45
    c = make_case(70, N, K, bits, 32, np.float16, has_zp=zp, has_bias=True, seed=5)
    op = MatMulNBits(K, N, bits, 32, dtype=dtype, has_zero_points=zp, has_bias=True, has_g_idx=g_idx)
    order = torch.randperm(K) // 32 if g_idx else None
    assert op.PrePack(dev(c.B), dev(c.scales).to(dtype), dev(c.zero_points), None if order is None else order.int().cuda())
    a, bias = dev(c.A).to(dtype), dev(c.bias).to(dtype)
    for rows in (1, 16, 70):
        for use in (None, bias):
            paths.both(lambda: op.Compute(a[:rows], bias=use))
    wide = torch.zeros(70, K + 24, dtype=dtype, device="cuda")
    wide[:, 8:8 + K] = a
    paths.both(lambda: op.Compute(wide[:, 8:8 + K], bias=bias))            # rows apart
    paths.both(lambda: op.Compute(wide[3:4, 8:8 + K], bias=bias))
    paths.both(lambda: op.Compute(a.clone().requires_grad_(), bias=bias))  # (the result has no gradient either way)
    for other in (a.t().contiguous().t(), a.reshape(7, 10, K), a[0], a[:0]):  # copied, reshaped, empty: the Python path's
        paths.both(lambda: op.Compute(other, bias=bias), native=False)
    paths.both(lambda: op.Compute(a, bias=bias, out=torch.empty(70, N, dtype=dtype, device="cuda")), native=False)


@gpu
@pytest.mark.parametrize("M", [1, 40])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_fused_operators(paths, M, dtype):
    K = 256
    parts = []
    for seed, n in enumerate((48, 48, 64, 24, 24)):
        c = make_case(M, n, K, 4, 32, np.float16, has_bias=True, seed=seed)
        parts.append((dev(c.B), dev(c.scales).to(dtype), dev(c.bias).to(dtype)))
    a, norm = dev(c.A).to(dtype), (1 + torch.rand(K, device="cuda")).to(dtype)
    mlp, qkv = MatMulNBitsMlp(K, 48, 4, 32, dtype=dtype), MatMulNBitsQkv(K, 64, 24, 4, 32, dtype=dtype)
    if not (mlp.supported and qkv.supported):
        pytest.skip("no kernel for this type")
    assert mlp.PrePack(*parts[0], *parts[1]) and qkv.PrePack(*parts[2], *parts[3], *parts[4])
    for op in (mlp, qkv):
        paths.both(lambda: op.Compute(a))
        paths.both(lambda: op.Compute(a, norm_scale=norm))
        for skip in (torch.randn_like(a), torch.randn_like(a[:1])):  # of A's rows, and one row for all
            paths.both(lambda: op.Compute(a, skip=skip, norm_scale=norm))
            paths.both(lambda: op.Compute(a, skip=skip, norm_scale=norm, want_skip_sum=True))
        paths.both(lambda: op.Compute(a, skip=a.reshape(1, M, K), norm_scale=norm), native=False)
        for bad in (dict(skip=a), dict(want_skip_sum=True, norm_scale=norm), dict(norm_scale=norm[:-1]),
                    dict(skip=a[:, :-1], norm_scale=norm)):
            with pytest.raises(MnbError):
                op.Compute(a, **bad)


@gpu
def test_what_was_refused_is_refused_and_wrappers_raise(paths):
    K, N = 256, 32
    c = make_case(4, N, K, 4, 32, np.float16, has_bias=True, seed=1)
    op = MatMulNBits(K, N, 4, 32, dtype=torch.float16, has_bias=True)
    assert op.PrePack(dev(c.B), dev(c.scales))
    a = dev(c.A)
    paths.patch.setattr(matmul_nbits, "_calls", paths.counting)
    for call, match in ((lambda: op.Compute(a.float()), "dtype"), (lambda: op.Compute(a[:, :-8]), "last dimension"),
                        (lambda: op.Compute(a, bias=dev(c.bias)[:-1]), None), (lambda: op.Compute(a[:1].expand(4, K)), "lda")):
        with pytest.raises(MnbError, match=match):
            call()
    with pytest.raises(RuntimeError):
        torch.func.vmap(op.Compute)(a[:, None])
    assert paths.taken == 0

    class Sub(torch.Tensor):
        pass
    paths.both(lambda: op.Compute(a.as_subclass(Sub)).as_subclass(torch.Tensor), native=False)
    with torch.device("cpu"):  # (a mode that sees torch.empty)
        paths.both(lambda: op.Compute(a), native=False)


@gpu
@pytest.mark.parametrize("dtype,bits,block", [(torch.float16, 4, 32), (torch.float32, 8, 64), (torch.float16, 2, 128)])
@pytest.mark.parametrize("symmetric", [True, False])
def test_quantiser(paths, dtype, bits, block, symmetric):
    w = torch.randn(200, 77, device="cuda").to(dtype)
    for src, native in ((w, True), (w[:, 3:70], True), (w[:1], True), (w.t(), False)):
        paths.both(lambda: matmul_nbits.quantize_blockwise(src, bits, block, symmetric), native=native)
    for bad in (3, 0):
        with pytest.raises((MnbError, ZeroDivisionError)):
            matmul_nbits.quantize_blockwise(w, bad, block, symmetric)


@gpu
def test_streams_and_threads(paths):
    K, N = 1024, 512
    c = make_case(37, N, K, 4, 32, np.float16, seed=2)
    op = MatMulNBits(K, N, 4, 32, dtype=torch.float16)
    assert op.PrePack(dev(c.B), dev(c.scales))
    a = dev(c.A)
    want, wrong = op.Compute(a), []
    torch.cuda.synchronize()

    def work():
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(20):
                y = op.Compute(a)
            stream.synchronize()
            if not torch.equal(y, want):
                wrong.append(1)
    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@gpu
def test_the_plan_outlives_its_replacement(monkeypatch):
    """The entry point (a stub) reads the plan after op.plan has been replaced while the call asked for its scratch."""
    K, N = 264, 45
    c = make_case(4, N, K, 4, 32, np.float16, seed=3)
    op = MatMulNBits(K, N, 4, 32, dtype=torch.bfloat16)
    assert op.PrePack(dev(c.B), dev(c.scales).to(torch.bfloat16))
    plan, seen = weakref.ref(op.plan), []
    want = bytes(op.plan)

    def workspace(device, nbytes, stream):
        op.plan = None
        gc.collect()
        return torch.empty(nbytes, dtype=torch.uint8, device=device)

    def gemm(address, *args):
        seen.append(plan() is not None and ctypes.string_at(address, len(want)) == want)
        return _lib.OK
    args = _lib.SIGNATURES["MnbVariantGemm"][1]
    stub = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, *args[1:])(gemm)
    monkeypatch.setitem(_lib.ADDRESS, "MnbVariantGemm", ctypes.cast(stub, ctypes.c_void_p).value)
    op._get_workspace = workspace
    op.Compute(dev(c.A).to(torch.bfloat16).repeat(10, 1))  # (40 rows: with scratch)
    assert seen == [True] and op.plan is None


@gpu
@pytest.mark.parametrize("name", ["MnbGemm", "MnbVariantGemm", "MnbMlpGemm", "MnbQkvGemm", "MnbQuantizeBlockwise"])
@pytest.mark.parametrize("code", ["EP_FAIL", "INVALID_ARGUMENT"])
def test_a_failed_call_raises_and_is_not_made_again(monkeypatch, name, code):
    """What the entry point (a stub) reports is raised from that call: a second one could hide it and would repeat its launches."""
    K, N, code = 256, 48, getattr(_lib, code)
    c = make_case(4, N, K, 4, 32, np.float16, seed=3)
    a, parts, calls = dev(c.A), (dev(c.B), dev(c.scales)), []
    if name == "MnbQuantizeBlockwise":
        call = lambda: matmul_nbits.quantize_blockwise(a, 4, 32, True)  # noqa: E731
    elif name == "MnbMlpGemm":
        op = MatMulNBitsMlp(K, N, 4, 32)
        assert op.PrePack(*parts, None, *parts, None)
        call = lambda: op.Compute(a)  # noqa: E731
    elif name == "MnbQkvGemm":
        op = MatMulNBitsQkv(K, N, N, 4, 32)
        assert op.PrePack(*parts, None, *parts, None, *parts, None)
        call = lambda: op.Compute(a)  # noqa: E731
    else:
        dtype = torch.bfloat16 if name == "MnbVariantGemm" else torch.float16
        op = MatMulNBits(K, N, 4, 32, dtype=dtype)
        assert op.PrePack(parts[0], parts[1].to(dtype))
        call = lambda: op.Compute(a.to(dtype))  # noqa: E731

    def entered(*args):
        calls.append(1)
        return code
    stub = ctypes.CFUNCTYPE(ctypes.c_int, *_lib.SIGNATURES[name][1])(entered)
    monkeypatch.setitem(_lib.ADDRESS, name, ctypes.cast(stub, ctypes.c_void_p).value)
    with pytest.raises(MnbError) as e:
        call()
    assert e.value.code == code and calls == [1]
