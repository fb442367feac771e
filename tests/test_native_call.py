"""The native form of the ordinary matmul call (host/call.cpp): what it takes comes out bit for bit as from the Python
path, what it does not take is left to that path, errors included."""
import numpy as np
import pytest
import torch

from _util import to_dev


class Subclass(torch.Tensor):
    pass


@pytest.fixture
def python_only(pkg, monkeypatch):
    def call(*args, **kw):
        with monkeypatch.context() as m:
            m.setattr(pkg.functional, "_native_matmul", None)
            return pkg.functional.woq_matmul_raw(*args, **kw)
    return call


def test_native_call_is_built(pkg):
    assert pkg.functional._native_matmul is not None


@pytest.mark.parametrize("other", ["torch", "abi", "python"])
def test_built_for_something_else(pkg, monkeypatch, other):
    """A file that loads but was compiled against another torch, library interface or Python is not used."""
    F = pkg.functional
    if other == "torch":
        monkeypatch.setattr(torch, "__version__", torch.__version__ + ".other")
    elif other == "abi":
        abi = F.lib.woq_abi_version()

        class Lib:
            woq_matmul, woq_workspace_bytes = F.lib.woq_matmul, F.lib.woq_workspace_bytes

            @staticmethod
            def woq_abi_version():
                return abi + 1

        monkeypatch.setattr(F, "lib", Lib)
    else:
        monkeypatch.setattr(F.sys, "version_info", (3, 99, 0, "final", 0))
    with pytest.warns(UserWarning, match="matmul calls go through Python"):
        assert F._load_native_call() is None


def test_not_a_library(pkg, tmp_path):
    (tmp_path / "woq_call.so").write_bytes(b"not one")
    with pytest.warns(UserWarning, match="does not load"):
        assert pkg.functional._load_native_call(str(tmp_path / "woq_call.so")) is None


@pytest.mark.parametrize("change", ["cpu", "strided", "subclass", "dtype", "k", "n_args"])
def test_not_for_the_native_path(pkg, change):
    """None: the Python path decides (on a machine without a GPU every tensor is refused there)."""
    native = pkg.functional._native_matmul
    act, weight, scales = torch.zeros(2, 64, dtype=torch.float16), torch.zeros(64, 64, dtype=torch.int8), torch.ones(64).half()
    if change == "strided":
        act = torch.zeros(64, 2, dtype=torch.float16).t()
    if change == "subclass":
        act = act.as_subclass(Subclass)
    args = [act, None, weight, scales, None, None, 64, 64, 0, 16, 1.0, 0]
    if change == "dtype":
        args[11] = -1
    if change == "k":
        args[7] = "64"
    assert native(*(args[:-1] if change == "n_args" else args)) is None


def test_errors_are_the_python_paths(pkg):
    F = pkg.functional
    with pytest.raises(RuntimeError, match="runs on the GPU only"):
        F.weight_only_quant_matmul(torch.zeros(1, 64).half(), torch.zeros(64, 64, dtype=torch.int8), torch.ones(64).half(), F.INT8)


def _operands(pkg, dev, fmt, dt, k=512, n=272, seed=0):
    g = torch.Generator().manual_seed(seed)
    F, bits = pkg.functional, 8 if fmt == "int8" else 4
    q = torch.randint(-128, 127, (k, n * bits // 8), generator=g, dtype=torch.int8)
    w = pkg.ops.preprocess_weights_for_mixed_gemm(q, torch.int8 if bits == 8 else torch.quint4x2, dt).to(dev)
    rows = () if fmt == "int8" else (k // 128,)
    table = torch.float16 if fmt == "w4a8" else dt
    scales = (torch.rand(*rows, n, generator=g) * 0.01 + 0.001).to(table).to(dev)
    zeros = None if fmt == "int8" else (torch.randn(*rows, n, generator=g) * 0.01).to(table).to(dev)
    return w, scales, zeros, torch.rand(k, generator=g).to(dt).to(dev), torch.randn(n, generator=g).to(dt).to(dev)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [(512,), (1, 512), (3, 7, 512), (0, 512), (70, 512)])
@pytest.mark.parametrize("fmt", ["int8", "int4", "w4a8", "w4a8 e4m3"])
def test_native_bits(pkg, dev, python_only, fmt, shape, dt):
    F = pkg.functional
    direct = fmt == "w4a8 e4m3"
    fmt = fmt.split()[0]
    w, scales, zeros, smooth, bias = _operands(pkg, dev, fmt, dt)
    act = torch.randn(*shape, generator=torch.Generator().manual_seed(1)).to(dt).to(dev)
    if direct:
        act = act.to(torch.float8_e4m3fn)
    smooth = None if direct or fmt == "int8" else smooth
    algo = (F.INT8_WEIGHT if fmt == "int8" else F.ZERO | F.BIAS) | (F.FP8_ALPHA if fmt == "w4a8" else 0) \
        | (F.PRE_QUANT_SCALE if smooth is not None else 0)
    kw = dict(n=272, k=512, group_size=0 if fmt == "int8" else 128, quant_algo=algo, alpha=0.5 if fmt == "w4a8" else 1.0, out_dtype=dt)
    args = (act, smooth, w, scales, zeros, None if fmt == "int8" else bias)
    got = F._native_matmul(*args, 272, 512, kw["group_size"], algo, kw["alpha"], F._WOQ_DT[dt])
    assert isinstance(got, torch.Tensor) and not got.requires_grad
    want = python_only(*args, **kw)
    assert got.shape == want.shape and got.dtype == want.dtype and torch.equal(got, want)
    assert torch.equal(F.woq_matmul_raw(*args, **kw), want)


@pytest.mark.gpu
def test_native_call_streams_graphs_and_modes(pkg, dev, python_only):
    """The current stream's queue, capture into a graph, and what the path leaves to Python on the GPU."""
    F = pkg.functional
    w, scales, zeros, smooth, bias = _operands(pkg, dev, "int4", torch.bfloat16)
    act = torch.randn(4, 512, generator=torch.Generator().manual_seed(2)).bfloat16().to(dev)
    kw = dict(n=272, k=512, group_size=128, quant_algo=F.ZERO, out_dtype=torch.bfloat16)
    want = python_only(act, None, w, scales, zeros, None, **kw)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        F.woq_matmul_raw(act, None, w, scales, zeros, None, **kw)
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = F.woq_matmul_raw(act, None, w, scales, zeros, None, **kw)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)

    native = lambda a: F._native_matmul(a, None, w, scales, zeros, None, 272, 512, 128, F.ZERO, 1.0, F._WOQ_DT[torch.bfloat16])
    assert torch.equal(native(torch.nn.Parameter(act)), want) and not native(torch.nn.Parameter(act)).requires_grad
    assert native(act.as_subclass(Subclass)) is None and native(act.float()) is None and native(act[:, ::2]) is None
    assert native(act.t().contiguous().t()) is None

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert native(act) is None
    with pytest.raises(RuntimeError):  # no data pointer inside vmap, as before
        torch.func.vmap(lambda a: F.woq_matmul_raw(a, None, w, scales, zeros, None, **kw))(act)
    with pytest.raises(pkg.WoqError):  # the library's own refusals come through
        F.woq_matmul_raw(act, None, w, scales, None, None, **kw)
