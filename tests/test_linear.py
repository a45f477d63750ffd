"""RansLinear host logic (no GPU): the uniform quantiser, the loud
failure without a device, and what reaches a kernel."""
import ctypes

import numpy as np
import pytest
import torch


def test_quantize_uniform_hits_entropy(rans):
    import rans_linear as L
    w = torch.from_numpy(np.random.default_rng(0).standard_normal((256, 512)).astype(np.float32))
    for bits in (2.25, 3.25, 4.25):
        codes, step = L.quantize_uniform(w, bits)
        assert codes.shape == (256, 512) and codes.dtype == np.int32
        assert step.shape == (512,) and np.all(step == step[0])
        assert abs(L._entropy(codes) - bits) < 0.02
        # dequantisation error of a uniform quantiser is at most step/2
        assert np.abs(codes * step[0] - w.numpy()).max() <= step[0] / 2 + 1e-6


def test_ranslinear_fails_without_gpu(rans):
    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    import rans_linear as L
    codes = np.random.default_rng(1).integers(-5, 6, size=(64, 128)).astype(np.int32)
    with pytest.raises(RuntimeError):
        L.RansLinear.from_codes(codes, np.ones(128, np.float32), tune=False)


class _Lib:
    """Stands in for the library: records the calls that would go to the GPU
    and answers 0, as after a launch."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        return lambda *a: (self.calls.append((name, a)), 0)[1]


@pytest.fixture
def on_cpu(rans, monkeypatch):
    """rans_linear with CPU tensors taken for plain ones of the GPU."""
    import rans_linear as L
    monkeypatch.setattr(L, "_plain", lambda *t: True)
    monkeypatch.setattr(rans, "_stream", lambda: 0)
    return L


@pytest.mark.parametrize("y_dtype", [torch.float32, torch.bfloat16, torch.float16, torch.float64])
@pytest.mark.parametrize("bias", [False, True])
def test_finish_takes_the_products_it_has_a_kernel_for(on_cpu, y_dtype, bias):
    """A product in f16 (what a dense layer returns under autocast's default
    type) or any other type but f32 and bf16 is finished by torch."""
    lib = _Lib()
    y = torch.randn(5, 16, generator=torch.Generator().manual_seed(1)).to(y_dtype)
    b = torch.full((16,), 0.25) if bias else None
    for out in (torch.float32, torch.bfloat16, torch.float16):
        got = on_cpu._finish(lib, y, b, out)
        assert got.dtype is out and got.shape == y.shape
        if y_dtype in (torch.float32, torch.bfloat16):
            assert bool(lib.calls) == (y_dtype is not out or bias and out is not torch.float32)
        else:
            assert not lib.calls
            assert torch.equal(got, (y.float() if b is None else y.float() + b).to(out))
        lib.calls.clear()
        if bias:
            assert on_cpu._finish(lib, y, b.double(), out).dtype is out and not lib.calls


class _Matrix:
    """Stands in for a RansMatrix of 8 rows and 16 columns on the CPU."""
    rows, cols, fused_rows_limit, matmul_rows = 8, 16, 8, 64

    def __init__(self):
        self.lib, self.fused = _Lib(), []
        self.w = torch.randn(8, 16, generator=torch.Generator().manual_seed(4)).bfloat16()

    def decode(self):
        return self.w

    def matmul(self, x, bias, dtype):
        self.fused.append(bias)
        return (x.float() @ self.w.float().t() + (0 if bias is None else bias)).to(dtype)


def test_bias_of_another_length_stays_with_torch(on_cpu):
    """A kernel reads one value per output: a single value, which torch's add
    broadcasts, and a wrong length, which it refuses, never reach one."""
    x = torch.randn(20, 16, generator=torch.Generator().manual_seed(5))
    for rows, kernel in ((20, "fused"), (100, "finish")):
        m = _Matrix()
        lin = on_cpu.RansLinear(m)
        full = torch.linspace(-1, 1, 8)
        xs = x.repeat(5, 1)[:rows]
        want = torch.nn.functional.linear(xs.bfloat16(), m.w).float()
        lin.bias = full
        lin(xs)
        assert len(m.fused) == (kernel == "fused")
        assert len(m.lib.calls) == (kernel == "finish")
        m.fused.clear(), m.lib.calls.clear()
        for bias in (full[:1], full[None], torch.tensor(0.5)):
            lin.bias = bias
            assert torch.equal(lin(xs), want + bias)
        for n in (7, 9, 16):
            lin.bias = torch.zeros(n)
            with pytest.raises(RuntimeError):
                lin(xs)
        assert not m.fused and not m.lib.calls


class _Device(torch.Tensor):
    is_cuda = True


def test_matmul_checks_its_bias(rans, monkeypatch):
    """RansMatrix.matmul hands the kernel f32 biases of the matrix's rows
    only: other types are converted, other lengths and devices refused."""
    monkeypatch.setattr(rans, "_CUDA", torch.device("cpu"))
    monkeypatch.setattr(rans, "_stream", lambda: 0)
    m = object.__new__(rans.RansMatrix)
    m.rows, m.cols, m.stream_cols, m.lib, m._desc = 8, 64, 64, _Lib(), rans.RansMatrixDesc()
    seen = []

    def kernel(desc, x, batch, bias, *rest):
        seen.append(None if bias is None else
                    np.ctypeslib.as_array((ctypes.c_float * m.rows).from_address(bias)).copy())
        return 0
    m.lib.rans_w64_matmul = kernel
    x = torch.zeros(3, 64).as_subclass(_Device)
    want = torch.arange(8, dtype=torch.float32)
    strided = torch.stack([want, -want], 1)[:, 0]
    for b in (want, want.bfloat16(), want.half(), want.double(), want.int(), strided):
        m.matmul(x, b)
        np.testing.assert_array_equal(seen.pop(), want.numpy())
    m.matmul(x)
    assert seen.pop() is None
    for b in (want[:7], want[:1], torch.tensor(1.0), torch.zeros(9), torch.zeros(1, 8),
              torch.zeros(8, device="meta")):
        with pytest.raises(ValueError):
            m.matmul(x, b)
    assert not seen


def test_what_watches_a_tensor_keeps_it_from_the_kernels(rans, monkeypatch):
    """A kernel called through a pointer is hidden from gradients, forward
    mode, vmap and dispatch and function modes, so tensors that one of these
    watches are not plain; the mode of a default device watches nothing."""
    import rans_linear as L
    from torch.autograd import forward_ad
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(rans, "_device", lambda: -1)

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    t = torch.zeros(3)
    assert L._plain(t) and L._plain(t, None) and L._plain(t, t)
    for mode in (Function, Dispatch):
        with mode():
            assert not L._plain(t)
    with torch.device("cpu"):
        assert L._plain(t)
        with Function():
            assert not L._plain(t)
    with forward_ad.dual_level():
        assert not L._plain(t)
    seen = []
    torch.func.vmap(lambda v: (seen.append(L._plain(v)), v)[1])(torch.zeros(2, 3))
    assert seen == [False]
    for other in (torch.zeros(3, requires_grad=True), torch.nn.Parameter(t, requires_grad=False)):
        assert not L._plain(other) and not L._plain(t, other) and not L._plain(other, t)
    assert L._plain(t)
