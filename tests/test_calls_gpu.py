"""The ordinary calls in csrc/py_calls.cc against the Python code they stand in for: the same results bit for bit (the same kernels on
the same operands), and None - so that the Python code runs - for everything that is not an ordinary call."""
import pytest

import torch


def module(tcu):
    return tcu._native()


@pytest.mark.gpu
def test_calls_give_what_python_gives(tcu, device, monkeypatch):
    half = lambda *shape: (torch.randn(*shape, device=device) * 0.3).half()
    a, b, s = half(48, 80), half(64, 80), half(1024, 8192)  # (s: split over K, through a workspace)
    q, k, v = half(2, 3, 64, 128), half(2, 3, 640, 128), half(2, 3, 640, 128)
    x, W, bias, h0, c0 = half(5, 32, 64), half(4 * 48, 64 + 48), half(4 * 48), half(32, 48), torch.randn(32, 48, device=device)
    A, B, C = half(3, 64, 64), half(3, 64, 64), half(3, 64, 64)
    idx = torch.tensor([[3], [1], [3], [9]], device=device)

    def op():
        o = torch.empty(64 * 128, dtype=torch.float16, device=device)
        tcu.flash_attention_fwd(q[0, 0].flatten(), k[0, 0].flatten(), v[0, 0].t().contiguous().flatten(), o, 64, 640, 128, 128, scale=0.1)
        return o

    def scatter():
        d = torch.ones(8, 6, device=device)
        tcu.scatter_nd(d, idx, torch.ones(4, 6, device=device), mode="add")
        return d

    long = half(24, 48, 64), half(4 * 272, 64 + 272), half(4 * 272)  # the time loop in one launch
    calls = [lambda: tcu.gemm(a, b), lambda: tcu.gemm(a, b, out_dtype=torch.float32), lambda: tcu.gemm(s, s),
             lambda: tcu.b2b_gemm(A, B, C), lambda: tcu.b2b_gemm(A[0], B[0], C[0], out_dtype=torch.float32),
             lambda: tcu.flash_attention(q, k, v), lambda: tcu.flash_attention(q, k, v, scale=0.25), op, scatter,
             lambda: tcu.lstm(x, W, bias), lambda: tcu.lstm(x, W, bias, h0, c0), lambda: tcu.lstm(*long)]
    native = [c() for c in calls]

    class Absent:
        def __getattr__(self, name):
            return lambda *args: None

    monkeypatch.setattr(tcu, "_ready_calls", Absent())
    for c, got in zip(calls, native):
        want = c()
        for g, w in zip(got if isinstance(got, tuple) else (got,), want if isinstance(want, tuple) else (want,)):
            assert g.shape == w.shape and g.dtype == w.dtype and g.device == w.device and torch.equal(g, w)


@pytest.mark.gpu
def test_calls_leave_the_rest_to_python(tcu, device):
    m = module(tcu)
    half = lambda *shape: torch.zeros(*shape, dtype=torch.float16, device=device)
    a, b = half(16, 16), half(16, 16)

    class Sub(torch.Tensor):
        pass

    f16 = torch.float16
    for args in ((a.cpu(), b, f16), (a.float(), b, f16), (a, half(32, 16).t()[:, :16], f16), (a, half(16, 32), f16), (a, b[0], f16), (a, b, torch.int32),
                 (a, b, None), (a.as_subclass(Sub), b, f16), (half(0, 16), b, f16), (half(17, 16), b, f16), (None, b, f16), (a, b)):
        assert m.gemm(*args) is None
    assert m.b2b_gemm(half(1, 32, 64), half(64, 64), half(64, 64), f16) is None and m.b2b_gemm(half(48, 64), half(64, 32), half(64, 64), f16) is None
    q = half(2, 64, 64)
    for args in ((q, half(1, 64, 64), q, None), (q, q, half(2, 32, 64), None), (q, q, q, 1), (q, q, q.float(), None), (q[0, 0], q[0, 0], q[0, 0], None)):
        assert m.flash_attention(*args) is None
    o = half(64 * 128)
    for sizes in ((64, 64, 128, 128, 1.0, 0), (64, 64, 128, 64, 1.0, 1), (64, 64, 128, 128, 1, 1), (2 ** 33, 64, 128, 128, 1.0, 1), (True, 64, 128, 128, 1.0, 1)):
        assert m.flash_attention_fwd(o, o, o, o, *sizes) is None
    x, W, bias = half(2, 16, 16), half(64, 32), half(64)
    assert m.lstm(x, W, bias[:48], None, None) is None and m.lstm(x, W, bias, half(16, 32), None) is None and m.lstm(x, W, bias, None, half(16, 16)) is None
    d, idx = torch.zeros(4, 4, device=device), torch.zeros(2, 1, dtype=torch.int64, device=device)
    for args in ((d, idx, d[:1], 0), (d, idx.int(), d[:2], 0), (d, idx, d[:2].half(), 0), (d, idx, d[:2], 7), (d, idx[:0], d[:0], 0)):
        assert m.scatter_nd(*args) is None
    assert m.gemm(torch.nn.Parameter(a), b, f16).requires_grad is False


def test_calls_without_a_device_leave_errors_to_python(tcu):
    with pytest.raises(ValueError, match="device memory"):
        tcu.gemm(torch.zeros(16, 16, dtype=torch.float16), torch.zeros(16, 16, dtype=torch.float16))
    with pytest.raises(ValueError, match="device memory"):
        tcu.scatter_nd(torch.zeros(4, 4), torch.zeros(1, 1, dtype=torch.int64), torch.zeros(1, 4))


def test_calls_are_those_of_this_interpreter(tcu, monkeypatch):
    """The module's name is one that other interpreters do not load; without it, or with one compiled for another torch, the Python code
    makes the calls and says so once."""
    import os
    import subprocess
    import sys
    import sysconfig
    import warnings

    assert module(tcu).__file__.endswith("_calls" + sysconfig.get_config_var("EXT_SUFFIX"))
    other = subprocess.run([sys.executable, "-c", "import torch; torch.__version__ = '0.0.1'; import tiledcuda_amd._calls"], text=True,
                           cwd=os.path.dirname(os.path.dirname(tcu.__file__)), capture_output=True)
    assert other.returncode != 0 and "ImportError: compiled for torch" in other.stderr
    monkeypatch.setattr(tcu, "_ready_calls", None)
    monkeypatch.delattr(tcu, "_calls", raising=False)
    monkeypatch.setitem(sys.modules, "tiledcuda_amd._calls", None)
    with pytest.warns(RuntimeWarning, match="_calls"):
        absent = tcu._native()
    assert absent.gemm(1, 2, 3) is None and absent.lstm() is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert tcu._native() is absent
    with pytest.raises(ValueError, match="device memory"):
        tcu.gemm(torch.zeros(16, 16, dtype=torch.float16), torch.zeros(16, 16, dtype=torch.float16))


@pytest.mark.gpu
def test_entries_inside_torch_compile(tcu, device):
    """Functions that torch.compile traces call the entries, every one of them, without a warning about a function it does not know."""
    import warnings

    half = lambda *shape: (torch.randn(*shape, device=device) * 0.3).half()
    a, q = half(64, 64), half(2, 64, 64)
    x, W, bias = half(5, 32, 64), half(4 * 48, 64 + 48), half(4 * 48)
    flat, idx = half(64 * 128), torch.tensor([[3], [1]], device=device)

    def op(t):
        o = torch.empty_like(t)
        tcu.flash_attention_fwd(t, flat, flat, o, 64, 64, 128, 128, scale=0.1)
        return o

    def scatter(t):
        d = torch.ones(8, 64, device=device).half()
        tcu.scatter_nd(d, idx, t[:2].contiguous(), mode="add")
        return d

    for f, t in ((lambda t: tcu.gemm(t * 2, a), a), (lambda t: tcu.b2b_gemm(t * 2, a, a), a), (lambda t: tcu.flash_attention(t * 2, q, q), q),
                 (lambda t: op(t * 2), flat), (lambda t: tcu.lstm(t * 2, W, bias)[0], x), (lambda t: scatter(t * 2), a)):
        want = f(t) + 1
        with warnings.catch_warnings():
            warnings.filterwarnings("error", message=".*does not know how to trace")
            assert torch.equal(torch.compile(lambda t: f(t) + 1, backend="eager")(t), want)
