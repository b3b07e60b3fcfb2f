"""The wrappers' native calls (nihilus_amd/csrc/py_calls.cpp) against the Python way they stand for: the same results, errors and routes.

On the CPU: whatever is not a plain call on GPU tensors is left to the Python way.  On the GPU: the same bits either way over the forms the
wrappers take, and the same errors for the ones they refuse.
"""
import sys
import types

import numpy as np
import pytest
import torch

from nihilus_amd import build, q8_0


def test_the_module_is_built():
    assert q8_0._calls is not None


def test_the_module_is_for_this_torch_and_python():
    tag = build.calls_tag()
    assert q8_0._calls.built_for == tag and torch.__version__ in tag
    assert q8_0._fitting(q8_0._calls) is q8_0._calls
    for other in None, types.SimpleNamespace(), types.SimpleNamespace(built_for=tag.replace(torch.__version__, "0.0.1")):
        assert q8_0._fitting(other) is None


def test_the_library_is_built_without_torch(monkeypatch):
    ran = []
    monkeypatch.setattr(build, "_run", lambda cmd: ran.append(" ".join(cmd)) or "")
    monkeypatch.setitem(sys.modules, "torch", None)  # import torch raises ImportError
    build.build_library()
    assert len(ran) == len(build.SOURCES) + 1 and not any(build.CALLS_SOURCE in c for c in ran)
    with pytest.raises(ImportError):
        build.build_calls()


def test_an_old_module_is_built_again_for_another_torch(monkeypatch):
    ran = []
    monkeypatch.setattr(build, "_run", lambda cmd: ran.append(cmd) or "")
    monkeypatch.setattr(build, "_newest_header_mtime", lambda include: 0.0)
    monkeypatch.setattr(build.os.path, "getmtime", lambda path: 2.0 if path == build.CALLS_PATH else 1.0)
    build.build_calls(incremental=True)
    assert not ran
    monkeypatch.setattr(build, "calls_tag", lambda: "torch 0.0.1 cpython-310")
    build.build_calls(incremental=True)
    assert len(ran) == 2


def test_what_is_no_plain_call_is_left_to_python():
    w, x = torch.zeros(4, dtype=torch.uint8), torch.zeros(4)
    calls = q8_0._calls
    assert calls.mul_mat(w, x, 1, 4, None) is None  # not on a GPU
    assert calls.mul_mat() is None and calls.mul_mat(w, x, 1) is None and calls.mul_mat(1, 2, 3, 4, 5) is None
    assert calls.mul_mat(w, x, 2**70, 4, None) is None and calls.mul_mat(w, x, 1.0, 4, None) is None
    assert calls.gemm(w, w, 1, 1, 1, None) is None and calls.rms_norm_quantize(x, x, 1e-5) is None and calls.gate_up_silu(w, w, w, 1, 1, 1) is None
    with pytest.raises(TypeError, match="w_tiled must be a contiguous"):
        q8_0.mul_mat(w, x, 1, 4)


class _Memory:
    """Stands for a uint8 tensor of n bytes on the GPU: what gate_up_silu asks of its operands, without one."""

    is_cuda, device = True, "cpu"

    def __init__(self, n):
        self.numel = lambda: n

    def is_contiguous(self):
        return True

    def element_size(self):
        return 1

    def data_ptr(self):
        return 4096


@pytest.mark.parametrize("debug", [False, True])
def test_gate_up_refuses_operands_that_are_too_small(monkeypatch, debug):
    # the launch reads what m, n_ff and k say, past the end of a smaller buffer: refused before it
    m, n_ff, k = 40, 256, 384
    real, launched = q8_0._lib.lib(), []

    class Library:
        nh_q8_0_tiled_bytes, nh_q8_0_gate_up_silu_workspace_bytes = real.nh_q8_0_tiled_bytes, real.nh_q8_0_gate_up_silu_workspace_bytes

        def __getattr__(self, name):
            return lambda *args: launched.append(name) or 0

    monkeypatch.setattr(q8_0, "_calls", None)
    monkeypatch.setattr(q8_0._lib, "lib", Library)
    monkeypatch.setattr(q8_0, "_stream", lambda: 0)
    w, a = q8_0.tiled_bytes(n_ff, k), q8_0.tiled_bytes(m, k)
    for sizes in (w - 1, w, a), (w, w - 1, a), (w, w, a - 1), (w // 2, w // 2, a), (0, w, a):
        with pytest.raises(ValueError, match="does not hold"):
            q8_0.gate_up_silu(*map(_Memory, sizes), m, n_ff, k, debug=debug)
    for wrong in (m + 32, n_ff, k), (m, n_ff + 128, k), (m, n_ff, k + 128):
        with pytest.raises(ValueError, match="does not hold"):
            q8_0.gate_up_silu(_Memory(w), _Memory(w), _Memory(a), *wrong, debug=debug)
    assert not launched
    q8_0.gate_up_silu(_Memory(w), _Memory(w + 5), _Memory(a), m, n_ff, k, debug=debug)  # buffers may be larger
    assert len(launched) == 1


class _Subclass(torch.Tensor):
    pass


def _both(monkeypatch, call):
    """call() with the native functions and without: results, or the exceptions' types and texts"""
    out = []
    for native in (q8_0._calls, None):
        monkeypatch.setattr(q8_0, "_calls", native)
        try:
            out.append(call().cpu().numpy())
        except Exception as e:  # noqa: BLE001
            out.append((type(e), str(e)))
    monkeypatch.undo()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("m", [0, 1, 3, 5, 40, 200])
def test_same_bits_either_way(q8, oracle, monkeypatch, m):
    n, k = 384, 1024
    w = q8.tile(q8.fill_weight_blocks(3, n, k), n, k)
    x = q8.fill_activations(4, m * k).reshape(m, k)
    add, norm = q8.fill_activations(5, m * n).reshape(m, n), q8.fill_activations(6, k)
    forms = [lambda: q8.mul_mat(w, x, n, k), lambda: q8.mul_mat(w, x, n, k, residual=add), lambda: q8.mul_mat(w, x, n, k, residual=add.reshape(-1)), lambda: q8.mul_mat(w.reshape(2, -1), x, n, k),
             lambda: q8.rms_norm_quantize(x, norm, 1e-5, tiled=True), lambda: q8.rms_norm_quantize(x, norm.reshape(1, -1), 0, tiled=True)]
    if m == 1:
        forms += [lambda: q8.mul_mat(w, x[0], n, k), lambda: q8.rms_norm_quantize(x[0], norm, 1e-5, tiled=True)]
    if m:
        a = q8.quantize_row_q8_0(x, tiled=True)
        forms += [lambda: q8.gemm(w, a, m, n, k, tiled=True), lambda: q8.gemm_residual(w, a, add, m, n, k), lambda: q8.gate_up_silu(w, w, a, m, n, k)]
    for call in forms:
        native, python = _both(monkeypatch, call)
        assert isinstance(native, np.ndarray) and native.dtype == python.dtype and native.shape == python.shape
        assert native.tobytes() == python.tobytes()
    assert q8._calls.mul_mat(w, x, n, k, None) is not None  # (and it was the native one)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 5, 40])
def test_plain_calls_are_native(q8, monkeypatch, m):
    # every function takes its plain call itself: with one that left it to Python, the comparison above would be of Python with itself
    n, k = 384, 1024
    w = q8.tile(q8.fill_weight_blocks(3, n, k), n, k)
    x, add, norm = q8.fill_activations(4, m * k).reshape(m, k), q8.fill_activations(5, m * n).reshape(m, n), q8.fill_activations(6, k)
    a = q8.quantize_row_q8_0(x, tiled=True)
    calls = q8._calls
    for out in (calls.mul_mat(w, x, n, k, None), calls.mul_mat(w, x, n, k, add), calls.gemm(w, a, m, n, k, None), calls.gemm(w, a, m, n, k, add), calls.rms_norm_quantize(x, norm, 1e-5), calls.gate_up_silu(w, w, a, m, n, k)):
        assert isinstance(out, torch.Tensor)

    def refuse(*args):
        raise AssertionError("the Python way")

    monkeypatch.setattr(q8_0._lib, "lib", refuse)  # ... and the wrappers hand it over
    for call in (lambda: q8.mul_mat(w, x, n, k), lambda: q8.mul_mat(w, x, n, k, residual=add), lambda: q8.gemm(w, a, m, n, k, tiled=True), lambda: q8.gemm_residual(w, a, add, m, n, k),
                 lambda: q8.rms_norm_quantize(x, norm, 1e-5, tiled=True), lambda: q8.gate_up_silu(w, w, a, m, n, k)):
        assert isinstance(call(), torch.Tensor)


@pytest.mark.gpu
def test_same_errors_either_way(q8, monkeypatch):
    n, k, m = 64, 256, 5
    w = q8.tile(q8.fill_weight_blocks(3, n, k), n, k)
    buf = q8.fill_activations(4, (m + 1) * k)
    x = buf[: m * k].reshape(m, k)
    a = q8.quantize_row_q8_0(x, tiled=True)
    refused = [lambda: q8.mul_mat(w, x, n, k + 128), lambda: q8.mul_mat(w[:-1], x, n, k), lambda: q8.mul_mat(w, x.t(), n, m), lambda: q8.mul_mat(w, x.half(), n, k), lambda: q8.mul_mat(w, x.cpu(), n, k),
               lambda: q8.mul_mat(w, buf[1 : 1 + m * k].reshape(m, k), n, k),  # not 16-byte aligned: the library's own status
               lambda: q8.mul_mat(w, x, n, 100), lambda: q8.mul_mat(w, x, -n, k), lambda: q8.mul_mat(w, x, n, k, residual=buf[:7]), lambda: q8.mul_mat(w, x, n, k, residual=buf[: m * n].double()),
               lambda: q8.gemm(w, a[:-1], m, n, k, tiled=True), lambda: q8.gemm_residual(w, a, buf[: m * n + 1], m, n, k), lambda: q8.gemm_residual(w, a, None, m, n, k),
               lambda: q8.rms_norm_quantize(x, buf[: k - 1], 1e-5, tiled=True), lambda: q8.rms_norm_quantize(x.reshape(1, m, k), buf[:k], 1e-5, tiled=True),
               lambda: q8.gate_up_silu(w, w, a, m, 100, k)]
    for i, call in enumerate(refused):
        native, python = _both(monkeypatch, call)
        assert isinstance(native, tuple), i
        assert native == python, i
    # tensors of a subclass, and modes that intercept torch's calls, go the Python way
    sub = x.as_subclass(_Subclass)
    assert q8._calls.mul_mat(w, sub, n, k, None) is None
    assert torch.equal(q8.mul_mat(w, sub, n, k).as_subclass(torch.Tensor), q8.mul_mat(w, x, n, k))
    from torch.utils._python_dispatch import TorchDispatchMode

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert q8._calls.mul_mat(w, x, n, k, None) is None
    with torch.device("cuda"):  # a torch-function mode
        assert q8._calls.mul_mat(w, x, n, k, None) is None
    # the output is on the weight's stream of work: a side stream's call is that stream's
    side = torch.cuda.Stream()
    want = q8.mul_mat(w, x, n, k)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = q8.mul_mat(w, x, n, k)
    side.synchronize()
    assert torch.equal(got, want)


@pytest.mark.gpu
def test_gate_up_operands_that_are_too_small_either_way(q8, monkeypatch):
    m, n_ff, k = 40, 256, 384
    w = q8.tile(q8.fill_weight_blocks(3, n_ff, k), n_ff, k)
    a = q8.quantize_row_q8_0(q8.fill_activations(4, m * k).reshape(m, k), tiled=True)
    for call in (lambda: q8.gate_up_silu(w[:-1], w, a, m, n_ff, k), lambda: q8.gate_up_silu(w, w[:-1], a, m, n_ff, k), lambda: q8.gate_up_silu(w, w, a[:-1], m, n_ff, k),
                 lambda: q8.gate_up_silu(w, w, a, m + 32, n_ff, k), lambda: q8.gate_up_silu(w, w, a, m, n_ff + 128, k), lambda: q8.gate_up_silu(w, w, a, m, n_ff, k + 128)):
        native, python = _both(monkeypatch, call)
        assert native == python and native[0] is ValueError
    native, python = _both(monkeypatch, lambda: q8.gate_up_silu(torch.cat([w, w]), w, torch.cat([a, w]), m, n_ff, k))  # larger buffers are taken
    assert native.tobytes() == python.tobytes() == q8.gate_up_silu(w, w, a, m, n_ff, k).cpu().numpy().tobytes()
