"""
The native host path of the op (csrc/torch_binding.cpp) against the Python path it stands in for: the same results in the
same layout for every form it takes, and the same outcome for every form it leaves alone.
"""
import os
import subprocess
import threading

import pytest
import torch

from scanscam_amd import hip, scan


def python_path(monkeypatch, fn, *args):
    with monkeypatch.context() as m:
        m.setattr(hip, "_native", None)
        return fn(*args)


def forms(dev, dtype):
    """(name, gate, value, output gradient) of one logical shape each."""
    g = torch.Generator(device=dev).manual_seed(3)
    new = lambda *shape: torch.rand(shape, generator=g, device=dev).to(dtype)  # noqa: E731
    rows = lambda: new(4, 6, 50)  # noqa: E731
    cl = lambda: new(4, 50, 6).mT  # noqa: E731
    yield "rows", rows(), rows(), rows()
    yield "2-D", new(7, 33), new(7, 33), new(7, 33)
    yield "4-D", new(2, 3, 4, 33), new(2, 3, 4, 33), new(2, 3, 4, 33)
    yield "halves of a projection", *new(4, 12, 50).chunk(2, 1), rows()
    yield "slices of longer rows", new(4, 6, 60)[..., 3:53], new(4, 6, 60)[..., 7:57], rows()
    yield "leading dimensions swapped", new(6, 4, 50).transpose(0, 1), rows(), new(6, 4, 50).transpose(0, 1)
    yield "three levels", new(2, 3, 5, 4, 20)[:, :, ::2].transpose(0, 3), new(4, 3, 3, 2, 20), new(4, 3, 3, 2, 20)
    yield "gate broadcast over the batch", new(1, 6, 50).expand(4, 6, 50), rows(), rows()
    yield "scan dimension strided", new(4, 6, 100)[..., ::2], rows(), rows()
    yield "output gradient expanded", rows(), rows(), new(1, 1, 1).expand(4, 6, 50)
    yield "channels-last", cl(), cl(), cl()
    yield "channels-last halves", *(t.mT for t in new(4, 50, 12).chunk(2, 2)), cl()
    yield "channels-last 4-D", new(2, 2, 50, 6).mT, new(2, 2, 50, 6).mT, new(2, 2, 50, 6).mT
    yield "channels-last batch strided twice", new(2, 4, 50, 6)[:, ::2].mT, new(2, 2, 50, 6).mT, new(2, 2, 50, 6).mT
    yield "channels-last, gradient in rows", cl(), cl(), rows()
    yield "layouts mixed", cl(), rows(), cl()
    yield "T of 1", new(4, 6, 1), new(4, 6, 1), new(4, 6, 1)
    yield "one channel", new(4, 50, 1).mT, new(4, 50, 1).mT, new(4, 50, 1).mT
    yield "empty", new(0, 6, 50), new(0, 6, 50), new(0, 6, 50)
    yield "workspace", new(2, 70000), new(2, 70000), new(2, 70000)
    yield "channels-last workspace", new(1, 4000, 64).mT, new(1, 4000, 64).mT, new(1, 4000, 64).mT
    yield "channels-last staged in parts", new(14, 2000, 24).mT, new(14, 2000, 24).mT, new(14, 2000, 24).mT
    yield "channels-last staged", new(600, 333, 33).mT, new(600, 333, 33).mT, new(600, 333, 33).mT
    if dtype != torch.float64:
        yield "off the vector border", rows().flatten()[1:1 + 4 * 6 * 49].view(4, 6, 49), new(4, 6, 49), new(4, 6, 49)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16, torch.float64])
def test_same_results_and_layout_as_the_python_path(gpu, dtype, monkeypatch):
    assert hip._native is not None
    taken = 0
    for name, a, b, gh in forms(gpu, dtype):
        print(f"case {name} {dtype}", flush=True)
        h = hip.scan_forward(a, b)
        grads = hip.scan_backward(a, h, gh)
        want_h = python_path(monkeypatch, hip.scan_forward, a, b)
        want = python_path(monkeypatch, hip.scan_backward, a, want_h, gh)
        for x, y in zip((h, *grads), (want_h, *want)):
            assert torch.equal(x, y) and x.stride() == y.stride() and x.dtype == y.dtype, name
        taken += hip._native.forward(a, b) is not None
    assert taken >= 15


@pytest.mark.gpu
def test_left_to_the_python_path(gpu, monkeypatch):
    a, b = torch.rand(4, 50, device=gpu), torch.rand(4, 50, device=gpu)

    class Sub(torch.Tensor):
        pass

    left = [(a.as_subclass(Sub), b), (a, b.cpu()), (a, b.double()), (a.int(), b.int()), (a, b[:, :49]), (a[0], b[0]), (a, None)]
    for args in left:
        assert hip._native.forward(*args) is None
        outcomes = []
        for native in (True, False):
            try:
                outcomes.append(hip.scan_forward(*args) if native else python_path(monkeypatch, hip.scan_forward, *args))
            except Exception as e:  # noqa: BLE001
                outcomes.append((type(e), str(e)))
        if isinstance(outcomes[0], tuple):
            assert outcomes[0] == outcomes[1]
        else:
            assert torch.equal(outcomes[0], outcomes[1])
    assert hip._native.forward(a) is None
    with pytest.raises(RuntimeError):
        torch.func.vmap(hip.scan_forward)(a[None], b[None])
    # With checking of waits on, the native path is not entered at all.
    class Untouched:
        def forward(self, *args):
            raise AssertionError("the native path was entered")

        backward = forward

    want = hip.scan_forward(a, b)
    with monkeypatch.context() as m:
        m.setattr(hip, "_native", Untouched())
        with pytest.raises(AssertionError, match="native path"):
            hip.scan_forward(a, b)
        hip.check_waits(True)
        try:
            assert torch.equal(hip.scan_forward(a, b), want)
            grads = hip.scan_backward(a, want, b)
        finally:
            hip.check_waits(False)
    for x, y in zip(grads, hip.scan_backward(a, want, b)):
        assert torch.equal(x, y)
    # Tensors a hook hands back.
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.to(gpu)):
        x, y = a.clone().requires_grad_(), b.clone().requires_grad_()
        h = scan(x, y)
    h.sum().backward()
    want = hip.scan_backward(a, h.detach(), torch.ones_like(a))
    assert torch.equal(x.grad, want[0]) and torch.equal(y.grad, want[1])


@pytest.mark.gpu
def test_modes_are_left_to_the_python_path(gpu, monkeypatch):
    """Under a function or a dispatch mode the calls go where the mode sees what the Python path does."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(getattr(func, "__name__", str(func)))
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    a, b = torch.rand(4, 50, device=gpu), torch.rand(4, 50, device=gpu)
    want = hip.scan_forward(a, b)
    for mode in (Functions, Dispatch):
        seen = []
        with mode():
            assert hip._native.forward(a, b) is None and hip._native.backward(a, b, b) is None
            del seen[:]
            got, calls = hip.scan_forward(a, b), list(seen)
            del seen[:]
            python_path(monkeypatch, hip.scan_forward, a, b)
            assert calls == seen and len(calls) > 0
        assert torch.equal(got, want)


@pytest.mark.gpu
def test_streams_and_threads(gpu):
    """Each thread on a stream of its own, with look-back workspaces; every result as on the default stream."""
    cases = [(torch.rand(2, 70000 + 64 * i, device=gpu), torch.rand(2, 70000 + 64 * i, device=gpu)) for i in range(4)]
    want = [hip.scan_forward(*c) for c in cases]
    torch.cuda.synchronize()
    wrong = []

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(20):
                got = hip.scan_forward(*cases[i])
                s.synchronize()
                if not torch.equal(got, want[i]):
                    wrong.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_declines_what_is_not_on_a_gpu():
    if hip._native is None:
        pytest.skip("the binding is not built")
    a = torch.rand(3, 4)
    assert hip._native.forward(a, a) is None and hip._native.backward(a, a, a) is None
    assert hip._native.forward(1, 2) is None


def test_a_binding_of_another_pytorch_is_not_used(monkeypatch):
    assert hip._bind_native(hip.lib()) is not None
    with monkeypatch.context() as m:
        m.setattr(torch, "__version__", "0.0")
        with pytest.warns(RuntimeWarning, match="built against PyTorch"):
            assert hip._bind_native(hip.lib()) is None


def test_the_c_libraries_build_without_python():
    """`make` alone names neither PyTorch nor a Python, only the compilers."""
    csrc = os.path.join(os.path.dirname(os.path.abspath(hip.__file__)), "csrc")
    done = subprocess.run(["make", "-C", csrc, "-n", "-B", "PYTHON=/nonexistent/python"], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stderr
    assert "libscanscam_hip.so" in done.stdout and "libscanscam_cpu.so" in done.stdout and "torch" not in done.stdout
