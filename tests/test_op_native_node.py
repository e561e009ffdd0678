"""
The op's native autograd node (csrc/torch_binding.cpp) against the Python function it stands in for: the same gradients, and
the same outcome of everything the engine, hooks and modes do to a node.
"""
import ctypes
import threading

import pytest
import torch

from scanscam_amd import hip, op, scan
from test_binding import forms


def leaves(*tensors):
    return [t.detach().requires_grad_() for t in tensors]


def is_native(h):
    return h.grad_fn is not None and not isinstance(h.grad_fn, torch.autograd.function.BackwardCFunction)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16, torch.float64])
def test_same_gradients_as_the_python_function(gpu, dtype):
    native = 0
    for name, a, b, gh in forms(gpu, dtype):
        print(f"case {name} {dtype}", flush=True)
        results = []
        for fn in (scan, op.Scan.apply):
            x, y = leaves(a, b)
            h = fn(x, y)
            native += is_native(h)
            results.append((h.detach(), *torch.autograd.grad(h, (x, y), gh)))
        for got, want in zip(*results):
            assert torch.equal(got, want) and got.stride() == want.stride() and got.dtype == want.dtype, name
        for mask in ((True, False), (False, True)):
            x, y = a.detach().requires_grad_(mask[0]), b.detach().requires_grad_(mask[1])
            scan(x, y).backward(gh)
            for leaf, want, on in zip((x, y), results[0][1:], mask):
                assert (leaf.grad is None) if not on else torch.equal(leaf.grad, want)
    assert native >= 15


def outcome(fn):
    """("values", the tensors' values) or ("raises", type and message); a test's own assertions are not an outcome."""
    try:
        r = fn()
        return "values", tuple(t.cpu().tolist() for t in r) if isinstance(r, tuple) else r
    except AssertionError:
        raise
    except Exception as e:  # noqa: BLE001
        return "raises", type(e), str(e).split("\n")[0][:60]


@pytest.mark.gpu
def test_same_outcomes_as_the_python_function(gpu):
    g = torch.Generator(device=gpu).manual_seed(5)
    a, b, gh = (torch.rand(4, 50, generator=g, device=gpu) for _ in range(3))

    def twice(fn, retain):
        x, y = leaves(a, b)
        h = fn(x, y)
        torch.autograd.grad(h, (x, y), gh, retain_graph=retain)
        return torch.autograd.grad(h, (x, y), gh)

    def changed(fn, which):
        x, y = leaves(a, b)
        x1 = x * 1
        h = fn(x1, y)
        with torch.no_grad():
            (x1 if which == 0 else h).add_(1)
        return torch.autograd.grad(h, (x, y), gh)

    def second_order(fn):
        x, y = leaves(a, b)
        ga, _ = torch.autograd.grad(fn(x, y), (x, y), gh, create_graph=True)
        return torch.autograd.grad(ga.sum(), (x,))

    def saved_elsewhere(fn):
        seen = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(t.shape), t.cpu())[1], lambda t: t.to(gpu)):
            x, y = leaves(a, b)
            h = fn(x, y)
        assert len(seen) == 2
        return torch.autograd.grad(h, (x, y), gh)

    def left_on_the_cpu(fn):  # an error in both: the output gradient is on the GPU
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t):
            x, y = leaves(a, b)
            h = fn(x, y)
        return torch.autograd.grad(h, (x, y), gh)

    def hooked(fn):
        x, y = leaves(a, b)
        h = fn(x, y)
        h.register_hook(lambda t: 2 * t)
        h.grad_fn.register_hook(lambda gin, gout: (gin[0] + 1, gin[1]))
        return torch.autograd.grad(h, (x, y), gh)

    def checkpointed(fn):
        x, y = leaves(a, b)
        return torch.autograd.grad(torch.utils.checkpoint.checkpoint(fn, x, y, use_reentrant=False), (x, y), gh)

    def checked(fn):  # switched on between the two passes
        x, y = leaves(a, b)
        h = fn(x, y)
        hip.check_waits(True)
        try:
            return torch.autograd.grad(h, (x, y), gh)
        finally:
            hip.check_waits(False)

    def vmapped(fn):
        return torch.func.vmap(fn)(a[None], b[None])

    def inside_a_transform(fn):
        return torch.func.grad(lambda t: t.sum() + fn(a, b).sum())(a)

    def dual(fn):
        with torch.autograd.forward_ad.dual_level():
            return fn(torch.autograd.forward_ad.make_dual(a, b), b)

    def unused(fn):  # no gradient reaches the output of the inner call
        x, y = leaves(a, b)
        h = fn(x, y)
        return torch.autograd.grad((h * 0).sum() + x.sum(), (x, y))

    def grads_off(fn):
        x, y = leaves(a, b)
        with torch.no_grad():
            h = fn(x, y)
        with torch.inference_mode():
            i = fn(x, y)
        return h.requires_grad, h.grad_fn, i.is_inference(), h.is_inference()

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    def under_a_mode(fn):
        x, y = leaves(a, b)
        with Mode():
            h = fn(x, y)
            assert not is_native(h)
            return torch.autograd.grad(h, (x, y), gh)

    calls = {"values": [lambda f: twice(f, True), saved_elsewhere, hooked, checkpointed, checked, unused, under_a_mode],
             "raises": [lambda f: twice(f, False), lambda f: changed(f, 0), lambda f: changed(f, 1), second_order, left_on_the_cpu,
                        vmapped, inside_a_transform, dual]}
    for kind, cases in calls.items():
        for i, call in enumerate(cases):
            got, want = outcome(lambda: call(scan)), outcome(lambda: call(op.Scan.apply))
            assert got[0] == want[0] == kind, (kind, i, got[:2] if got[0] == "raises" else "", want[:2] if want[0] == "raises" else "")
            assert got == want, (kind, i, got if kind == "raises" else "values", want if kind == "raises" else "values")
    assert grads_off(scan) == grads_off(op.Scan.apply)
    assert is_native(scan(*leaves(a, b)))


@pytest.mark.gpu
def test_the_node_shows_what_the_python_function_s_shows(gpu):
    """Name, saved tensors and which inputs need gradients; what a profile calls the two passes."""
    a, b, gh = (torch.rand(4, 50, device=gpu) for _ in range(3))
    for mask in ((True, True), (True, False), (False, True)):
        seen = []
        for fn in (scan, op.Scan.apply):
            x, y = a.detach().requires_grad_(mask[0]), b.detach().requires_grad_(mask[1])
            h = fn(x, y)
            node = h.grad_fn
            gate, output = node.saved_tensors
            assert gate is x and torch.equal(output, h) and output.grad_fn is node
            assert isinstance(node, torch.autograd.graph.Node) and repr(h).endswith("grad_fn=<ScanBackward>)")
            edges = [None if n is None else type(n).__name__ for n, _ in node.next_functions]
            shown = [type(node).__name__, node.name(), node.needs_input_grad, node.metadata, edges]
            h.backward(gh)
            with pytest.raises(RuntimeError, match="second time"):
                node.saved_tensors
            seen.append(shown)
        assert seen[0] == seen[1]
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.to(gpu)):
        h = scan(*leaves(a, b))
    assert is_native(h) and all(t.is_cuda for t in h.grad_fn.saved_tensors)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as profile:
        x, y = leaves(a, b)
        torch.autograd.grad(scan(x, y), (x, y), gh)
    assert {"Scan", "ScanBackward"} <= {e.name for e in profile.events()}


def test_calls_left_to_python_are_profiled_once():
    x, y = (torch.rand(4, 50, requires_grad=True) for _ in range(2))
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as profile:
        scan(x, y).sum().backward()
    names = [e.name for e in profile.events()]
    assert names.count("Scan") == 1 and names.count("ScanBackward") == 1


@pytest.mark.gpu
def test_compiled_autograd(gpu):
    """A backward pass that is traced into a graph calls the node as it is."""
    from torch._dynamo import compiled_autograd

    a, b, gh = (torch.rand(4, 50, device=gpu) for _ in range(3))
    results = []
    for fn in (scan, op.Scan.apply):
        torch._dynamo.reset()
        x, y = leaves(a, b)
        h = fn(x, y)
        with compiled_autograd._enable(torch.compile(backend="eager")):
            h.backward(gh)
        results.append((x.grad, y.grad))
    assert all(torch.equal(p, q) for p, q in zip(*results))


@pytest.mark.gpu
def test_errors_on_the_engine_s_thread(gpu):
    """The library's errors, and memory that cannot be had, in a backward pass: exceptions of the caller, as the Python function
    raises them; the next pass works."""
    a, b, gh = (torch.rand(4, 50, device=gpu) for _ in range(3))
    lib = hip.lib()
    names = ["scan_fwd_strided", "scan_bwd_strided", "scan_fwd_cl_strided", "scan_bwd_cl_strided", "workspace_bytes",
             "workspace_bytes_cl", "strerror"]
    entries = [ctypes.cast(getattr(lib, f"scanscam_{n}"), ctypes.c_void_p).value for n in names]
    refuse = ctypes.CFUNCTYPE(ctypes.c_int)(lambda: 1)  # an error code for every call
    x, y = leaves(a, b)
    h = scan(x, y)
    try:
        hip._native.bind(entries[0], ctypes.cast(refuse, ctypes.c_void_p).value, *entries[2:], hip._backward_in_python)
        with pytest.raises(RuntimeError) as raised:
            torch.autograd.grad(h, (x, y), gh, retain_graph=True)
    finally:
        hip._native.bind(*entries, hip._backward_in_python)
    assert str(raised.value).startswith(f"scanscam_scan_bwd_strided: {hip.strerror(1)}")
    want = torch.autograd.grad(op.Scan.apply(x, y), (x, y), gh)
    assert all(torch.equal(p, q) for p, q in zip(torch.autograd.grad(h, (x, y), gh), want))

    x, y = (torch.rand(64, 1 << 20, device=gpu).requires_grad_() for _ in range(2))
    steps = [(fn(x, y), torch.rand_like(x)) for fn in (scan, op.Scan.apply)]
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (64 << 20)) / total)
    try:
        for h, g in steps:
            with pytest.raises(torch.OutOfMemoryError):
                torch.autograd.grad(h, (x, y), g)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    x, y = leaves(a, b)
    assert all(torch.equal(p, q) for p, q in zip(torch.autograd.grad(scan(x, y), (x, y), gh), want))


@pytest.mark.gpu
def test_threads_and_streams(gpu):
    """Steps of several threads, each on a stream of its own."""
    g = torch.Generator(device=gpu).manual_seed(6)
    sets = [[torch.rand(8, 64, 4096, generator=g, device=gpu) for _ in range(3)] for _ in range(4)]
    want = []
    for a, b, gh in sets:
        x, y = leaves(a, b)
        want.append(torch.autograd.grad(op.Scan.apply(x, y), (x, y), gh))
    torch.cuda.synchronize()
    bad = []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(5):
                    x, y = leaves(*sets[i][:2])
                    got = torch.autograd.grad(scan(x, y), (x, y), sets[i][2])
                    torch.cuda.current_stream().synchronize()
                    if not all(torch.equal(p, q) for p, q in zip(got, want[i])):
                        bad.append(i)
        except BaseException as e:  # noqa: BLE001
            bad.append((i, e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
