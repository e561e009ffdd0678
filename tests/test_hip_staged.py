"""
The channels-last kernel that stages contiguous tiles through LDS: parity with the CPU oracle at the edges of its
tiles (256 threads x 2 vectors; spans of at most 32 / element size - 1 steps), through the C ABI.
"""
import ctypes

import numpy as np
import pytest
import torch

import oracle
import scanscam_amd
from scanscam_amd import hip
from test_hip_channels_last import as_rows, prev_abs, rel_err

STAGED = hip.Plan(mode=hip.MODE_STAGED)
# fp32 chains differ from the oracle's by a few roundings per step that the gates (below 1) do not amplify; results of
# 16-bit storage by one rounding of the type, and the gate gradient by that of the stored output as well.
BAR = {torch.float32: 1e-5, torch.float64: 1e-13, torch.bfloat16: 1e-2, torch.float16: 2e-3}


def scan_pair(gpu, shape, dtype, plan, seed=0):
    g = torch.Generator().manual_seed(seed)
    wide = torch.float64 if dtype == torch.float64 else torch.float32
    a = torch.rand(shape, generator=g, dtype=wide).to(dtype)
    b, gh = (torch.randn(shape, generator=g, dtype=wide).to(dtype) for _ in range(2))
    da, db, dgh = a.to(gpu), b.to(gpu), gh.to(gpu)
    h = hip.transposed_linear_scan_forward(da, db, plan=plan)
    ga, gb = hip.transposed_linear_scan_backward(da, h, dgh, plan=plan)
    return (a, b, gh), (da, db, dgh), (h, ga, gb)


def check(inputs, results, dtype):
    a, b, gh = (as_rows(t) for t in inputs)
    h, ga, gb = (as_rows(t) for t in results)
    assert rel_err(h, oracle.fwd(a, b)) <= BAR[dtype]
    want_ga, want_gb = oracle.bwd(a, h, gh)
    assert rel_err(gb, want_gb) <= BAR[dtype]
    assert rel_err(ga, want_ga, prev_abs(h)) <= BAR[dtype]


def check_special_values(gpu, shape, dtype, plan, channels):
    """Infinities and NaN in one step each of some channels: the outputs that are no numbers are those of the recurrence, and
    all others as with numbers in their place. Gates of 0.95 and more: no product over the time steps is zero, which times an
    infinity is NaN where the recurrence stays infinite."""
    print(f"case special {dtype} {shape} {plan}", flush=True)
    g, T = torch.Generator().manual_seed(4), shape[1]
    a = (0.95 + 0.05 * torch.rand(shape, generator=g, dtype=torch.float64)).to(dtype)
    b, h, gh = (torch.randn(shape, generator=g, dtype=torch.float64).to(dtype) for _ in range(3))
    for i, c in enumerate(channels):
        value, t = (float("nan"), float("inf"), float("-inf"))[i % 3], (0, 1, T // 2, T - 2, T - 1)[i % 5]
        b[0, t, c] = gh[0, t, c] = value
        a[1, t, c] = float("nan")
        h[2, t, c] = value
    with np.errstate(invalid="ignore"):
        want_h, (want_ga, want_gb) = oracle.fwd(as_rows(a), as_rows(b)), oracle.bwd(as_rows(a), as_rows(h), as_rows(gh))
    got_h = hip.transposed_linear_scan_forward(a.to(gpu), b.to(gpu), plan=plan)
    got_ga, got_gb = hip.transposed_linear_scan_backward(a.to(gpu), h.to(gpu), gh.to(gpu), plan=plan)
    for got, want in ((got_h, want_h), (got_ga, want_ga), (got_gb, want_gb)):
        got = as_rows(got)
        numbers = np.isfinite(want)
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isfinite(got), numbers)
        assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
        floor = prev_abs(as_rows(h))[numbers] if want is want_ga else None
        # (gates near 1 add up the roundings of a thousand steps and more)
        assert rel_err(got[numbers], want[numbers], None if floor is None else np.where(np.isfinite(floor), floor, 1)) <= 4 * BAR[dtype]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", list(BAR))
@pytest.mark.parametrize("C", [2, 3, 17, 40, 91, 127, 129, 255, 256])
def test_edges_of_tiles_and_spans(gpu, dtype, C):
    esize = torch.empty(0, dtype=dtype).element_size()
    steps = 32 // esize - 1
    tile = min((256 * 2 * 16 - 16) // (C * esize), 256 // C * steps)  # the longest tile
    for T in sorted({2, steps, steps + 1, tile - 1, tile, tile + 1, 2 * tile + 1, 3 * tile + steps // 2}):
        if T < 2:
            continue
        print(f"case staged {dtype} C={C} T={T}", flush=True)
        inputs, _, results = scan_pair(gpu, (3, T, C), dtype, STAGED, seed=T)
        check(inputs, results, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", list(BAR))
@pytest.mark.parametrize("C", [2, 24, 64, 91, 129, 256])
def test_time_in_parts(gpu, dtype, C):
    """Two launches: the parts' pairs, then every part from the pairs before it. Parts of one and of several tiles, the
    last one short, more parts than tiles, and as many as the runs of threads that fold the pairs do not divide."""
    esize = torch.empty(0, dtype=dtype).element_size()
    tile = min((256 * 2 * 16 - 16) // (C * esize), 256 // C * (32 // esize - 1))
    for T, parts in ((tile + 1, 2), (5 * tile + 3, 2), (5 * tile + 3, 5), (7 * tile, 64), (67 * tile + 1, 66)):
        print(f"case staged in parts {dtype} C={C} T={T} parts={parts}", flush=True)
        inputs, _, results = scan_pair(gpu, (2, T, C), dtype, hip.Plan(mode=hip.MODE_STAGED, unroll=parts), seed=T)
        check(inputs, results, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,shape", [(torch.bfloat16, (250, 1000, 39)), (torch.float32, (3, 4000, 40))])
def test_a_short_workspace_leaves_the_other_kernels(gpu, dtype, shape):
    """A workspace below the size asked for is no error where the plan in reserve, a walk or tiles, can do with it."""
    code, L = hip._dtype_code(dtype), hip.lib()
    _, (a, b, gh), (h, ga, gb) = scan_pair(gpu, shape, dtype, None)
    stream = torch.cuda.current_stream().cuda_stream
    for direction in (hip.FORWARD, hip.BACKWARD):
        other = hip.resolve_plan_cl(*shape, dtype, direction)
        assert other.waves_per_row > 1
        other.waves_per_row = 0
        need = hip.workspace_bytes_cl(*shape, dtype, direction, other)
        assert need < hip.workspace_bytes_cl(*shape, dtype, direction)
        ws = torch.empty(max(need, 8), dtype=torch.uint8, device=gpu)
        x, y = torch.empty_like(a), torch.empty_like(a)
        if direction == hip.FORWARD:
            rc = L.scanscam_scan_fwd_cl(a.data_ptr(), b.data_ptr(), x.data_ptr(), *shape, code, ws.data_ptr(), need, stream, None)
            got, auto = (x,), (h,)
            want = (hip.transposed_linear_scan_forward(a, b, plan=other),)
        else:
            rc = L.scanscam_scan_bwd_cl(a.data_ptr(), h.data_ptr(), gh.data_ptr(), x.data_ptr(), y.data_ptr(), *shape, code,
                                        ws.data_ptr(), need, stream, None)
            got, auto = (x, y), (ga, gb)
            want = hip.transposed_linear_scan_backward(a, h, gh, plan=other)
        assert rc == 0
        for g, w, s in zip(got, want, auto):
            assert torch.equal(g, w) and rel_err(as_rows(g), as_rows(s)) <= BAR[dtype]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,shape", [(torch.float32, (600, 333, 33)), (torch.bfloat16, (2048, 167, 40)),
                                         (torch.float16, (513, 400, 19)), (torch.float64, (520, 70, 130)),
                                         (torch.float32, (512, 512, 12)), (torch.float32, (14, 2000, 24)),
                                         (torch.bfloat16, (100, 1100, 33)), (torch.float64, (1, 30000, 8)),
                                         (torch.float16, (150, 1700, 37))])
def test_automatic_route(gpu, dtype, shape):
    """Calls whose automatic plan is this kernel give its very results, and agree with the other kernels."""
    inputs, device, results = scan_pair(gpu, shape, dtype, None)
    plans = [hip.resolve_plan_cl(*shape, dtype, d) for d in (hip.FORWARD, hip.BACKWARD)]
    assert plans[0].waves_per_row == plans[1].waves_per_row > 0
    staged = hip.Plan(mode=hip.MODE_STAGED, unroll=plans[0].waves_per_row)
    _, _, forced = scan_pair(gpu, shape, dtype, staged)
    ga, gb = hip.transposed_linear_scan_backward(device[0], results[0], device[2], plan=plans[1])
    resolved = (hip.transposed_linear_scan_forward(device[0], device[1], plan=plans[0]), ga, gb)
    for x, y, z in zip(results, forced, resolved):
        assert torch.equal(x, y) and torch.equal(x, z)
    few = [t[:7].contiguous() for t in inputs]
    check(few, [t[:7] for t in results], dtype)
    other = plans[0]
    other.waves_per_row = 0
    h = hip.transposed_linear_scan_forward(device[0], device[1], plan=other)
    assert rel_err(as_rows(results[0]), as_rows(h)) <= BAR[dtype] and not torch.equal(h, results[0])
    # An output in place of an input, and bases off the 16-byte border (which this kernel leaves to the others).
    L, code = hip.lib(), hip._dtype_code(dtype)
    ws = torch.empty(max(8, hip.workspace_bytes_cl(*shape, dtype)), dtype=torch.uint8, device=gpu)
    stream = torch.cuda.current_stream().cuda_stream
    b = device[1].clone()
    assert L.scanscam_scan_fwd_cl(device[0].data_ptr(), b.data_ptr(), b.data_ptr(), *shape, code, ws.data_ptr(), ws.numel(),
                                  stream, None) == 0
    assert torch.equal(b, results[0])
    off = torch.empty(b.numel() + 1, dtype=dtype, device=gpu)[1:].view(shape)
    off.copy_(device[1])
    h = hip.transposed_linear_scan_forward(device[0], off)
    assert not torch.equal(h, results[0]) and rel_err(as_rows(results[0]), as_rows(h)) <= BAR[dtype]
    with pytest.raises(RuntimeError):
        hip.transposed_linear_scan_forward(device[0], off, plan=staged)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", list(BAR))
@pytest.mark.parametrize("C,parts", [(2, 16), (8, 0), (8, 3), (24, 40), (130, 9)])
def test_growing_gates_over_a_zero_carry_in_parts(gpu, dtype, C, parts):
    """Gates of 1.5 over 3000 steps of zeros: their product is beyond every type (2 ** 1754), the recurrence stays zero."""
    plan = hip.Plan(mode=hip.MODE_STAGED, unroll=parts) if parts else None
    T, grown = 12000, 3000
    g = torch.Generator().manual_seed(C)
    wide = torch.float64 if dtype == torch.float64 else torch.float32
    a = torch.rand((1, T, C), generator=g, dtype=wide).to(dtype)
    b, h, gh = (torch.randn((1, T, C), generator=g, dtype=wide).to(dtype) for _ in range(3))
    a[:, :grown], b[:, :grown] = 1.5, 0
    print(f"case growing gates {dtype} C={C} parts={parts}", flush=True)
    got = hip.transposed_linear_scan_forward(a.to(gpu), b.to(gpu), plan=plan)
    assert rel_err(as_rows(got), oracle.fwd(as_rows(a), as_rows(b))) <= BAR[dtype]
    # Backwards: the gates of the last steps, under no gradient.
    a, gh = a.flip(1).contiguous(), gh.clone()
    gh[:, -grown:] = 0
    ga, gb = hip.transposed_linear_scan_backward(a.to(gpu), h.to(gpu), gh.to(gpu), plan=plan)
    want_ga, want_gb = oracle.bwd(as_rows(a), as_rows(h), as_rows(gh))
    assert rel_err(as_rows(gb), want_gb) <= BAR[dtype]
    assert rel_err(as_rows(ga), want_ga, prev_abs(as_rows(h))) <= BAR[dtype]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_small_carry_through_a_part_that_grows_and_shrinks(gpu, dtype):
    """2 ** -100, doubled 160 times and halved again inside every part: powers of two throughout, so nothing rounds."""
    T, C = 6400, 24
    a, b = torch.ones((1, T, C), dtype=dtype), torch.zeros((1, T, C), dtype=dtype)
    for t in range(100, T - 400, 400):
        a[:, t:t + 160], a[:, t + 160:t + 320] = 2.0, 0.5
    b[:, 0] = 2.0 ** -100
    want = torch.cumprod(a.double(), 1) * 2.0 ** -100
    for parts in (2, 5, 100):
        got = hip.transposed_linear_scan_forward(a.to(gpu), b.to(gpu), plan=hip.Plan(mode=hip.MODE_STAGED, unroll=parts))
        assert torch.equal(got.cpu().double(), want), parts


# In parts in both directions; in one launch beside a look-back workspace in reserve (backwards), and without any.
FLAG_SHAPES = [(torch.float32, (14, 2000, 24)), (torch.float64, (1, 30000, 8)), (torch.bfloat16, (100, 1100, 33)),
               (torch.float16, (1, 4000, 5)), (torch.float32, (600, 333, 33)), (torch.bfloat16, (2048, 167, 40))]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,shape", FLAG_SHAPES)
def test_no_expired_wait_is_reported(gpu, dtype, shape):
    """This kernel waits for no other workgroup: whatever the workspace held before, its flag says so after the call."""
    inputs, (a, b, gh), _ = scan_pair(gpu, shape, dtype, None)
    L, code, stream = hip.lib(), hip._dtype_code(dtype), torch.cuda.current_stream().cuda_stream
    h, g0, g1 = (torch.empty_like(a) for _ in range(3))
    for direction in (hip.FORWARD, hip.BACKWARD):
        need = max(16, hip.workspace_bytes_cl(*shape, dtype, direction))
        ws = torch.full((need,), 255, dtype=torch.uint8, device=gpu)
        print(f"case flag {dtype} {shape} direction={direction} workspace={need}", flush=True)
        if direction == hip.FORWARD:
            rc = L.scanscam_scan_fwd_cl(a.data_ptr(), b.data_ptr(), h.data_ptr(), *shape, code, ws.data_ptr(), need, stream, None)
        else:
            rc = L.scanscam_scan_bwd_cl(a.data_ptr(), h.data_ptr(), gh.data_ptr(), g0.data_ptr(), g1.data_ptr(), *shape, code,
                                        ws.data_ptr(), need, stream, None)
        assert rc == 0
        flag = ctypes.c_int(-1)
        assert L.scanscam_workspace_timed_out(ws.data_ptr(), stream, ctypes.byref(flag)) == 0 and flag.value == 0
    check([t[:2].contiguous() for t in inputs], [t[:2] for t in (h, g0, g1)], dtype)
    # The same through the op, with checking on; the allocator hands it memory that held something.
    hip.check_waits(True)
    try:
        x, y = a.mT.requires_grad_(), b.mT.requires_grad_()
        torch.full((hip.workspace_bytes_cl(*shape, dtype),), 255, dtype=torch.uint8, device=gpu)
        out = scanscam_amd.scan(x, y)
        grads = torch.autograd.grad(out, (x, y), gh.mT)
    finally:
        hip.check_waits(False)
    for got, want in zip((out, *grads), (h, g0, g1)):
        assert torch.equal(got.mT, want)


@pytest.mark.gpu
@pytest.mark.parametrize("parts", [1, 6])
def test_nonfinite_values_stay_in_their_channel_and_batch_element(gpu, parts):
    shape, plan = (3, 700, 33), hip.Plan(mode=hip.MODE_STAGED, unroll=parts)
    (a, b, gh), _, clean = scan_pair(gpu, shape, torch.float32, plan)
    b[1, 350, 7] = np.nan
    a, b, gh = a.to(gpu), b.to(gpu), gh.to(gpu)
    h = hip.transposed_linear_scan_forward(a, b, plan=plan)
    hit = torch.zeros(shape, dtype=torch.bool)
    hit[1, 350:, 7] = True
    assert torch.equal(torch.isnan(h).cpu(), hit)
    assert torch.equal(h.cpu()[~hit], clean[0].cpu()[~hit])


def test_only_channels_last_calls_take_it():
    with pytest.raises(RuntimeError):
        hip.resolve_plan(64, 4096, torch.float32, hip.FORWARD, STAGED)
    with pytest.raises(RuntimeError):
        hip.resolve_plan_cl(64, 4096, 40, torch.float32, hip.FORWARD, STAGED)


def test_a_resolved_plan_says_what_runs():
    """What scanscam_resolve_plan_cl reports holds the staged kernel's parts as well; it resolves to itself, also in place,
    and asks for the automatic call's workspace; without the parts it is the plan in reserve."""
    L, staged = hip.lib(), 0
    for dtype in BAR:
        code = hip._dtype_code(dtype)
        for batch, T, C in ((14, 2000, 24), (1, 30000, 8), (600, 333, 33), (2048, 512, 40), (200, 9000, 37), (8, 4096, 512),
                            (64, 2048, 1001), (1, 4000, 64), (90, 700, 257)):
            for direction in (hip.FORWARD, hip.BACKWARD):
                plan, again, reserve = hip.resolve_plan_cl(batch, T, C, dtype, direction), hip.Plan(), hip.Plan()
                staged += plan.waves_per_row > 0
                need = hip.workspace_bytes_cl(batch, T, C, dtype, direction)
                assert hip.workspace_bytes_cl(batch, T, C, dtype, direction, plan) <= need
                ctypes.memmove(ctypes.byref(again), ctypes.byref(plan), ctypes.sizeof(hip.Plan))
                ref = ctypes.byref(again)
                assert L.scanscam_resolve_plan_cl(batch, T, C, code, direction, ref, ref) == 0
                assert bytes(again) == bytes(plan)
                ctypes.memmove(ctypes.byref(reserve), ctypes.byref(plan), ctypes.sizeof(hip.Plan))
                reserve.waves_per_row = 0
                back = hip.resolve_plan_cl(batch, T, C, dtype, direction, reserve)
                assert bytes(back) == bytes(reserve)
    assert staged >= 20


@pytest.mark.parametrize("dtype,takes,leaves", [
    (torch.float32, [(1000, 1023, 17), (851, 467, 27), (435, 988, 5), (14, 13990, 24), (1, 1000000, 2), (6, 607, 51)],
     [(435, 988, 3), (423, 115, 30), (12, 95, 61), (4, 5315, 2), (2, 982, 5), (512, 4096, 8), (192, 2000, 33)]),
    (torch.bfloat16, [(2048, 512, 40), (1000, 1023, 17), (39, 11559, 30), (2, 39951, 2), (250, 1000, 39), (2129, 1365, 8)],
     [(506, 4528, 2), (338, 2002, 4), (255, 54672, 2), (242, 68888, 8), (687, 483, 8), (11, 188, 53), (8, 723, 23), (1, 7948, 2)]),
    (torch.float64, [(1000, 1023, 17), (1024, 90, 130), (3, 200000, 24), (4, 222, 62)],
     [(463, 14524, 3), (343, 8902, 5), (665, 246, 7), (14, 4134, 38)])])
def test_calls_that_take_it_and_calls_that_do_not(dtype, takes, leaves):
    """Both sides of the automatic choice, each shape measured against the plan in reserve."""
    parts = lambda s: [hip.resolve_plan_cl(*s, dtype, d).waves_per_row for d in (hip.FORWARD, hip.BACKWARD)]  # noqa: E731
    assert all(p > 0 for s in takes for p in parts(s)), [s for s in takes if min(parts(s)) == 0]
    assert all(p == 0 for s in leaves for p in parts(s)), [s for s in leaves if max(parts(s)) > 0]


def test_forced_plans_that_it_refuses():
    """Refused before anything is launched, so made-up pointers will do: fields it has no use for, more threads than one
    launch can have, more channels than a workgroup has threads, bases off the 16-byte border."""
    L = hip.lib()

    def call(plan, batch=4, T=100, C=8, base=4096):
        return L.scanscam_scan_fwd_cl(base, base, base, batch, T, C, 0, None, 0, None, ctypes.byref(plan))

    refused = [call(hip.Plan(mode=hip.MODE_STAGED, vec=1)), call(hip.Plan(mode=hip.MODE_STAGED, waves=4)),
               call(hip.Plan(mode=hip.MODE_STAGED, waves_per_row=2)), call(hip.Plan(mode=hip.MODE_STAGED, unroll=-1)),
               call(STAGED, C=257), call(STAGED, base=4100), call(STAGED, batch=1 << 24, T=1, C=1)]
    assert refused == [4] * len(refused)
    assert call(hip.Plan(mode=hip.MODE_STAGED, unroll=4), T=10000) == 5  # in parts: a workspace
