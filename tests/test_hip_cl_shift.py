"""
Channels-last calls of odd channel counts whose channels move between neighbouring lanes: parity with the CPU oracle at
the edges of its groups (63 vectors of 4 channels, 2 in float64), spans and tiles, and its route.
"""
import os
import random
import shutil
import subprocess

import pytest
import torch

import oracle
from scanscam_amd import hip
from test_hip_channels_last import as_rows, prev_abs, rel_err
from test_hip_staged import BAR, check, check_special_values, scan_pair


def forced(steps, waves, tiles):
    return hip.Plan(waves_per_row=-(64 * steps + 2 * waves + tiles))


def runs(dtype, steps, waves, tiles, T):
    """Whether these lanes are built for the launch: 16 steps only for 16-bit types, and only in tiles, two of them at least
    (the tiles start up to a vector's channels in steps early)."""
    vec = 2 if dtype == torch.float64 else 4
    return steps < 16 or (dtype in (torch.bfloat16, torch.float16) and tiles == 1 and T + vec - 1 > steps * waves)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", list(BAR))
@pytest.mark.parametrize("steps,waves,tiles", [(4, 1, 0), (4, 3, 0), (8, 8, 0), (4, 2, 1), (8, 8, 1), (16, 4, 1), (16, 8, 1), (8, 4, 1), (4, 8, 1)])
def test_edges_of_groups_and_spans(gpu, dtype, steps, waves, tiles):
    """Either odd remainder of C, a last group of two vectors up to a whole one, every phase of a batch element's first
    step, two time steps up to several tiles; outputs of nothing but their own elements."""
    vec = 2 if dtype == torch.float64 else 4
    plan = forced(steps, waves, tiles)
    tile = steps * waves
    for C in (63 * vec + 1, 63 * vec + 3, 70 * vec - 1, 126 * vec - 1, 126 * vec + 1):
        for batch, T in ((5, 2), (3, tile - 1), (2, tile + 1), (1, 3 * tile + 2)):
            print(f"case shift {dtype} C={C} batch={batch} T={T} {steps}x{waves} tiles={tiles}", flush=True)
            for direction in (hip.FORWARD, hip.BACKWARD):  # (others run the plan in reserve)
                taken = hip.resolve_plan_cl(batch, T, C, dtype, direction, plan).waves_per_row
                assert taken == (plan.waves_per_row if runs(dtype, steps, waves, tiles, T) else 0)
            inputs, (a, b, gh), results = scan_pair(gpu, (batch, T, C), dtype, plan, seed=C + T)
            check(inputs, results, dtype)
    # The last shape again, into the middle of buffers, and a forward pass in place.
    n, L, code, stream = a.numel(), hip.lib(), hip._dtype_code(dtype), torch.cuda.current_stream().cuda_stream
    pad = 16 * vec
    for direction, count in ((hip.FORWARD, 1), (hip.BACKWARD, 2)):
        ws = torch.empty(max(8, hip.workspace_bytes_cl(*a.shape, dtype, direction, plan)), dtype=torch.uint8, device=gpu)
        out = [torch.full((n + 2 * pad,), 77.0, dtype=dtype, device=gpu) for _ in range(count)]
        p = [o[pad:].data_ptr() for o in out]
        if direction == hip.FORWARD:
            rc = L.scanscam_scan_fwd_cl(a.data_ptr(), b.data_ptr(), p[0], *a.shape, code, ws.data_ptr(), ws.numel(), stream, plan)
        else:
            rc = L.scanscam_scan_bwd_cl(a.data_ptr(), results[0].data_ptr(), gh.data_ptr(), p[0], p[1], *a.shape, code,
                                        ws.data_ptr(), ws.numel(), stream, plan)
        assert rc == 0
        for o, want in zip(out, results[:1] if count == 1 else results[1:]):
            assert torch.equal(o[pad:pad + n].view(a.shape), want)
            assert (o[:pad] == 77).all() and (o[pad + n:] == 77).all()
    ws = torch.empty(max(8, hip.workspace_bytes_cl(*a.shape, dtype, hip.FORWARD, plan)), dtype=torch.uint8, device=gpu)
    for place in (a, b):
        x, y = a.clone(), b.clone()
        target = x if place is a else y
        assert L.scanscam_scan_fwd_cl(x.data_ptr(), y.data_ptr(), target.data_ptr(), *a.shape, code, ws.data_ptr(), ws.numel(),
                                      stream, plan) == 0
        assert torch.equal(target, results[0])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,shape", [(torch.float32, (100, 300, 1001)), (torch.bfloat16, (64, 1100, 1003)),
                                         (torch.float64, (60, 300, 701)), (torch.float32, (2, 8000, 1601))])
def test_automatic_route(gpu, dtype, shape):
    """Calls that take these lanes by themselves give the results of the plan they report, bit for bit, and those of the plan
    in reserve to within the bar; tensors off the vector border, or not dense, keep the plan in reserve."""
    _, (a, b, gh), results = scan_pair(gpu, shape, dtype, None)
    plans = [hip.resolve_plan_cl(*shape, dtype, d) for d in (hip.FORWARD, hip.BACKWARD)]
    assert plans[0].waves_per_row < 0 and plans[1].waves_per_row < 0
    call = lambda x, h, g, p: (hip.transposed_linear_scan_forward(x, b, plan=p[0]),  # noqa: E731
                               *hip.transposed_linear_scan_backward(x, h, g, plan=p[1]))
    same = call(a, results[0], gh, plans)
    reserve = [hip.Plan(mode=p.mode, vec=p.vec, unroll=p.unroll, waves=p.waves) for p in plans]
    other = call(a, results[0], gh, reserve)
    for got, x, y in zip(results, same, other):
        assert torch.equal(got, x)
        assert rel_err(as_rows(got[:2]), as_rows(y[:2])) <= 2 * BAR[dtype]
    # One element off the border: the same results as the plan in reserve gives there.
    off = torch.empty(a.numel() + 1, dtype=dtype, device=gpu)[1:].view(shape)
    off.copy_(a)
    got = hip.transposed_linear_scan_forward(off, b)
    assert torch.equal(got, hip.transposed_linear_scan_forward(off, b, plan=plans[0]))
    assert rel_err(as_rows(got[:2]), as_rows(results[0][:2])) <= 2 * BAR[dtype]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,shape,code", [(torch.bfloat16, (8, 3000, 741), -1033), (torch.float16, (3, 1497, 2345), -521),
                                              (torch.bfloat16, (36, 290, 1003), -272), (torch.float32, (6, 1087, 3393), -273)])
def test_automatic_route_backwards(gpu, dtype, shape, code):
    """Calls that take these lanes backwards only."""
    plans = [hip.resolve_plan_cl(*shape, dtype, d) for d in (hip.FORWARD, hip.BACKWARD)]
    assert [p.waves_per_row for p in plans] == [0, code]
    print(f"case automatic {dtype} {shape} {plans[1]}", flush=True)
    _, (a, b, gh), results = scan_pair(gpu, shape, dtype, None)
    reserve = hip.Plan(mode=plans[1].mode, vec=plans[1].vec, unroll=plans[1].unroll, waves=plans[1].waves)
    same = hip.transposed_linear_scan_backward(a, results[0], gh, plan=plans[1])
    other = hip.transposed_linear_scan_backward(a, results[0], gh, plan=reserve)
    for got, x, y in zip(results[1:], same, other):
        assert torch.equal(got, x)
        floor = prev_abs(as_rows(results[0][:2])) if got is results[1] else None
        assert rel_err(as_rows(got[:2]), as_rows(y[:2]), floor) <= 2 * BAR[dtype]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", list(BAR))
@pytest.mark.parametrize("steps,waves,tiles", [(4, 8, 0), (8, 4, 0), (8, 4, 1)])
def test_values_that_are_no_numbers_stay_in_their_channels(gpu, dtype, steps, waves, tiles):
    """At the edges of groups, lanes and steps, whose vectors neighbours load as well."""
    vec = 2 if dtype == torch.float64 else 4
    shape = (3, 3 * steps * waves + 2, 126 * vec + 1)  # three groups of 43 vectors, the last of 41
    channels = [0, 1, vec, 43 * vec - 1, 43 * vec, 86 * vec - 1, 86 * vec, shape[2] - 2, shape[2] - 1]
    check_special_values(gpu, shape, dtype, forced(steps, waves, tiles), channels)


def test_where_the_route_lies():
    """Even or few channels, short or small calls keep the cost model's plan; the numbers that are no launch are not taken."""
    code = lambda b, T, C, dt, d: hip.resolve_plan_cl(b, T, C, dt, d).waves_per_row  # noqa: E731
    f32, bf16 = torch.float32, torch.bfloat16
    assert code(64, 2048, 1001, f32, hip.FORWARD) < 0 and code(64, 2048, 1001, bf16, hip.BACKWARD) < 0
    for shape in ((64, 2048, 1000), (64, 2048, 1002), (300, 2048, 251), (512, 255, 1001), (8, 256, 1001)):
        assert code(*shape, f32, hip.FORWARD) == 0, shape
    for bad in (-1, -(64 * 5 + 2 * 4), -(64 * 12 + 8), -(64 * 16 + 9), -(64 * 8), -(64 * 8 + 2 * 16), -(1 << 20)):
        assert hip.resolve_plan_cl(64, 2048, 1001, f32, hip.FORWARD, hip.Plan(waves_per_row=bad)).waves_per_row == 0, bad


HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_no_buffer_resource_starts_between_vectors(tmp_path):
    """The walk backwards addresses its tensors from a constant number of elements before a time step, i.e. from any element:
    buffer instructions, which want their resource to start on 4 bytes at least, have no place there."""
    csrc = os.path.join(os.path.dirname(os.path.abspath(hip.__file__)), "csrc")
    kernel = "template __global__ void scanscam::scan_cl_kernel<{}, {}, {}, true, scanscam::cl_max_threads({}, {}), false, {}>(scanscam::ClArgs);\n"
    source = tmp_path / "walks.hip"
    source.write_text('#include "scan_launch.hpp"\n' + "".join(
        kernel.format(t, v, s, v, s, m) for t, v, ms in (("__bf16", 4, (1, 3)), ("_Float16", 4, (1,)), ("float", 4, (1,)), ("double", 2, (1,)))
        for s in (4, 8) for m in ms))
    done = subprocess.run([HIPCC, "-O3", "-std=c++17", "--offload-arch=gfx950", "--offload-device-only", "-S", "-Xclang", "-target-feature",
                           "-Xclang", "-packed-fp32-ops", "-Wno-unused-command-line-argument", f"-I{csrc}",
                           f"-I{os.path.join(csrc, '../../include')}", str(source), "-o", str(tmp_path / "walks.s")],
                          capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stderr
    code = (tmp_path / "walks.s").read_text()
    assert code.count("global_load") > 100 and code.count("global_store") > 100
    assert "buffer_load" not in code and "buffer_store" not in code


def test_calls_that_the_cost_model_s_plan_runs_faster_keep_it():
    """Walks whose second round of workgroups is nearly empty, fp32 forwards below 1 GiB, tiles against a walk."""
    code = lambda b, T, C, dt, d: hip.resolve_plan_cl(b, T, C, dt, d).waves_per_row  # noqa: E731
    f32, f64, bf16, fwd, bwd = torch.float32, torch.float64, torch.bfloat16, hip.FORWARD, hip.BACKWARD
    for call in ((90, 1064, 531, bf16, fwd), (19, 831, 3293, bf16, fwd), (19, 831, 3293, bf16, bwd), (30, 857, 2161, bf16, bwd),
                 (32, 505, 2851, bf16, fwd), (29, 415, 2021, f32, fwd), (29, 415, 2021, f32, bwd), (88, 1133, 689, f32, bwd),
                 (44, 1080, 723, f64, bwd), (16, 1000, 3225, f32, fwd), (56, 1000, 993, f32, fwd), (9, 2173, 1651, f32, fwd),
                 (3, 4153, 2549, f32, fwd), (26, 260, 3223, f32, bwd), (1, 2361, 3531, bf16, bwd), (54, 368, 441, bf16, bwd)):
        assert code(*call) == 0, call
    for call in ((64, 1000, 977, bf16, fwd), (64, 1000, 977, bf16, bwd), (104, 1370, 965, bf16, fwd), (60, 600, 1001, f32, bwd),
                 (64, 2048, 1001, f32, fwd), (100, 300, 1001, f32, fwd), (42, 600, 741, f64, bwd), (2, 15698, 1589, f32, fwd),
                 (23, 1442, 871, f32, bwd), (36, 1357, 923, bf16, bwd), (11, 3192, 813, bf16, bwd)):
        assert code(*call) < 0, call


def test_tiles_multiply_no_more_gates_than_the_plan_in_reserve():
    """A super-tile's product of gates is a plain number: where the plan in reserve multiplies fewer, gates above one would
    take it out of range earlier (a walk multiplies a wave's own steps)."""
    rng, taken = random.Random(3), 0
    for _ in range(4000):
        dtype = rng.choice((torch.float32, torch.bfloat16, torch.float64))
        C = int(2 ** rng.uniform(8, 12)) | 1
        T = int(2 ** rng.uniform(8, 15))
        batch = max(1, int(2 ** rng.uniform(22, 27)) // (C * T))
        p = hip.resolve_plan_cl(batch, T, C, dtype, rng.randrange(2))
        if p.waves_per_row >= 0 or p.waves_per_row % 2 == 0:
            continue
        taken += 1
        steps, waves = -p.waves_per_row // 64, -p.waves_per_row // 2 % 32
        assert p.mode == hip.MODE_LOOKBACK and waves * waves * steps <= p.waves * p.waves * p.unroll, (batch, T, C, dtype, p)
    assert taken > 100


@pytest.mark.gpu
def test_gates_above_one_after_the_last_gradient(gpu):
    """Backwards over 563 steps of gates of 1.5 before the first output gradient other than zero: the gradients stay zero
    there, also in calls wide enough for tiles."""
    shape, last = (4, 1228, 2937), 665
    print(f"case {shape} {hip.resolve_plan_cl(*shape, torch.bfloat16, hip.BACKWARD)}", flush=True)
    g = torch.Generator().manual_seed(8)
    a = torch.rand(shape, generator=g)
    h, gh = torch.randn(shape, generator=g).bfloat16(), torch.randn(shape, generator=g)
    a[:, last:], gh[:, last:] = 1.5, 0
    a, gh = a.bfloat16(), gh.bfloat16()
    ga, gb = hip.transposed_linear_scan_backward(a.to(gpu), h.to(gpu), gh.to(gpu))
    want_ga, want_gb = oracle.bwd(as_rows(a), as_rows(h), as_rows(gh))
    assert rel_err(as_rows(gb), want_gb) <= BAR[torch.bfloat16]
    assert rel_err(as_rows(ga), want_ga, prev_abs(as_rows(h))) <= BAR[torch.bfloat16]
