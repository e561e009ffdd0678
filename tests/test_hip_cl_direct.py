"""
The time split's look-back over all tiles before a tile (few tiles per row-group): parity with the CPU oracle at the edges
of the waves' runs of tiles, up to the first count of tiles that goes through super-tiles instead.
"""
import pytest
import torch

import oracle
from scanscam_amd import hip
from test_hip_channels_last import as_rows, prev_abs, rel_err
from test_hip_staged import BAR, check, check_special_values, scan_pair


def through_super_tiles(gpu, shape, dtype, direction, plan):
    """Whether a call of more tiles than waves goes through the chain of super-tiles: it publishes their aggregates, in the
    last words of the workspace, all of which are alike to begin with."""
    batch, T, C = shape
    tiles, L = -(-T // (plan.unroll * plan.waves)), hip.lib()
    assert tiles > plan.waves
    supers = batch * -(-C // (64 * plan.vec)) * -(-tiles // plan.waves) * 64 * plan.vec * (6 if dtype == torch.float64 else 2)
    n = hip.workspace_bytes_cl(*shape, dtype, direction, plan)
    ws, t = torch.empty(n, dtype=torch.uint8, device=gpu), [torch.rand(shape, device=gpu).to(dtype) for _ in range(5)]
    p, tail = [x.data_ptr() for x in t], (*shape, hip._dtype_code(dtype), ws.data_ptr(), n, torch.cuda.current_stream().cuda_stream, plan)
    rc = L.scanscam_scan_fwd_cl(*p[:3], *tail) if direction == hip.FORWARD else L.scanscam_scan_bwd_cl(*p, *tail)
    assert rc == 0
    words = ws.view(torch.int64)[-supers:]
    return bool((words != words[-1]).any())


@pytest.mark.gpu
def test_where_the_chain_takes_over(gpu):
    """8 tiles per wave, 1024 steps per wave, 2048 workgroups (16 single 16-bit channels backwards: 896), no fp64."""
    f32, bf16, f64, fwd, bwd = torch.float32, torch.bfloat16, torch.float64, hip.FORWARD, hip.BACKWARD
    for shape, dtype, steps, waves, chain in [
            ((2, 2048, 70), f32, 4, 8, (False, False)), ((2, 2049, 70), f32, 4, 8, (True, True)),
            ((1, 8192, 64), f32, 16, 8, (False, False)), ((1, 8193, 64), bf16, 16, 8, (True, True)),
            ((227, 288, 64), f32, 4, 8, (False, False)), ((228, 288, 64), f32, 4, 8, (True, True)),
            ((99, 576, 64), bf16, 16, 4, (False, False)), ((100, 576, 64), bf16, 16, 4, (False, True)),
            ((100, 576, 64), f32, 16, 4, (False, False)), ((100, 288, 64), bf16, 8, 4, (False, False)),
            ((2, 2048, 70), f64, 4, 8, (True, True))]:
        plan = hip.Plan(mode=hip.MODE_LOOKBACK, vec=1, unroll=steps, waves=waves)
        print(f"case {shape} {dtype} {plan}", flush=True)
        assert tuple(through_super_tiles(gpu, shape, dtype, d, plan) for d in (fwd, bwd)) == chain, (shape, dtype, steps, waves)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", list(BAR))
@pytest.mark.parametrize("vec,steps,waves", [(1, 4, 8), (1, 4, 3), (2, 4, 4), (1, 8, 1)])
def test_runs_of_tiles(gpu, dtype, vec, steps, waves):
    """2 tiles to 8 per wave and one more, the last one whole, of one step, and short; the same bits every time. The chain
    takes the count beyond, and all of fp64."""
    plan = hip.Plan(mode=hip.MODE_LOOKBACK, vec=vec, unroll=steps, waves=waves)
    tile = steps * waves
    for tiles in sorted({2, 9, waves, waves + 1, 2 * waves + 1, 5 * waves, 8 * waves, 8 * waves + 1} - {1}):
        for T in (tiles * tile, tiles * tile - tile + 1, tiles * tile - 1):
            print(f"case direct {dtype} {plan} tiles={tiles} T={T}", flush=True)
            inputs, (a, b, gh), results = scan_pair(gpu, (2, T, 130), dtype, plan, seed=T)
            check(inputs, results, dtype)
        again = (hip.transposed_linear_scan_forward(a, b, plan=plan),
                 *hip.transposed_linear_scan_backward(a, results[0], gh, plan=plan))
        for x, y in zip(results, again):
            assert torch.equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("steps,waves,tiles,grown,rate", [(8, 4, 28, (0, 28), 1.6),    # runs of 7 tiles, super-tiles of 4
                                                          (4, 8, 42, (6, 12), 1.75)])  # a run of 6, inside two super-tiles of 8
def test_gates_above_one_before_the_first_value(gpu, dtype, steps, waves, tiles, grown, rate):
    """Growing gates whose product over a wave's run of tiles is beyond fp32 and over the chain's super-tiles is not, while
    the scan value still is zero: it stays zero."""
    plan, tile = hip.Plan(mode=hip.MODE_LOOKBACK, vec=1, unroll=steps, waves=waves), steps * waves
    T, lo, hi = tiles * tile, grown[0] * tile, grown[1] * tile
    print(f"case {dtype} {plan} T={T}", flush=True)
    g = torch.Generator().manual_seed(7)
    a = torch.rand((2, T, 70), generator=g)
    x, h = (torch.randn((2, T, 70), generator=g).to(dtype) for _ in range(2))
    last = min(hi, T - tile)  # (the last tile holds the first values)
    a[:, lo:last] = rate
    x[:, :last] = 0
    a = a.to(dtype)
    got = hip.transposed_linear_scan_forward(a.to(gpu), x.to(gpu), plan=plan)
    assert rel_err(as_rows(got), oracle.fwd(as_rows(a), as_rows(x))) <= BAR[dtype]
    a, x = a.flip(1).roll(1, 1).contiguous(), x.flip(1).contiguous()  # (the gate of step t is a[t + 1] backwards)
    ga, gb = hip.transposed_linear_scan_backward(a.to(gpu), h.to(gpu), x.to(gpu), plan=plan)
    want_ga, want_gb = oracle.bwd(as_rows(a), as_rows(h), as_rows(x))
    assert rel_err(as_rows(gb), want_gb) <= BAR[dtype]
    assert rel_err(as_rows(ga), want_ga, prev_abs(as_rows(h))) <= BAR[dtype]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("vec,steps,waves,tiles", [(1, 4, 8, 20), (2, 4, 4, 9), (4, 4, 8, 3)])
def test_values_that_are_no_numbers(gpu, dtype, vec, steps, waves, tiles):
    plan = hip.Plan(mode=hip.MODE_LOOKBACK, vec=vec, unroll=steps, waves=waves)
    check_special_values(gpu, (3, tiles * steps * waves - 1, 132), dtype, plan, [0, 1, 63, 64, 65, 70, 127, 128, 130, 131])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_an_expired_wait_ends_and_is_reported(gpu, dtype):
    """One poll per wait: every wave still ends, and either no wait expired and the result is the usual one, or the flag is
    raised and there are NaN; what is neither NaN nor the usual result there is none."""
    shape, L = (4, 2048, 256), hip.lib()
    g = torch.Generator(device=gpu).manual_seed(29)
    x, y = (torch.rand(shape, generator=g, device=gpu).to(dtype) for _ in range(2))
    plan = hip.Plan(mode=hip.MODE_LOOKBACK, vec=1, unroll=4, waves=8)
    assert not through_super_tiles(gpu, shape, dtype, hip.FORWARD, plan)
    good = hip.transposed_linear_scan_forward(x, y, plan=plan)
    once = hip.Plan(mode=hip.MODE_LOOKBACK, vec=1, unroll=4, waves=8, spin_limit=1)
    n = hip.workspace_bytes_cl(*shape, dtype, hip.FORWARD, once)
    ws, out = torch.empty(n, dtype=torch.uint8, device=gpu), torch.empty_like(x)
    rc = L.scanscam_scan_fwd_cl(x.data_ptr(), y.data_ptr(), out.data_ptr(), *shape, hip._dtype_code(dtype), ws.data_ptr(), n,
                                torch.cuda.current_stream().cuda_stream, once)
    assert rc == 0
    expired = int(ws.view(torch.int64)[1].item()) != 0
    print(f"case one poll {dtype}: {'expired' if expired else 'no wait expired'}", flush=True)
    assert bool(torch.isnan(out).any()) == expired
    assert torch.equal(out[~torch.isnan(out)], good[~torch.isnan(out)])
    assert torch.equal(hip.transposed_linear_scan_forward(x, y, plan=plan), good)
