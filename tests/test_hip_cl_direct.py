"""
The time split's look-back over all tiles before a tile (few tiles per row-group): parity with the CPU oracle at the edges
of the waves' runs of tiles, up to the first count of tiles that goes through super-tiles instead.
"""
import pytest
import torch

import oracle
from scanscam_amd import hip
from test_hip_channels_last import as_rows, prev_abs, rel_err
from test_hip_staged import BAR, check, scan_pair


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", list(BAR))
@pytest.mark.parametrize("vec,steps,waves", [(1, 4, 8), (1, 4, 3), (2, 4, 4), (1, 8, 1)])
def test_runs_of_tiles(gpu, dtype, vec, steps, waves):
    """2 tiles to 8 per wave and one more, the last one whole, of one step, and short; the same bits every time."""
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
