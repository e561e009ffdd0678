"""
The time split's look-back over all tiles before a tile (few tiles per row-group): parity with the CPU oracle at the edges
of the waves' runs of tiles, up to the first count of tiles that goes through super-tiles instead.
"""
import pytest
import torch

from scanscam_amd import hip
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
