"""The marching stencil at the edges of its dispatch: grids on both sides of
the sizes where it takes over from the tiles (2^18 cells at 1 sweep, and
at 2 on 4-8 layers, 5 * 2^16 at 2 otherwise, 2^20 at 3-4), short, long and ragged segments, single-step and two-step
passes, calls of one and two steps, against
the CPU restatement of the grid step, bit for bit."""
import numpy as np
import pytest

from hbfsim_amd import engine as eng
from test_gpu_thermal import f, grid_kw

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,sweeps,steps,passes", [
    ((128, 256, 8), 1, 3, 2), ((127, 258, 8), 1, 3, 3),       # 2^18 cells, one fewer strip
    ((128, 256, 8), 2, 4, 2), ((127, 258, 8), 2, 4, 4), ((128, 512, 4), 2, 4, 2),
    ((121, 2167, 1), 2, 4, 4), ((121, 2709, 1), 2, 4, 2), ((119, 2760, 1), 2, 4, 4),
    ((128, 284, 9), 2, 4, 4), ((128, 285, 9), 2, 4, 2),
    # calls of one and two steps: tiles, single passes, the fused pass from 2^21 cells
    ((128, 256, 8), 1, 2, 2), ((128, 512, 8), 1, 1, 1), ((128, 512, 8), 1, 2, 2),
    ((128, 512, 8), 2, 2, 2), ((128, 512, 8), 2, 3, 2), ((512, 512, 8), 1, 2, 1),
    ((512, 511, 8), 1, 2, 2), ((512, 512, 8), 1, 5, 3),
    # segments of eight rows a level (one sweep, up to three layers), and of two
    ((1001, 700, 3), 1, 5, 3), ((151, 13_900, 1), 1, 4, 2), ((1449, 1451, 1), 1, 4, 2),
    ((725, 727, 4), 1, 4, 2),
    ((116, 3100, 3), 3, 4, 2), ((128, 1024, 8), 4, 4, 4), ((127, 1024, 8), 4, 3, 3),
    ((513, 511, 4), 4, 3, 3), ((512, 128, 16), 4, 2, 2), ((517, 64, 8), 2, 5, 3),
    ((130, 1030, 8), 3, 5, 3), ((110, 9533, 1), 4, 3, 3),
    # the last grid of single-step passes at 4 sweeps, and the first fused one
    ((1181, 1183, 8), 4, 2, 2), ((1183, 1183, 8), 4, 2, 1),
])
def test_march_bit_exact(oracle, shape, sweeps, steps, passes):
    import torch
    nx, ny, nz = shape
    n = nx * ny * nz
    g = grid_kw(nx=nx, ny=ny, nz=nz, sweeps=sweeps)
    rng = np.random.default_rng(n)
    t0 = rng.uniform(318.0, 340.0, n)
    power = rng.uniform(0.0, 0.05, n)
    th = eng.Thermal(**g)
    try:
        t = torch.from_numpy(t0.copy()).cuda()
        th.step(torch.from_numpy(power).cuda(), t, steps)
        got = t.cpu().numpy()
        assert th.last_launches() == passes
    finally:
        th.close()
    want = t0.copy()
    for _ in range(steps):
        assert oracle.orc_thermal_grid_step(nx, ny, nz, g["capacity_j_per_k"], g["gx_w_per_k"],
                                            g["gy_w_per_k"], g["gz_w_per_k"], g["top_g_w_per_k"],
                                            g["ambient_k"], g["dt_s"], f(power), f(want), -1.0,
                                            sweeps) == sweeps
    np.testing.assert_array_equal(got, want)
