"""The step's partitioned tridiagonal solve (one thread per eigenvalue class and
segment) against the sequential one: a step in one call, which takes the first,
against the same step through the module routines, whose solve runs k_trid.
Grids of one column pair, a whole tile of pairs and one more, rows that are no
multiple of a tile, and depths on both sides of every change of the segments."""
import numpy as np
import pytest

import powerllel_channel_sycl_amd as pll

pytestmark = pytest.mark.gpu

SIZES = [(4, 4, 2), (4, 6, 8), (16, 6, 10), (18, 20, 16), (32, 10, 126), (36, 12, 130),
         (50, 18, 256), (20, 36, 258), (12, 10, 384), (12, 16, 386), (30, 12, 512), (12, 10, 514),
         (16, 18, 768), (8, 6, 770)]


def one_step(nx, ny, nz, precision, fused):
    dz = pll.mesh_by_func(1, 0, 1.5, nz, 2.0)
    with pll.Channel(nx, ny, nz, 6.0, 3.0, 2.0, 2800.0, 1e-4, dz, precision=precision) as ch:
        ch.initFlow("poi", noise_intensity=0.1)
        ch.updateBoundVel(0)
        ch.updateBoundP()
        if fused:
            ch.step(1)
        else:
            ch.timeIntVelRK1()
            ch.updateBoundVel(1)
            ch.timeIntVelRK2()
            ch.updateBoundVel(0)
            ch.calcRHS()
            ch.execute_poisson_solver()
            ch.updateBoundP()
            ch.correctVel()
            ch.forceVel()
            ch.updateBoundVel(0)
        return [ch.download(f).astype(np.float64) for f in ("u", "v", "w")]


@pytest.mark.parametrize("nx,ny,nz", SIZES)
def test_step_solve_matches_sequential_solve(nx, ny, nz):
    print(f"CASE step solve {nx}x{ny}x{nz}", flush=True)
    # velocities of order one, round-off 1e-16 times the condition of the
    # elimination, at most ~nz^2 = 6e5
    for a, b in zip(one_step(nx, ny, nz, "fp64", True), one_step(nx, ny, nz, "fp64", False)):
        assert np.max(np.abs(a - b)) < 1e-10


@pytest.mark.parametrize("nx,ny,nz", SIZES)
def test_fp32_step_solve_is_as_accurate_as_sequential_solve(nx, ny, nz):
    """Both solves round p to FP32 (p is large after one step of a noisy start, so
    the velocity's error depends on the grid): the error against FP64 is compared."""
    print(f"CASE fp32 step solve {nx}x{ny}x{nz}", flush=True)
    ref = one_step(nx, ny, nz, "fp64", False)
    for r, a, b in zip(ref, one_step(nx, ny, nz, "fp32_mixed", True),
                       one_step(nx, ny, nz, "fp32_mixed", False)):
        assert np.max(np.abs(a - r)) <= 2.0 * np.max(np.abs(b - r)) + 1e-6
