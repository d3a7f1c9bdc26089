"""The bulk mean that a run's forcing takes from stage 2's partial sums: every
forward transform that combines them (whole planes, compiled-in lengths with blocks
of one wave and of 60 threads, run-time plans)."""
import numpy as np
import pytest

import powerllel_channel_sycl_amd as pll

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(24, 20, 12), (48, 48, 32), (64, 64, 64), (128, 96, 48),
                                      (1250, 8, 24)])
def test_forcing_holds_the_bulk_velocity_to_rounding(nx, ny, nz):
    """After a run the bulk velocity is 1 up to the mean's own rounding, about 8e-17
    rms for a tree of sums near 1 and two divisions (units of 1.1e-16, uniform
    errors); 24 runs scatter their rms by 15 %.  A chain of 64 sums gives 2e-16."""
    print(f"CASE bulk mean {nx}x{ny}x{nz}", flush=True)
    dz = pll.mesh_by_func(1, 0, 1.5, nz, 2.0)
    err = []
    for seed in range(1, 73, 3):
        with pll.Channel(nx, ny, nz, 6.0, 3.0, 2.0, 2800.0, 1e-3 if nx < 1000 else 1e-4, dz) as ch:
            ch.initFlow("poi", noise_intensity=0.1, seeds=(seed, seed + 1, seed + 2))
            ch.updateBoundVel(0)
            ch.updateBoundP()
            ch.step(4)
            u = ch.download("u")[1:-1, 1:-1, 1:-1].astype(np.longdouble)
        w = (dz[1:-1] / 2.0).astype(np.longdouble)
        err.append(float((u.sum((1, 2)) * w).sum() / (nx * ny) - 1))
    rms = np.sqrt(np.mean(np.square(err)))
    print(f"  rms {rms:.2e}", flush=True)
    assert rms < 1.4e-16
