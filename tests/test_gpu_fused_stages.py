"""The two RK stages in one kernel (k_rk12) against the separate ones: n steps
in one call, which fuse the stages of every step but the first and leave u1 on
the last, against n calls of one step, which do not.  Grids smaller than a tile,
one cell past a tile edge in x and y, one and several chunks of planes, and a
convecting frame (the u_crf terms)."""
import numpy as np
import pytest

import powerllel_channel_sycl_amd as pll

pytestmark = pytest.mark.gpu

SIZES = [(4, 4, 2), (64, 12, 4), (64, 16, 10), (72, 18, 8), (120, 24, 6), (128, 48, 50), (60, 50, 96)]


@pytest.mark.parametrize("precision", ["fp64", "fp32_mixed"])
@pytest.mark.parametrize("u_crf", [0.0, 0.3])
@pytest.mark.parametrize("nx,ny,nz", SIZES)
def test_fused_stages_match_separate_ones(nx, ny, nz, u_crf, precision):
    print(f"CASE fused stages {nx}x{ny}x{nz} crf {u_crf} {precision}", flush=True)
    dz = pll.mesh_by_func(1, 0, 1.5, nz, 2.0)
    out = []
    for calls in ((5,), (1,) * 5):
        with pll.Channel(nx, ny, nz, 6.0, 3.0, 2.0, 2800.0, 1e-3, dz, precision=precision,
                         u_crf=u_crf) as ch:
            ch.initFlow("poi", noise_intensity=0.1)
            ch.updateBoundVel(0)
            ch.updateBoundP()
            for n in calls:
                ch.step(n)
            out.append([ch.download(f) for f in ("u", "v", "w", "u1", "v1", "w1")])
    for a, b in zip(*out):
        # velocities of order one, a few roundings a step: FP64 ~1e-14, FP32 ~3e-6
        assert np.max(np.abs(a - b)) < (1e-12 if precision == "fp64" else 1e-5)
