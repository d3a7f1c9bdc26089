"""The rounding of the fused RK stages of an FP64 run (k_rk12): they may round in
another order than the reference's separate stages, but no more."""
import numpy as np
import pytest

import powerllel_channel_sycl_amd as pll

pytestmark = pytest.mark.gpu

STEPS = 50


def diffusion(u, dt, nu, dz):
    """Heun steps of u_t = nu u_zz between walls, in 80 bits."""
    u, dt, nu, dz = u.astype(np.longdouble), np.longdouble(dt), np.longdouble(nu), np.longdouble(dz)

    def rate(a):
        b = np.concatenate([-a[:1], a, -a[-1:]])
        return nu * ((b[2:] - b[1:-1]) - (b[1:-1] - b[:-2])) / (dz * dz)
    for _ in range(STEPS):
        one = u + dt * rate(u)
        u = (u + one + dt * rate(one)) / 2
    return u


@pytest.mark.parametrize("number", [0.01, 0.2])
def test_fused_stages_round_no_more_than_separate_ones(number):
    """u varies in z alone, so it diffuses (p, v and w stay 0): the errors of 6144
    values after 50 steps in one call (fused) and in 50 calls (the separate
    stages), of a diffusion number dt nu/dz^2.  The ratio of two such rms errors
    scatters by about 1.3 %.  Adding the old value first in stage 2 makes it 1.16, and
    the viscous terms as neighbours minus a rounded diagonal 5.8 at 0.2."""
    print(f"CASE rounding of diffusion, number {number}", flush=True)
    nx, ny, nz, dt = 4, 4, 768, 1e-3
    dz = 2.0 / nz
    re = dt / (number * dz * dz)
    sq = {1: 0.0, STEPS: 0.0}
    for seed in range(8):
        start = 0.5 + 0.5 * np.random.default_rng(seed).random(nz)
        want = diffusion(start, dt, 1.0 / np.longdouble(re), dz)
        for n in sq:
            u = np.zeros((nz + 2, ny + 2, nx + 2))
            u[1:-1] = start[:, None, None]
            with pll.Channel(nx, ny, nz, 2.0, 2.0, 2.0, re, dt, np.full(nz + 2, dz),
                             is_forced=(0, 0, 0)) as ch:
                ch.upload("u", u)
                ch.updateBoundVel(0)
                ch.updateBoundP()
                for _ in range(STEPS // n):
                    ch.step(n)
                got = ch.download("u")[1:-1, 1:-1, 1:-1]
                assert np.all(ch.download("w") == 0.0)
            assert np.all(got == got[:, :1, :1])
            sq[n] += float(np.sum((got[:, 0, 0] - want) ** 2))
    ratio = np.sqrt(sq[STEPS] / sq[1])
    print(f"  rms {np.sqrt(sq[STEPS] / (8 * nz)):.2e} fused, {np.sqrt(sq[1] / (8 * nz)):.2e} "
          f"separate, ratio {ratio:.3f}", flush=True)
    assert ratio < 1.08
