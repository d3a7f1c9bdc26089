"""The transforms of lengths without a compiled-in kernel: every radix of the
run-time plans (2..16), one to four passes, ragged last tiles and blocks, the
shortest and the longest rows and columns, against numpy's rfft in the perm
packing [X0, X(n/2), Re X1, Im X1, ...] of src/mod_fft.cc:60-187."""
import numpy as np
import pytest

import powerllel_channel_sycl_amd as pll

pytestmark = pytest.mark.gpu

# (nx, ny): x points nx/2 and y points ny
SIZES = [
    (4, 4), (6, 10), (18, 16), (30, 18), (36, 24), (50, 30), (54, 50), (90, 36), (200, 90),
    (250, 162), (320, 100), (324, 150), (450, 240), (480, 270), (500, 360), (540, 54),
    (4096, 8), (12, 2048), (4050, 6),
]


def perm(a, axis):
    """numpy's half spectrum along axis in perm packing."""
    f = np.moveaxis(np.fft.rfft(a, axis=axis), axis, -1)
    out = np.empty(f.shape[:-1] + (a.shape[axis],))
    out[..., 0], out[..., 1] = f[..., 0].real, f[..., -1].real
    out[..., 2::2], out[..., 3::2] = f[..., 1:-1].real, f[..., 1:-1].imag
    return np.moveaxis(out, -1, axis)


@pytest.mark.parametrize("precision", ["fp64", "fp32_mixed"])
@pytest.mark.parametrize("nx,ny", SIZES)
def test_transforms_of_any_length(nx, ny, precision):
    print(f"CASE fft lengths {nx}x{ny} {precision}", flush=True)
    # relative to the largest coefficient: a few roundings (2^-53, 2^-24) for each pass
    tol = 1e-13 if precision == "fp64" else 2e-6
    nz = 2
    p = np.random.default_rng(nx * 1000 + ny).standard_normal((nz + 2, ny + 2, nx + 2))
    if precision != "fp64":
        p = p.astype(np.float32).astype(np.float64)
    with pll.Channel(nx, ny, nz, 2.0, 1.0, 2.0, 100.0, 1e-3, np.ones(nz + 2),
                     precision=precision) as ch:
        ch.upload("p", p)
        a = p[1:-1, 1:-1, 1:-1]
        for f, axis, n in ((ch.execute_fft_fwd_xpen, 2, nx), (ch.execute_fft_fwd_ypen, 1, ny)):
            f()
            a = perm(a, axis)
            got = ch.download_spec().reshape(a.shape)
            assert np.max(np.abs(got - a)) < tol * np.max(np.abs(a)), (axis, n)
        ch.upload("p", np.zeros_like(p))
        ch.execute_fft_bwd_ypen()
        ch.execute_fft_bwd_xpen()
        got = ch.download("p")
        assert np.max(np.abs((got - p)[1:-1, 1:-1, 1:-1])) < tol * np.max(np.abs(p))


@pytest.mark.parametrize("precision", ["fp64", "fp32_mixed"])
@pytest.mark.parametrize("nx,ny,nz", [(18, 10, 8), (200, 90, 12), (90, 54, 20)])
def test_steps_of_any_length_match_the_routines(nx, ny, nz, precision):
    """Three steps in one call (calcRHS inside the forward transform's loads,
    p's periodic halos in the inverse's stores) against the routines one by one."""
    print(f"CASE step lengths {nx}x{ny}x{nz} {precision}", flush=True)
    dz = pll.mesh_by_func(1, 0, 1.5, nz, 2.0)
    out = []
    for whole in (True, False):
        with pll.Channel(nx, ny, nz, 6.0, 3.0, 2.0, 2800.0, 2e-3, dz, precision=precision) as ch:
            ch.initFlow("poi", noise_intensity=0.1)
            ch.updateBoundVel(0)
            ch.updateBoundP()
            if whole:
                ch.step(3)
            else:
                for _ in range(3):
                    ch.timeIntVelRK1(); ch.updateBoundVel(1); ch.timeIntVelRK2()
                    ch.updateBoundVel(0); ch.calcRHS(); ch.execute_poisson_solver()
                    ch.updateBoundP(); ch.correctVel(); ch.forceVel(); ch.updateBoundVel(0)
            out.append([ch.download(f) for f in ("u", "v", "w", "u1", "v1", "w1")])
    for a, b in zip(*out):
        # velocities of order one: FP64 round-off; FP32 the step's accumulated rounding
        assert np.max(np.abs(a - b)) < (1e-12 if precision == "fp64" else 1e-5)
