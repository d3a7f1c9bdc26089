"""The compiled-in transforms: every length, against numpy's rfft in the perm packing
of src/mod_fft.cc:60-187; rows that do not fill the last block and ragged last
tiles of columns; and the step's forms of them (calcRHS in the forward loads, p's
boundary update in the inverse's stores) against the routines.  The run-time plans
of the same lengths as well, which PLL_FFT_GENERIC selects."""
import numpy as np
import pytest

import powerllel_channel_sycl_amd as pll
from test_gpu_fft_lengths import SIZES, perm

pytestmark = pytest.mark.gpu


def smooth(lo, hi, step=1):
    out = []
    for n in range(lo, hi + 1, step):
        m = n
        for p in (2, 3, 5):
            while m % p == 0:
                m //= p
        if m == 1:
            out.append(n)
    return out


X = [2 * n for n in smooth(2, 768)]
Y = smooth(4, 768, 2)


def check(nx, ny, nz, precision):
    # relative to the largest coefficient: a few roundings (2^-53, 2^-24) for each pass
    tol = 1e-13 if precision == "fp64" else 2e-6
    p = np.random.default_rng(nx * 1000 + ny).standard_normal((nz + 2, ny + 2, nx + 2))
    if precision != "fp64":
        p = p.astype(np.float32).astype(np.float64)
    with pll.Channel(nx, ny, nz, 2.0, 1.0, 2.0, 100.0, 1e-3, np.ones(nz + 2),
                     precision=precision) as ch:
        ch.upload("p", p)
        a = p[1:-1, 1:-1, 1:-1]
        for f, axis in ((ch.execute_fft_fwd_xpen, 2), (ch.execute_fft_fwd_ypen, 1)):
            f()
            a = perm(a, axis)
            got = ch.download_spec().reshape(a.shape)
            assert np.max(np.abs(got - a)) < tol * np.max(np.abs(a)), axis
        ch.upload("p", np.zeros_like(p))
        ch.execute_fft_bwd_ypen()
        ch.execute_fft_bwd_xpen()
        got = ch.download("p")
        assert np.max(np.abs((got - p)[1:-1, 1:-1, 1:-1])) < tol * np.max(np.abs(p))


@pytest.mark.parametrize("precision", ["fp64", "fp32_mixed"])
@pytest.mark.parametrize("nx", X)
def test_x_lengths(nx, precision):
    print(f"CASE fixed x {nx} {precision}", flush=True)
    check(nx, 6, 2, precision)


@pytest.mark.parametrize("precision", ["fp64", "fp32_mixed"])
@pytest.mark.parametrize("ny", Y)
def test_y_lengths(ny, precision):
    print(f"CASE fixed y {ny} {precision}", flush=True)
    check(36, ny, 2, precision)


@pytest.mark.parametrize("precision", ["fp64", "fp32_mixed"])
@pytest.mark.parametrize("nx,ny", [s for s in SIZES if max(s) <= 768])
def test_run_time_plans(nx, ny, precision, monkeypatch):
    print(f"CASE run-time plan {nx}x{ny} {precision}", flush=True)
    monkeypatch.setenv("PLL_FFT_GENERIC", "1")
    check(nx, ny, 2, precision)


@pytest.mark.parametrize("precision", ["fp64", "fp32_mixed"])
@pytest.mark.parametrize("nx,ny,nz", [(8, 6, 6), (32, 16, 10), (50, 50, 4), (192, 64, 6), (250, 162, 4),
                                      (768, 12, 4), (1458, 6, 2), (1536, 4, 2)])
def test_steps_match_the_routines(nx, ny, nz, precision):
    print(f"CASE fixed steps {nx}x{ny}x{nz} {precision}", flush=True)
    dz = pll.mesh_by_func(1, 0, 1.5, nz, 2.0)
    out = []
    for whole in (True, False):
        with pll.Channel(nx, ny, nz, 6.0, 3.0, 2.0, 2800.0, 1e-3, dz, precision=precision) as ch:
            ch.initFlow("poi", noise_intensity=0.02)
            ch.updateBoundVel(0)
            ch.updateBoundP()
            if whole:
                ch.step(2)
                p = ch.download("p")
                # the halos are copies (src/mod_updateBound.cc:253-296)
                q = p[1:-1, 1:-1, 1:-1]
                img = np.pad(np.pad(q, ((0, 0), (1, 1), (1, 1)), mode="wrap"),
                             ((1, 1), (0, 0), (0, 0)), mode="edge")
                assert np.array_equal(p, img)
            else:
                for _ in range(2):
                    ch.timeIntVelRK1(); ch.updateBoundVel(1); ch.timeIntVelRK2()
                    ch.updateBoundVel(0); ch.calcRHS(); ch.execute_poisson_solver()
                    ch.updateBoundP(); ch.correctVel(); ch.forceVel(); ch.updateBoundVel(0)
            out.append([ch.download(f) for f in ("u", "v", "w")])
    for a, b in zip(*out):
        # velocities of order one: FP64 round-off; FP32 the step's accumulated rounding
        assert np.max(np.abs(a - b)) < (1e-12 if precision == "fp64" else 1e-5)


@pytest.mark.parametrize("precision", ["fp64", "fp32_mixed"])
@pytest.mark.parametrize("nx,ny,nz", [(4, 4, 2), (24, 20, 12), (30, 18, 6), (6, 162, 4), (250, 4, 4),
                                      (32, 32, 8), (64, 16, 6)])
def test_steps_of_whole_planes_match_the_routines(nx, ny, nz, precision):
    """Planes of up to 512 complex slots, odd nx/2 and the limit among them."""
    test_steps_match_the_routines(nx, ny, nz, precision)


@pytest.mark.parametrize("precision", ["fp64", "fp32_mixed"])
@pytest.mark.parametrize("nx,ny,nz", [(18, 10, 8), (200, 90, 12), (90, 54, 20)])
def test_steps_with_run_time_plans_match_the_routines(nx, ny, nz, precision, monkeypatch):
    monkeypatch.setenv("PLL_FFT_GENERIC", "1")
    test_steps_match_the_routines(nx, ny, nz, precision)


@pytest.mark.parametrize("precision", ["fp64", "fp32_mixed"])
@pytest.mark.parametrize("nx,ny,nz", [(1600, 6, 4), (12, 800, 4)])
def test_steps_of_long_lengths_match_the_routines(nx, ny, nz, precision):
    """Lengths beyond the compiled-in ones."""
    test_steps_match_the_routines(nx, ny, nz, precision)
