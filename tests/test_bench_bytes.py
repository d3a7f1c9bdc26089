"""The bytes that bench.py rates its kernels by, from the arrays that each launched
kernel reads and writes.  Nothing here touches a GPU."""
import pytest

from test_bench_cpu import _bench

VEL, P, WORK, U = 3, 1, 1, 1  # arrays
# kernel: arrays read + arrays written
MOVED = {"rk1": VEL + VEL, "rk2": 2 * VEL + VEL, "rk12": VEL + P + VEL, "calc_rhs": VEL + P,
         "fft_x_fwd": P + WORK, "fft_x_fwd_rhs": VEL + WORK, "fft_y_fwd": 2 * WORK,
         "solve_trid": 2 * WORK, "fft_y_bwd": 2 * WORK, "fft_x_bwd": WORK + P,
         "correct_vel": P + VEL + VEL, "mean_partial": U, "force_add": 2 * U}


@pytest.mark.parametrize("precision,size", [("fp64", 8), ("fp32_mixed", 4)])
def test_launch_bytes_are_the_arrays_moved(precision, size):
    b = _bench()
    assert b.LAUNCH_BYTES[precision] == {k: n * size for k, n in MOVED.items()}
    # a step inside a run reads and writes u, v, w, reads p, and passes over the
    # work array five times after its right-hand side, the last time into p
    assert sum(b.LAUNCH_BYTES[precision][k] for k in b.RUN_STEP) == 19 * size


def test_a_step_is_rated_by_its_own_bytes(monkeypatch):
    """A step at the memory's peak rate is 1.0 of it, and the unfused sequence's
    312 B a point are given as an equivalent rate."""
    b = _bench()
    npts = 10 ** 9

    class Run:
        def step(self, n):
            clock[0] += n * 152 * npts / (b.HBM_PEAK_GBS * 1e9)

        def timing_read(self):
            return {"rk12": (56 * npts / (b.HBM_PEAK_GBS * 1e9) * 1e3, 1)}

        def __getattr__(self, name):
            return lambda *a: 0.0 if name in ("Mean", "device_bytes") else (0.0, 0)
    clock = [0.0]
    monkeypatch.setattr(b.time, "perf_counter", lambda: clock[0])
    monkeypatch.setattr(b, "build_channel", lambda wl, precision: (Run(), npts))
    r = b.measure("none", "fp64", 4, 1)["roofline"]
    assert r["step_frac"] == pytest.approx(1.0, abs=1e-3) and r["frac"] == pytest.approx(1.0, abs=1e-3)
    assert r["bytes_per_point_step"] == 152
    assert r["unfused_equivalent_GBps"] == pytest.approx(8000.0 * 312 / 152, rel=1e-3)
