"""Stages of an attached context and changes of the closure's weights, enqueued
one behind the other without a wait: as if each had been waited for."""
import numpy as np
import pytest

import powerllel_channel_sycl_amd as pll
from test_gpu_closure import _data, _dev, _random_params

pytestmark = pytest.mark.gpu


def change(cl, how, data):
    if how == "train":
        cl.train_step(data[0].data_ptr(), data[1].data_ptr(), len(data[1]), 0.05)
    else:
        cl.set_params(_random_params(9))


@pytest.mark.parametrize("how", ["train", "set_params"])
@pytest.mark.parametrize("detach", [False, True])
def test_weights_change_behind_enqueued_stages(how, detach):
    print(f"CASE weights change by {how} behind enqueued stages, detached {detach}", flush=True)
    data = [_dev(a) for a in _data(64, 2)]  # a short step: it would overtake the run
    out = []
    for wait in (True, False):
        cl = pll.Closure(seed=1)
        cl.set_params(_random_params(5))
        cl.set_scales(0.05, 2.0, 1e-4)
        with pll.Channel(96, 64, 64, 6.0, 3.0, 2.0, 6875.0, 2e-3,
                         pll.mesh_by_func(1, 0, 1.5, 64, 2.0)) as ch:
            ch.initFlow("poi", noise_intensity=0.1)
            ch.updateBoundVel(0)
            ch.updateBoundP()
            ch.attach_closure(cl)
            ch.synchronize()
            for _ in range(3):
                ch.step(20)
                if wait:
                    ch.synchronize()
                if detach:
                    ch.attach_closure(None)
                change(cl, how, data)
                if wait:
                    cl.synchronize()
                if detach:
                    ch.attach_closure(cl)
            ch.step(2)
            out.append([ch.download(f) for f in ("u", "v", "w")] + [ch.closure_nut(), cl.params()])
        cl.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert not np.array_equal(out[0][-1], _random_params(5))


def test_context_and_closure_go_in_any_order():
    print("CASE context outlives its closure, closure outlives its context", flush=True)
    data = [_dev(a) for a in _data(64, 2)]
    for first in ("closure", "context"):
        cl = pll.Closure(seed=1)
        ch = pll.Channel(16, 12, 8, 6.0, 3.0, 2.0, 6875.0, 2e-3, pll.mesh_by_func(1, 0, 1.5, 8, 2.0))
        ch.initFlow("poi", noise_intensity=0.1)
        ch.updateBoundVel(0)
        ch.attach_closure(cl)
        ch.step(2)
        if first == "closure":
            cl.close()
            ch.close()
        else:
            ch.close()
            change(cl, "train", data)
            assert np.all(np.isfinite(cl.params()))
            cl.close()
