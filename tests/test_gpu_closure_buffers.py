"""A closure's device buffers are allocated when it is created: no gradient or
training step allocates, whatever its sample count, so none can fail half way."""
import numpy as np
import pytest

import powerllel_channel_sycl_amd as pll
from test_gpu_closure import _data, _dev

pytestmark = pytest.mark.gpu


def test_training_allocates_nothing():
    import torch
    print("CASE training allocates nothing", flush=True)
    x, y = (_dev(a) for a in _data(70_000, 3))  # more tiles than waves: the largest grid
    first = pll.Closure(seed=1)  # the kernels' own first-launch allocations
    first.gradient(x.data_ptr(), y.data_ptr(), len(y))
    first.train_step(x.data_ptr(), y.data_ptr(), len(y), 1e-3)
    first.synchronize()
    cl = pll.Closure(seed=1)
    cl.synchronize()
    free = torch.cuda.mem_get_info()[0]
    for n in (100, len(y), 33):
        g, loss = cl.gradient(x.data_ptr(), y.data_ptr(), n)
        assert np.all(np.isfinite(g)) and np.isfinite(loss)
        cl.train_step(x.data_ptr(), y.data_ptr(), n, 1e-3)
        cl.synchronize()
        assert torch.cuda.mem_get_info()[0] == free, n
    cl.close()
    first.close()
