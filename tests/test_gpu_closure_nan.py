"""A NaN among the inputs of a batch: its sample's hidden units count as 0 (a
pre-activation that is NaN is not above 0), and no other sample changes."""
import numpy as np
import pytest

import powerllel_channel_sycl_amd as pll
from test_gpu_closure import _close_to_oracle, _data, _dev, _random_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("row", [0, 31, 32, 99])
def test_predict_with_a_nan_input(row):
    import torch
    print(f"CASE predict with NaN in row {row}", flush=True)
    n, p = 100, _random_params(3)
    x, _ = _data(n, 4)
    cl = pll.Closure(seed=1)
    cl.set_params(p)
    out = []
    for bad in (False, True):
        q = np.array(x)
        if bad:
            q[row, 4] = np.nan
        dx = _dev(q)
        o = torch.empty(n, dtype=torch.float32, device="cuda:0")
        torch.cuda.synchronize()
        cl.predict(dx.data_ptr(), n, o.data_ptr())
        out.append(o.cpu().numpy())
    keep = np.arange(n) != row
    assert np.array_equal(out[0][keep], out[1][keep])
    bf = lambda a: torch.tensor(a).to(torch.bfloat16).to(torch.float64).numpy()  # noqa: E731
    o = 16 * 64 + 64 + 64 * 64
    b2, w3, b3 = p[o:o + 64], p[o + 64:o + 128], float(p[o + 128])
    z = float(bf(np.maximum(b2, 0.0)) @ bf(w3)) + b3
    _close_to_oracle(out[1][row:row + 1], np.array([np.logaddexp(0.0, z)], dtype=np.float32))
