"""The rounding of a gradient's sums over many samples, against the FP64 sum of the
samples' own gradients.  With a power of two of samples each one's contribution is
exactly its own gradient divided by it, every BF16 rounding included."""
import numpy as np
import pytest

import powerllel_channel_sycl_amd as pll
from oracle import pll_closure_oracle as mo
from test_gpu_closure import _data, _dev, _random_params

pytestmark = pytest.mark.gpu


def test_gradient_sums_round_like_trees():
    """FP32 values rounded once differ by about 2.5e-8 rms (2^-24 at most); the waves'
    own sums and trees of the partials add less than as much again twice over.  A
    chain through a quarter of the 256 partials makes it 6.5-6.9e-8."""
    import torch
    print("CASE gradient sums", flush=True)
    m, n = 512, 1 << 18
    x, y = _data(m, 6)
    cl = pll.Closure(seed=1)
    cl.set_params(_random_params(5))
    dx, dy = _dev(x), _dev(y)
    own = np.stack([cl.gradient(dx[i:].data_ptr(), dy[i:].data_ptr(), 1)[0].astype(np.float64)
                    for i in range(m)])
    rng = np.random.default_rng(7)
    err = {"W1": [], "W2": []}
    for _ in range(6):
        idx = rng.integers(0, m, n)
        pick = _dev(idx)
        xs, ys = dx[pick].contiguous(), dy[pick].contiguous()
        torch.cuda.synchronize()
        g, _ = cl.gradient(xs.data_ptr(), ys.data_ptr(), n)
        want = (np.bincount(idx, minlength=m) / n) @ own
        for name, a, b in (("W1", mo.O_W1, mo.O_B1), ("W2", mo.O_W2, mo.O_B2)):
            err[name].append(np.linalg.norm(g[a:b] - want[a:b]) / np.linalg.norm(want[a:b]))
    cl.close()
    for name, e in err.items():
        rms = np.sqrt(np.mean(np.square(e)))
        print(f"  {name} {rms:.2e}", flush=True)
        assert rms < 6e-8
