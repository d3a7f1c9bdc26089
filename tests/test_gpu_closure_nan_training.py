"""A NaN or an infinity among the inputs of a training batch: a pre-activation that
is NaN, of either sign, counts as 0, so the loss and every gradient but the bad
feature's row of W1 are those of a sample whose first hidden layer is 0."""
import numpy as np
import pytest

import powerllel_channel_sycl_amd as pll
from oracle import pll_closure_oracle as mo
from test_gpu_closure import _data, _dev, _random_params

pytestmark = pytest.mark.gpu

FEATURE = 4
BAD = {"nan": np.float32(np.nan), "negative nan": -np.float32(np.nan), "infinity": np.float32(np.inf)}


@pytest.mark.parametrize("bad", sorted(BAD))
@pytest.mark.parametrize("row", [0, 31, 32, 99])
def test_gradient_with_a_bad_input(row, bad):
    print(f"CASE gradient with {bad} in row {row}", flush=True)
    n, p = 100, _random_params(3)
    w1 = p[mo.O_W1:mo.O_B1].reshape(16, 64)
    w1[FEATURE] = -np.abs(w1[FEATURE])  # an infinite feature closes every unit
    x, y = _data(n, 4)
    q = np.array(x)
    q[row, FEATURE] = BAD[bad]
    cl = pll.Closure(seed=1)
    cl.set_params(p)
    dx, dy = _dev(q), _dev(y)
    g, loss = cl.gradient(dx.data_ptr(), dy.data_ptr(), n)
    cl.close()
    # the other samples: the bad one made finite, with the label that it predicts
    y0 = y.astype(np.float64)
    y0[row] = mo.predict(p, x)[row]
    want, want_loss = mo.gradient(p, x, y0)
    # the bad one: h1 = 0, so h2 = relu(b2)
    h2 = mo.bf16(np.maximum(p[mo.O_B2:mo.O_W3], 0.0)).astype(np.float64)
    w3 = mo.bf16(p[mo.O_W3:mo.O_B3]).astype(np.float64)
    o = h2 @ w3 + float(p[mo.O_B3])
    d = np.logaddexp(0.0, o) - float(y[row])
    go = 2.0 * d / n / (1.0 + np.exp(-o))
    want[mo.O_W3:mo.O_B3] += h2 * go
    want[mo.O_B2:mo.O_W3] += np.where(h2 > 0, go * w3, 0.0)
    want[mo.O_B3] += go
    want_loss += d * d / n
    assert abs(loss - want_loss) <= 1e-4 * abs(want_loss)
    at = slice(mo.O_W1 + FEATURE * 64, mo.O_W1 + (FEATURE + 1) * 64)
    assert np.all(np.isnan(g[at]))  # the feature times a delta of 0
    g[at] = want[at] = 0.0
    for a, b in ((mo.O_W1, mo.O_B1), (mo.O_B1, mo.O_W2), (mo.O_W2, mo.O_B2), (mo.O_B2, mo.O_W3),
                 (mo.O_W3, mo.O_B3), (mo.O_B3, mo.N_PARAM)):
        err = np.linalg.norm(g[a:b] - want[a:b]) / np.linalg.norm(want[a:b])
        assert err < 2e-3, (a, err)
