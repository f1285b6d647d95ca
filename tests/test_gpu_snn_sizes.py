"""The adjoint's kernels at sizes around their tiles, against the FP64 model
(oracle/snn.py).

The backward scan takes 256 hidden units a block, the products 16-byte rows
(inputs a multiple of 8, hidden units of 4) in tiles of 112, 128 and 256, the
output table 16 steps and 16 outputs.  Rate mode, whose gradient is smooth:
FP32 recurrences of up to 32 steps stay within 1e-4 of the largest entry
(an FP32 rounding, 6e-8, grown by the unit's slope of 12.5 and the steps).
"""

import numpy as np
import pytest

from synaptogenesis_amd import adjoint as adj
from test_gpu_snn import _case, _close, _oracle, _run

# batch, steps, inputs, hidden, outputs, checkpoint
SIZES = [(1, 12, 8, 1, 1, 4), (2, 16, 40, 63, 10, 16),
         (3, 32, 113, 255, 16, 16), (4, 12, 127, 257, 2, 3),
         (5, 20, 129, 260, 10, 10), (2, 12, 784, 500, 10, 6),
         (130, 12, 16, 513, 3, 12),
         # dW2 summed by 1, 2 and 6 slices of blocks beside dW1's product
         (409, 6, 8, 64, 5, 3), (410, 6, 8, 64, 5, 3),
         (700, 4, 120, 128, 16, 2)]


@pytest.mark.gpu
@pytest.mark.parametrize("batch,steps,n_in,n_hid,n_out,ck", SIZES)
def test_rate_gradients(batch, steps, n_in, n_hid, n_out, ck):
    print("case snn sizes", batch, steps, n_in, n_hid, n_out, ck, flush=True)
    cfg, x, w1, w2, labels = _case(adj.RATE, batch, steps, n_in, n_hid,
                                   n_out, ck, scale=1.5)
    loss, counts, g1, g2 = _run(cfg, x, w1, w2, labels)
    _, _, oloss, ocounts, d1, d2 = _oracle(cfg, x, w1, w2, labels)
    assert abs(loss - oloss) <= 1e-5 * max(1.0, abs(oloss))
    _close(counts, ocounts, 1e-5)
    if n_out == 1:      # one class: no gradient
        assert not np.any(g1) and not np.any(g2)
        return
    _close(g1, d1, 1e-4)
    _close(g2, d2, 1e-4)


@pytest.mark.gpu
@pytest.mark.parametrize("n_hid", [255, 256, 257])
def test_potentials_past_the_derivative(n_hid):
    """Potentials of 2e37 to 2e38, finite, whose 1 + slope |u| is not: the
    surrogate derivative there is 0 (in FP64 below 1e-75), in the hidden
    layer (one unit, from one step on) and in the output layer (one output,
    whose large weight comes from a unit that spikes at the first step).
    Spike mode: the bounds of test_gpu_snn.py."""
    print("case snn potentials past the derivative", n_hid, flush=True)
    cfg, x, w1, w2, labels = _case(adj.SPIKE, batch=3, steps=8, n_in=24,
                                   n_hid=n_hid, n_out=5, ck=4)
    x[:, :, 0] = 0
    x[2, 1, 0] = 1
    w1[7, 0] = 1e38             # row 1 of the batch, from step 2
    x[0, :, 1] = 1
    w1[9, 1] = 8
    w2[:, 9] = 0
    w2[2, 9] = 3e37             # every row, from step 0
    w1, w2 = (w.bfloat16().float() for w in (w1, w2))
    loss, counts, g1, g2 = _run(cfg, x, w1, w2, labels)
    _, _, oloss, ocounts, d1, d2 = _oracle(cfg, x, w1, w2, labels)
    assert np.array_equal(counts, ocounts)
    assert abs(loss - oloss) <= 1e-5 * abs(oloss)
    assert np.isfinite(g1).all() and np.isfinite(g2).all()
    _close(g1, d1, 1e-3)
    _close(g2, d2, 1e-3)
