"""sg_hip_float_neurons: rate-encoding and relay layers of a list in one
launch, through the C-ABI of libsg_hip.so.

Lists of one layer, of a launch's worth (SG_MAX_FLOAT_BATCH = 32) and of one
more, with sizes around a block (256), empty layers and histories of several
registers.  Relay values are copies or a comparison, so exact; the rate unit
rounds an FP64 tanh once to FP32, and two FP64 libraries' tanh can round to
neighbouring floats: one ulp.
"""

import ctypes

import numpy as np
import pytest

from test_zz_no_alloc import LIB

RATE, RELAY, RAMP = 0, 1, 2
SIZES = [1, 255, 0, 256, 257, 1000, 64, 3]


class Layer(ctypes.Structure):
    _fields_ = [("size", ctypes.c_int), ("history", ctypes.c_int),
                ("model", ctypes.c_int), ("input", ctypes.c_void_p),
                ("output", ctypes.c_void_p)]


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, 2, 32, 33])
def test_layers_in_one_launch(count):
    import torch
    L = ctypes.CDLL(LIB)
    L.sg_hip_float_neurons.argtypes = [ctypes.POINTER(Layer), ctypes.c_int,
                                       ctypes.c_void_p]
    rng = np.random.default_rng(count)
    layers = (Layer * count)()
    keep = []
    for i in range(count):
        n, history = SIZES[i % len(SIZES)], 1 + i % 3
        x = rng.standard_normal(n).astype(np.float32)
        old = rng.standard_normal((history, n)).astype(np.float32)
        dx, dout = torch.from_numpy(x).cuda(), torch.from_numpy(old).cuda()
        layers[i] = Layer(n, history, i % 3, dx.data_ptr(), dout.data_ptr())
        keep.append((i % 3, x, old, dx, dout))
    assert L.sg_hip_float_neurons(
        layers, count, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    for model, x, old, _, dout in keep:
        got = dout.cpu().numpy()
        np.testing.assert_array_equal(got[1:], old[:-1])
        if model == RATE:
            want = np.where(x > 0, np.tanh(x.astype(np.float64)), 0.0)
            np.testing.assert_allclose(got[0], want.astype(np.float32),
                                       rtol=1.2e-7, atol=0)
        else:
            want = np.maximum(x, 0) if model == RAMP else x
            np.testing.assert_array_equal(got[0], want)
