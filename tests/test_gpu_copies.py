"""sg_hip_copies_u32: copies of any length and alignment in one launch, into
device and mapped host memory, exact."""

import ctypes

import numpy as np
import pytest

from test_zz_no_alloc import LIB

LENGTHS = [1, 3, 4, 5, 255, 256, 257, 1000, 0, 4097, 70000, 2]


class Copy(ctypes.Structure):
    _fields_ = [("src", ctypes.c_void_p), ("dst", ctypes.c_void_p),
                ("n", ctypes.c_long)]


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, 2, 32, 33])
@pytest.mark.parametrize("shift", [0, 1])
def test_copies(count, shift):
    import torch
    L = ctypes.CDLL(LIB)
    L.sg_hip_copies_u32.argtypes = [ctypes.POINTER(Copy), ctypes.c_int,
                                    ctypes.c_void_p]
    rng = np.random.default_rng(count)
    copies, keep = (Copy * count)(), []
    for i in range(count):
        n = LENGTHS[i % len(LENGTHS)]
        a = torch.from_numpy(rng.integers(0, 2 ** 31, n + 8).astype(
            np.int32)).cuda()
        b = torch.zeros(n + 8, dtype=torch.int32, device="cuda")
        copies[i] = Copy(a.data_ptr() + 4 * shift, b.data_ptr() + 4, n)
        keep.append((n, a, b))
    assert L.sg_hip_copies_u32(
        copies, count, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    for n, a, b in keep:
        want = torch.zeros_like(b)
        want[1:1 + n] = a[shift:shift + n]
        assert torch.equal(b, want)
    bad = Copy(keep[0][1].data_ptr() + 2, keep[0][2].data_ptr(), 1)
    assert L.sg_hip_copies_u32(ctypes.byref(bad), 1, None) != 0
