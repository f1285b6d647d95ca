"""The base activator's kernels -- FLOAT and INT sources, and BIT sources
through a spike plane -- against a serial FP32 sum in visit order (activate_base, synapse_kernel.h:887-912), through
the C-ABI of libsg_hip.so.

Sizes sit where the kernels can go wrong: destinations around 16 and 64 (the
destinations of a block) and around the rules' lines (64 tiles, 1024 tiles),
visits around the batches and chunks (8, 64, 512), arbors that leave the
source layer.  Every sum runs in the serial order, so the comparison is bit
for bit.
"""

import ctypes

import numpy as np
import pytest

from test_zz_no_alloc import (ADD, CONV, FC, OUT_FLOAT, Conn, _lib, _tiled)

OUT_BIT, OUT_INT, SUB = 1, 2, 1

FULL = [(1, 1), (3, 15), (8, 16), (64, 17), (65, 63), (511, 65), (512, 64),
        (513, 10), (1100, 33), (100, 64 * 64), (70, 64 * 64 + 1)]

# rows, columns, field, stride, wrap, offset, shared kernel
ARBOR = [(1, 1, 3, 1, True, -1, False), (9, 7, 3, 1, False, -1, False),
         (30, 33, 5, 1, False, -2, False), (13, 13, 9, 2, True, -4, False),
         (64, 64, 9, 1, True, -4, False), (65, 63, 3, 1, True, -1, True),
         (256, 256, 3, 1, False, -1, False),
         (257, 256, 3, 1, True, -1, True), (128, 96, 7, 1, True, -3, False),
         (128, 257, 9, 1, False, -4, False), (129, 256, 9, 1, True, -4, False),
         (256, 256, 9, 1, True, -4, False)]


def _serial(x, w):
    """x, w [destinations][visits] float32: the sum in visit order."""
    total = np.zeros(len(x), np.float32)
    for k in range(x.shape[1]):
        total = total + x[:, k] * w[:, k]
    return total


def _run(c, host_src, weights, n, before):
    import torch
    if c.out_type == OUT_BIT:
        plane = torch.zeros((c.from_size + 63) // 64, dtype=torch.int64,
                            device="cuda")
        c.plane, c.skip_silent = plane.data_ptr(), 1
    src = torch.from_numpy(host_src.view(np.float32).copy()).cuda()
    w = torch.from_numpy(weights).cuda()
    dst = torch.from_numpy(before.copy()).cuda()
    c.src, c.weights, c.dst = src.data_ptr(), w.data_ptr(), dst.data_ptr()
    rc = _lib().sg_hip_activate_base(
        ctypes.byref(c), torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    return dst.cpu().numpy()


def _same(got, want):
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("n_from,n_to", FULL)
@pytest.mark.parametrize("out", [OUT_FLOAT, OUT_INT])
def test_fully_connected(n_from, n_to, out):
    rng = np.random.default_rng(n_from * 7919 + n_to)
    if out == OUT_FLOAT:
        src = rng.standard_normal(n_from).astype(np.float32)
        x = src
    else:
        src = rng.integers(0, 1000, n_from).astype(np.uint32)
        x = src.astype(np.float32)
    w = rng.standard_normal((n_to, n_from)).astype(np.float32)
    before = rng.standard_normal(n_to).astype(np.float32)
    c = Conn(type=FC, opcode=SUB, out_type=out, from_size=n_from,
             from_rows=1, from_cols=n_from, to_size=n_to, to_rows=1,
             to_cols=n_to, k_per_dest=n_from, num_dest=n_to,
             num_weights=n_from * n_to)
    got = _run(c, src, _tiled(w, n_to, n_from), n_to, before)
    _same(got, before - _serial(np.broadcast_to(x, w.shape), w))


# past 4096 sources, which a spike list takes
@pytest.mark.gpu
@pytest.mark.parametrize("n_from,n_to", [(4097, 65), (4100, 4160)])
def test_fully_connected_spikes(n_from, n_to):
    rng = np.random.default_rng(n_from)
    bits = rng.random(n_from) < 0.2
    w = rng.standard_normal((n_to, n_from)).astype(np.float32)
    before = rng.standard_normal(n_to).astype(np.float32)
    c = Conn(type=FC, opcode=SUB, out_type=OUT_BIT, from_size=n_from,
             from_rows=1, from_cols=n_from, to_size=n_to, to_rows=1,
             to_cols=n_to, k_per_dest=n_from, num_dest=n_to,
             num_weights=n_from * n_to)
    got = _run(c, bits.astype(np.uint32) << 31, _tiled(w, n_to, n_from),
               n_to, before)
    x = np.broadcast_to(bits.astype(np.float32), w.shape)
    _same(got, before - _serial(x, w))


@pytest.mark.gpu
@pytest.mark.parametrize("out", [OUT_FLOAT, OUT_BIT])
@pytest.mark.parametrize("rows,cols,field,stride,wrap,offset,shared", ARBOR)
def test_convergent(rows, cols, field, stride, wrap, offset, shared, out):
    rng = np.random.default_rng(rows * 31 + field)
    to_rows, to_cols = -(-rows // stride), -(-cols // stride)
    n, K = to_rows * to_cols, field * field
    if out == OUT_BIT:
        words = (rng.random(rows * cols) < 0.3).astype(np.uint32) << 31
        src = (words >> 31).astype(np.float32)
    else:
        src = words = rng.standard_normal(rows * cols).astype(np.float32)
    w = rng.standard_normal((1 if shared else n, K)).astype(np.float32)
    before = rng.standard_normal(n).astype(np.float32)
    k = np.arange(K)
    r = (np.arange(to_rows) * stride + offset)[:, None] + k // field
    q = (np.arange(to_cols) * stride + offset)[:, None] + k % field
    r = np.repeat(r, to_cols, 0)
    q = np.tile(q, (to_rows, 1))
    inside = (r >= 0) & (r < rows) & (q >= 0) & (q < cols)
    x = src[(r % rows) * cols + q % cols]
    W = np.broadcast_to(w, (n, K))
    if not wrap:
        # a skipped visit adds nothing: +0 leaves the sum's bits alone
        x, W = np.where(inside, x, 0), np.where(inside, W, 0)
    c = Conn(type=CONV, opcode=ADD, out_type=out,
             from_size=rows * cols, from_rows=rows, from_cols=cols,
             to_size=n, to_rows=to_rows, to_cols=to_cols, row_field=field,
             col_field=field, row_stride=stride, col_stride=stride,
             row_spacing=1, col_spacing=1, row_offset=offset,
             col_offset=offset, wrap=int(wrap), convolutional=int(shared),
             k_per_dest=K, num_dest=n, num_weights=K if shared else n * K)
    weights = w.reshape(-1) if shared else _tiled(w, n, K)
    got = _run(c, words, weights, n, before)
    _same(got, before + _serial(x, W))
