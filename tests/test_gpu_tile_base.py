"""The base activator's kernels -- FLOAT and INT sources, and BIT sources
through a spike plane -- against a serial FP32 sum in visit order
(activate_base, synapse_kernel.h:887-912), through the C-ABI of
libsg_hip.so.

Sizes sit where the kernels can go wrong: destinations around 16 and 64 (the
destinations of a block) and around the rules' lines (64, 512, 1024 and 2048
tiles), visits around the batches and chunks (8, 64, 512), arbors that leave
the source layer, rectangles off the layer's origin, padded visit lists.
Every sum runs in the serial order, so the comparison is bit for bit.
"""

import ctypes

import numpy as np
import pytest

from test_zz_no_alloc import (ADD, CONV, FC, OUT_FLOAT, Conn, _lib, _tiled)

OUT_BIT, OUT_INT, SUB = 1, 2, 1
SUBSET, DIV, SPARSE = 1, 4, 5

FULL = [(1, 1), (3, 15), (8, 16), (64, 17), (65, 63), (511, 65), (512, 64),
        (513, 10), (1100, 33), (100, 64 * 64), (70, 64 * 64 + 1),
        # few visits in many tiles: a lane each, or not
        (16, 64 * 512), (16, 64 * 512 + 1), (17, 64 * 512 + 1),
        (32, 64 * 2048), (33, 64 * 2048), (1, 64 * 2048 + 1)]

# rows, columns, field, stride, wrap, offset, shared kernel
ARBOR = [(1, 1, 3, 1, True, -1, False), (9, 7, 3, 1, False, -1, False),
         (30, 33, 5, 1, False, -2, False), (13, 13, 9, 2, True, -4, False),
         (64, 64, 9, 1, True, -4, False), (65, 63, 3, 1, True, -1, True),
         (256, 256, 3, 1, False, -1, False),
         (257, 256, 3, 1, True, -1, True), (128, 96, 7, 1, True, -3, False),
         (128, 257, 9, 1, False, -4, False), (129, 256, 9, 1, True, -4, False),
         (256, 256, 9, 1, True, -4, False), (256, 256, 6, 1, True, -3, False),
         (360, 300, 7, 1, False, -3, False), (410, 400, 9, 1, True, -4, True),
         (192, 180, 4, 1, False, -2, False)]


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


def _sources(rng, n, out):
    """Source words of a layer, and the values they show."""
    if out == OUT_BIT:
        bits = rng.random(n) < 0.3
        return bits.astype(np.uint32) << 31, bits.astype(np.float32)
    x = rng.standard_normal(n).astype(np.float32)
    return x, x


def _trunc(a, b):
    """C division."""
    return np.sign(a) * (np.abs(a) // b)


# rows, columns, field, stride, wrap, offset: up to 64 tiles with 81 and 625
# visits, 520, 1032 (25 visits) and 2064 tiles
DIVERGENT = [(13, 11, 9, 1, True, -4), (20, 22, 18, 2, False, -8),
             (24, 24, 25, 1, True, -12), (130, 256, 9, 1, False, -4),
             (128, 129, 10, 2, False, -4), (129, 256, 18, 2, True, -8)]


@pytest.mark.gpu
@pytest.mark.parametrize("out", [OUT_FLOAT, OUT_BIT])
@pytest.mark.parametrize("rows,cols,field,stride,wrap,offset", DIVERGENT)
def test_divergent(rows, cols, field, stride, wrap, offset, out):
    print("divergent", rows, cols, field, stride, wrap, out, flush=True)
    rng = np.random.default_rng(rows * 31 + field)
    to_rows, to_cols = rows * stride, cols * stride
    n = to_rows * to_cols
    words, src = _sources(rng, rows * cols, out)
    span = (field - stride) // stride + 1       # sources along an axis
    K = span * span
    w = rng.standard_normal((n, K)).astype(np.float32)
    before = rng.standard_normal(n).astype(np.float32)
    k = np.arange(K)
    # synapse_kernel.h:506-550: the first source by C division
    shift = -offset - field + stride
    r = _trunc(np.arange(to_rows) + shift, stride)[:, None] + k // span
    q = _trunc(np.arange(to_cols) + shift, stride)[:, None] + k % span
    r = np.repeat(r, to_cols, 0)
    q = np.tile(q, (to_rows, 1))
    inside = (r >= 0) & (r < rows) & (q >= 0) & (q < cols)
    x = src[(r % rows) * cols + q % cols]
    W = w
    if not wrap:
        x, W = np.where(inside, x, 0), np.where(inside, W, 0)
    c = Conn(type=DIV, opcode=ADD, out_type=out, from_size=rows * cols,
             from_rows=rows, from_cols=cols, to_size=n, to_rows=to_rows,
             to_cols=to_cols, row_field=field, col_field=field,
             row_stride=stride, col_stride=stride, row_spacing=1,
             col_spacing=1, row_offset=offset, col_offset=offset,
             wrap=int(wrap), k_per_dest=K, num_dest=n, num_weights=n * K)
    got = _run(c, words, _tiled(w, n, K), n, before)
    _same(got, before + _serial(x, W))


# source layer and rectangle (rows, columns, ends), destinations' likewise
RECTANGLES = [((40, 30), (3, 37, 5, 29), (20, 50), (2, 19, 7, 48)),
              ((9, 8), (1, 8, 2, 8), (300, 250), (10, 290, 5, 250)),
              ((12, 9), (1, 11, 1, 9), (400, 360), (5, 395, 1, 359))]


@pytest.mark.gpu
@pytest.mark.parametrize("out", [OUT_FLOAT, OUT_BIT])
@pytest.mark.parametrize("size,rect,to,to_rect", RECTANGLES)
def test_subset(size, rect, to, to_rect, out):
    print("subset", size, rect, to, to_rect, out, flush=True)
    rng = np.random.default_rng(size[0])
    words, src = _sources(rng, size[0] * size[1], out)
    x = src.reshape(size)[rect[0]:rect[1], rect[2]:rect[3]].reshape(-1)
    at = np.arange(to[0] * to[1]).reshape(to)[
        to_rect[0]:to_rect[1], to_rect[2]:to_rect[3]].reshape(-1)
    n, K = at.size, x.size
    w = rng.standard_normal((n, K)).astype(np.float32)
    before = rng.standard_normal(to[0] * to[1]).astype(np.float32)
    c = Conn(type=SUBSET, opcode=ADD, out_type=out,
             from_size=size[0] * size[1], from_rows=size[0],
             from_cols=size[1], to_size=to[0] * to[1], to_rows=to[0],
             to_cols=to[1], from_row_start=rect[0], from_row_end=rect[1],
             from_col_start=rect[2], from_col_end=rect[3],
             to_row_start=to_rect[0], to_row_end=to_rect[1],
             to_col_start=to_rect[2], to_col_end=to_rect[3], k_per_dest=K,
             num_dest=n, num_weights=n * K)
    got = _run(c, words, _tiled(w, n, K), n, before)
    want = before.copy()
    want[at] = want[at] + _serial(np.broadcast_to(x, w.shape), w)
    _same(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("out", [OUT_FLOAT, OUT_BIT])
@pytest.mark.parametrize("n_from,n,K", [(500, 697, 600), (200, 65601, 40),
                                        (300, 131100, 70), (90, 66000, 70),
                                        (90, 33000, 16), (70, 131073, 30)])
def test_sparse(n_from, n, K, out):
    import torch
    print("sparse", n_from, n, K, out, flush=True)
    rng = np.random.default_rng(n)
    words, src = _sources(rng, n_from, out)
    counts = rng.integers(0, K + 1, n)
    counts[0] = K
    used = np.arange(K) < counts[:, None]
    from_ = np.where(used, rng.integers(0, n_from, (n, K)), -1).astype(
        np.int32)
    w = np.where(used, rng.standard_normal((n, K)), 0).astype(np.float32)
    before = rng.standard_normal(n).astype(np.float32)
    pad = np.full((-(-n // 64) * 64, K), -1, np.int32)
    pad[:n] = from_
    table = torch.from_numpy(np.ascontiguousarray(
        pad.reshape(-1, 64, K).transpose(0, 2, 1)).reshape(-1)).cuda()
    c = Conn(type=SPARSE, opcode=ADD, out_type=out, from_size=n_from,
             from_rows=1, from_cols=n_from, to_size=n, to_rows=1, to_cols=n,
             k_per_dest=K, num_dest=n, num_weights=n * K)
    c.sparse_from = table.data_ptr()
    got = _run(c, words, _tiled(w, n, K), n, before)
    x = np.where(used, src[np.maximum(from_, 0)], 0).astype(np.float32)
    _same(got, before + _serial(x, w))
