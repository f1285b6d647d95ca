"""The launch shape an ensemble gets by itself, on both sides of its rule's
lines (512 row tiles, a mean fan-in of 1024), against the shape of one
wavefront a row tile.

A row's sum is the same products in another grouping: FP32 accumulation over
up to 1056 terms of size 1/sqrt(1056) differs by far less than 1e-5 of the
largest state.
"""

import numpy as np
import pytest

from synaptogenesis_amd.ensemble import RateEnsemble

# widths, precision, the shape expected
SHAPES = [([[40, 4096, 4096]], "bf16", (1, 8)),      # 512 row tiles
          ([[40, 4096, 4097]], "bf16", (2, 4)),      # 513, long rows
          ([[33, 8192, 16], [17, 5, 3]], "bf16", (2, 2)),   # 515, short rows
          ([[31, 17, 3]], "bf16", (1, 8)),
          ([[100, 33, 65], [7, 1, 2]], "fp32", (8, 1))]


@pytest.mark.gpu
@pytest.mark.parametrize("widths,precision,shape", SHAPES)
def test_default_shape(widths, precision, shape):
    states = []
    for tile in (None, (4, 1)):
        e = RateEnsemble(widths, precision, leak=0.3)
        if tile is None:
            assert e.tile == shape
        else:
            e.set_tile(*tile)
        e.run(5)
        states.append([e.state(i, k) for i in range(len(widths))
                       for k in (1, 2)])
        e.close()
    for a, b in zip(*states):
        assert np.abs(a - b).max() <= 1e-5 * max(1e-3, np.abs(b).max())
