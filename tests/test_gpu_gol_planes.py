"""Game of life as bit planes (long runs of 0/1 kernels), bit for bit: the
engine's long runs against the oracle, and sg_hip_gol_planes against as many
steps of sg_hip_gol_steps.

Boards narrower than the halo, ragged last words (wrapping: put together at
the edges), rows off a multiple of four, other rules and kernels; run lengths
around the engine's line (128 steps) and its remainders; and both sides of
the rule for 16 or 8 steps a launch (4096 wavefronts).
"""

import ctypes

import numpy as np
import pytest

import harness
import netdefs
from test_zz_no_alloc import LIB

RUNS = [(20, 20, True, 129, "life", 401), (37, 45, False, 145, "wide", 402),
        (5, 3, True, 160, "life", 403), (66, 96, True, 128, "life", 404),
        (51, 101, True, 200, "wide", 405), (33, 64, False, 161, "01", 406),
        (1, 70, True, 150, "life", 407)]


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,wrap,steps,kind,seed", RUNS)
def test_long_runs(gpu_lib, rows, cols, wrap, steps, kind, seed):
    from oracle import stepper
    print("gol planes", rows, cols, wrap, steps, kind, flush=True)
    case = netdefs.gol("gol_planes_%d" % seed, rows, cols, steps, seed,
                       wrap=wrap)
    case.capture = []
    if kind == "wide":
        case.net["structures"][0]["layers"][0].update(
            {"survival_min": "1", "survival_max": "4", "birth_min": "3",
             "birth_max": "5"})
    elif kind == "01":
        case.weights = {"life": np.array([1, 0, 1, 1, 0, 1, 0, 1, 1],
                                         np.float32)}
    captures, finals, report = harness.run_case(case, gpu_lib)
    assert report.get("iterations") == str(steps)
    if steps > 128:      # 16 a launch, the two turns and the last steps
        planes = (steps - 1) // 16
        assert report.get("game of life launches") == str(
            planes + 2 + -(-(steps - 16 * planes) // 8))
    problems = stepper.compare(case, captures, finals)
    assert not problems, "\n".join(problems)


BOARDS = [(2048, 2048, 1, 32), (2048, 2050, 1, 32), (2049, 2048, 0, 16),
          (2100, 2111, 1, 48), (70, 33, 0, 64)]


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,wrap,steps", BOARDS)
@pytest.mark.parametrize("rule", [(2, 3, 3, 3), (1, 4, 3, 5)])
def test_planes_match_words(rows, cols, wrap, steps, rule):
    import torch
    print("gol planes and words", rows, cols, wrap, steps, flush=True)
    L = ctypes.CDLL(LIB)
    i, p = ctypes.c_int, ctypes.c_void_p
    L.sg_hip_gol_steps.argtypes = [p, p, p, i, i, i, p, i, i, i, i, i, p]
    L.sg_hip_gol_planes.argtypes = [p, p, p, i, i, i, p, i, i, i, i, i, p, p]
    L.sg_hip_gol_planes_bytes.argtypes = [p, i, i]
    L.sg_hip_gol_planes_bytes.restype = ctypes.c_long
    kernel = (ctypes.c_float * 9)(1, 1, 1, 1, 0, 1, 1, 1, 1)
    stream = torch.cuda.current_stream().cuda_stream
    gen = torch.Generator("cuda").manual_seed(rows + cols)
    words = torch.randint(-2 ** 31, 2 ** 31 - 1, (rows * cols,),
                          generator=gen, device="cuda",
                          dtype=torch.int64).to(torch.int32)
    planes = torch.empty(
        L.sg_hip_gol_planes_bytes(kernel, rows, cols) // 4,
        dtype=torch.int32, device="cuda")
    got = torch.empty_like(words)
    assert L.sg_hip_gol_planes(
        words.data_ptr(), got.data_ptr(), planes.data_ptr(), rows, cols, wrap,
        kernel, *rule, steps, None, stream) == 0
    a, b = words.clone(), torch.empty_like(words)
    for _ in range(0, steps, 8):
        assert L.sg_hip_gol_steps(a.data_ptr(), b.data_ptr(), None, rows,
                                  cols, wrap, kernel, *rule, 8, stream) == 0
        a, b = b, a
    assert torch.equal(a, got)
    # refused before any launch: too tall a board, another kernel
    assert L.sg_hip_gol_planes_bytes(kernel, 4 * 65535 + 1, 20) == 0
    assert L.sg_hip_gol_planes(
        words.data_ptr(), got.data_ptr(), planes.data_ptr(), 4 * 65535 + 1,
        1, wrap, kernel, *rule, 16, None, stream) != 0
    other = (ctypes.c_float * 9)(1, 2, 1, 1, 0, 1, 1, 1, 1)
    assert L.sg_hip_gol_planes_bytes(other, rows, cols) == 0
    assert L.sg_hip_gol_planes(
        words.data_ptr(), got.data_ptr(), planes.data_ptr(), rows, cols, wrap,
        kernel, *rule, 8, None, stream) != 0
