"""The Izhikevich neuron update where no neuron of a wavefront has
conductances (its divisions left out), bit for bit against the oracle: plain
and odd wavefronts side by side, voltages whose square overflows, infinities,
NaN and zeros of both signs."""

import numpy as np
import pytest

import harness
import netdefs

VOLTAGES = [-65.0, -1e17, -1e19, -3e38, -np.inf, np.inf, np.nan, 0.0, -0.0,
            29.999, 30.0, 1e18, 1e-40]


@pytest.mark.gpu
@pytest.mark.parametrize("size", [1, 64, 130])
@pytest.mark.parametrize("conductance", [False, True])
def test_odd_voltages(gpu_lib, size, conductance):
    from oracle import stepper
    print("iz plain", size, conductance, flush=True)
    case = netdefs.iz_fc(size, 6, "iz_plain", workload=141)
    v = case.init[("izfc", "L1", "voltage")]
    v[:] = np.resize(np.array(VOLTAGES, np.float32), size)
    if size > 64:       # the first wavefront keeps to ordinary values
        v[:64] = -65.0
    if conductance:     # one neuron of the last wavefront
        for key in ("ampa", "nmda", "gabaa", "gabab"):
            g = np.zeros(size, np.float32)
            g[-1] = 0.25
            case.init[("izfc", "L1", key)] = g
    captures, finals, _ = harness.run_case(case, gpu_lib)
    problems = stepper.compare(case, captures, finals)
    assert not problems, "\n".join(problems)
