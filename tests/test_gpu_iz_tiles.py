"""The E/I sheet at the line between sixteen and four wavefronts a tile (256
tiles of 64 destinations, a tile per CU), against the oracle: every spike,
voltage and plasticity array bit for bit."""

import pytest

import harness
import netdefs


@pytest.mark.gpu
@pytest.mark.parametrize("records", ["true", "false"])
@pytest.mark.parametrize("rows,cols", [(128, 128), (130, 128)])
def test_sheet_around_the_line(gpu_lib, rows, cols, records):
    from oracle import stepper
    print("iz tiles", rows, cols, records, flush=True)
    case = netdefs.iz_sheet(rows, cols, 5, "iz_tiles", noise=(6.0, 4.0),
                            workload=131)
    captures, finals, _ = harness.run_case(
        case, gpu_lib, {"compact records": records})
    assert stepper.check_case(case, captures, finals)
