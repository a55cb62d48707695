"""bench.py's bytes per cell-step, by solver and V-cycles counted."""
import bench


def test_bytes_per_cell_step():
    assert bench.step_bytes("fp64", True, 0.0) == bench.step_bytes("mixed", True, 0.0) == (0, 392)
    assert bench.step_bytes("fp64", False, 1.5) == (2.5, 312 + 352 * 2.5)
    assert bench.step_bytes("mixed", False, 1.0) == (2.0, 312 + 256 * 2.0)
    # V-cycle solves whose predictor has decayed to no cycle before the first
    # test still run the one after it
    assert bench.step_bytes("fp64", False, 0.0) == (1.0, 312 + 352)
    assert bench.step_bytes("mixed", False, 0.25) == (1.25, 312 + 256 * 1.25)
