"""bench.py's account of what ran."""
import pytest


@pytest.mark.parametrize("tune,want", [
    ((1, 4, 50, 2, 1.0e6, 0), True), ((1, 4, 50, 1, 1.0e6, 0), False),   # the autotuner's
    ((1, 4, 50, -1), True), ((2, 8, 50, -1), False), ((2, 8, 50, 0), False)])  # --chem-tune
def test_jacobian_form(tune, want):
    import bench
    assert bench.closed_form(tune) is want
