"""bench.py looks the measured HBM traffic of the kernels it reports up by name:
the headline's names are in profiles/traffic.json, with at least the bytes that
the kernel cannot do without."""
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("N", [5, 9])
@pytest.mark.parametrize("sweeps", ["FP64", "fp32 + 1 FP64 sweep(s)"])
def test_default_predictors_have_a_measured_traffic(N, sweeps):
    sys.path.insert(0, ROOT)
    import bench
    traffic = bench.measured_traffic(bench.predictor_name(N, sweeps, True), 81, N)
    assert traffic is not None
    assert traffic >= 0.95 * 81 ** 3 * 8 * 5 * (2 * (N + 1) ** 3 + 12 * (N + 1) ** 2)
