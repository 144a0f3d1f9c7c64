"""Limits of the far-field kernel."""

import numpy as np
import pytest

from meep_amd.capi import Ez, green

pytestmark = pytest.mark.gpu


def test_distance_whose_square_overflows(gpu_lib, oracle_lib):
    """A 2D distance whose square overflows: the fields are zero, as the oracle's."""
    for x in ((1e200, 0, 0), (1e155, 1e155, 0)):
        print("[farfield]", x, flush=True)
        a = green(gpu_lib, 2, x, 0.5, 1.0, 1.0, (0, 0, 0), Ez)
        b = green(oracle_lib, 2, x, 0.5, 1.0, 1.0, (0, 0, 0), Ez)
        assert np.array_equal(a, b), (a, b)
