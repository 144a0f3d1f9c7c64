"""The FP32 row kernel's two group widths with poles, on both sides of the size where the launch
changes from 8-byte to 16-byte groups (2.6 million points of its box), rows of every remainder.
The whole cell radiates and every cell has its own eps, so all points are live after a step; FP32
bounds as in test_gpu_parity.py (1e-4 of each array's maximum)."""

import numpy as np
import pytest

from meep_amd.capi import Ex, Ey, Ez, Z, fields, gaussian_src_time, pml, structure
from scenarios import state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,poles", [((20, 18, 21), 1), ((20, 18, 22), 2), ((20, 18, 23), 2), ((140, 136, 141), 1), ((139, 138, 142), 2),
                                     ((138, 139, 143), 2), ((141, 137, 144), 1)])
def test_group_widths(gpu_lib, oracle_lib, n, poles):
    print(f"[row groups] {n} poles={poles}", flush=True)
    size = tuple(q / 10 for q in n)
    out = []
    for lib in (gpu_lib, oracle_lib):
        rng = np.random.default_rng(n)
        s = structure(lib, dim=3, size=size, a=10, pml=pml(0.4, Z), single=True)
        sig = rng.uniform(0.2, 0.8, size=s.shape)
        sig[:, :, : s.shape[2] // 3] = 0.0
        for c in (Ex, Ey, Ez):
            s.set_chi1inv(c, 1.0 / rng.uniform(1.0, 4.0, size=s.shape))
        for q in range(poles):
            i = s.add_susceptibility(None, 0.9 + 0.2 * q, 0.1)
            for c in (Ex, Ey, Ez):
                s.set_sigma(i, c, sig if q else np.where(sig > 0, 0.7, 0.0))
        f = fields(s)
        f.use_real_fields()
        f.add_volume_source(Ex, gaussian_src_time(0.6, 0.6, start_time=-4.0), (0, 0, 0), size)
        f.step_n(4)
        out.append(state(f, s, poles))
    a, b = out
    assert set(a) == set(b)
    for key in sorted(b):
        scale = max(np.abs(b[key]).max(), 1e-30)
        assert np.abs(a[key] - b[key]).max() <= 1e-4 * scale, key
