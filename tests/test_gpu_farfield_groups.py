"""The far-field kernel's branches against the oracle: frequency groups of every size with and
without a remainder, uniform and uneven frequencies (phases by recurrence or one by one), 2D
distances on both sides of kr = 30 (library Bessel functions, asymptotic expansion), one-point
calls and planes of points (one or several segments of the currents).  The two sum the same terms
in different orders: 1e-10 of the largest value, as in test_gpu_near2far.py."""

import numpy as np
import pytest

from meep_amd.capi import Ex, Ez, Hz, X, Y, Z, fields, gaussian_src_time, structure

pytestmark = pytest.mark.gpu


def run(lib, dim, freqs):
    size = (3.0, 2.5, 2.2)[:dim] if dim == 3 else (3.0, 2.5)
    s = structure(lib, dim=dim, size=size, a=10, pml=[(d, side, 0.5) for d in (X, Y, Z)[:dim] for side in (0, 1)])
    f = fields(s)
    zc = 1.1 if dim == 3 else 0.0
    for c, x in ((Ez, 1.43), (Hz if dim == 2 else Ex, 1.62)):
        f.add_volume_source(c, gaussian_src_time(0.7, 0.6, start_time=-4.0), (x, 1.27, zc), (x, 1.27, zc))
    z0, z1 = (0.7, 1.5) if dim == 3 else (0.0, 0.0)
    box = [((0.9, 1.8, z0), (2.1, 1.8, z1), 1.0), ((2.1, 0.7, z0), (2.1, 1.8, z1), 1.0 + 0.25j),
           ((0.9, 0.7, z0), (2.1, 0.7, z1), -1.0), ((0.9, 0.7, z0), (0.9, 1.8, z1), -1.0)]
    n2f = f.add_dft_near2far(box, np.asarray(freqs), decimation_factor=1)
    f.step_n(120)
    pts = [(1.5, 4.0, zc), (4.5, -2.0, 0.3 * zc), (1.5, 9.0, zc), (-40.0, 21.0, 3 * zc)]
    one = np.array([n2f.farfield(p) for p in pts])
    near, _ = n2f.get_farfields_array((-2.0, 5.0, 0.0), (5.0, 5.0, zc), 2.0)
    far, _ = n2f.get_farfields_array((-9.0, 30.0, 0.0), (9.0, 30.0, 0.0), 9.0)
    return one, near, far


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("nf,even", [(1, True), (2, True), (3, True), (4, True), (5, True), (7, True), (10, True), (4, False), (5, False)])
def test_groups(gpu_lib, oracle_lib, dim, nf, even):
    print(f"[farfield] dim={dim} nf={nf} even={even}", flush=True)
    freqs = np.linspace(0.5, 0.9, nf) if even else 0.5 + 0.4 * np.linspace(0.0, 1.0, nf) ** 2
    for k, (g, w) in enumerate(zip(run(gpu_lib, dim, freqs), run(oracle_lib, dim, freqs))):
        scale = np.abs(w).max()
        assert g.shape == w.shape and scale > 0, k
        assert np.abs(g - w).max() <= 1e-10 * scale, (k, np.abs(g - w).max() / scale)
