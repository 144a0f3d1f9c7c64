"""The multi-step kernel of 2D chunks against the oracle.

Cells whose sizes meet the edges of the kernel's tiles (a core of 15 x 47 points: cells smaller
than a core, of exactly one or two cores, one point more, and uneven ones), both polarisations,
with uPML, walls, poles and long sources, over step counts that make one, two and several
launches, odd ones among them.  Bounds as in test_gpu_parity.py: 1e-10 of each array's maximum
in FP64 and 1e-4 in FP32, from rounding alone.
"""

import numpy as np
import pytest

from meep_amd.capi import (Dx, Dy, Dz, Ex, Ey, Ez, Hx, Hy, Hz, High, Low, X, Y, Magnetic, continuous_src_time, fields,
                           gaussian_src_time, linspace, pml, structure)
from scenarios import state

pytestmark = pytest.mark.gpu

A = 10.0


def build(lib, nx, ny, tm, poles, single, npml=3, walls=False, real=True):
    """nx x ny cells: random eps per cell, npml cells of uPML on every side (0: none), `poles`
    dispersive poles over part of the cell (the second with a graded sigma), a point current, a
    dipole line longer than a source table, a flux line, a decimated field map over the cell."""
    rng = np.random.default_rng([nx, ny, poles])
    size = (nx / A, ny / A)
    s = structure(lib, dim=2, size=size, a=A, pml=pml(npml / A)[:4] if npml else (), single=single)
    ele = [Ez] if tm else [Ex, Ey]
    for c in ele:
        s.set_chi1inv(c, 1.0 / rng.uniform(1.0, 6.0, size=s.shape))
    if poles > 0:
        s.add_susceptibility(lambda x, y, z: 1.2 if x > 0.3 * size[0] else 0.0, 1.0, 0.1, drude=True)
    if poles > 1:
        s.add_susceptibility(lambda x, y, z: 0.5 + 0.2 * y if y < 0.6 * size[1] else 0.0, 0.9, 0.05)
    f = fields(s)
    if real:
        f.use_real_fields()
    if walls:
        f.set_boundary(Low, X, Magnetic)
    cen = (0.52 * size[0], 0.47 * size[1], 0.0)
    f.add_volume_source(ele[0], gaussian_src_time(0.6, 0.6, start_time=-6.0), cen, cen, 1.0 + 0.5j)
    f.add_volume_source(Hx if tm else Hz, continuous_src_time(0.5, 1.0, start_time=-3.0), cen, cen, 0.3)
    f.add_volume_source(ele[-1], gaussian_src_time(0.5, 0.5, start_time=-8.0, is_integrated=True), (0.31, 0.0, 0.0),
                        (0.31, size[1], 0.0), 0.2)
    fl = f.add_dft_flux(X, (0.6 * size[0], 0.2, 0), (0.6 * size[0], size[1] - 0.2, 0), linspace(0.4, 0.8, 3), decimation_factor=1)
    df = f.add_dft_fields([ele[0], Dz if tm else Dy], (0, 0, 0), (size[0], size[1], 0), linspace(0.4, 0.8, 2), decimation_factor=3)
    return s, f, fl, df


def compare(gpu, oracle, nsteps, single, **kw):
    out = []
    for lib in (gpu, oracle):
        s, f, fl, df = build(lib, single=single, **kw)
        for n in nsteps:
            f.step_n(n)
        out.append((state(f, s, 2), fl, df))
    (a, fa, da), (b, fb, db) = out
    assert set(a) == set(b), sorted(set(a) ^ set(b))
    tol = 1e-4 if single else 1e-10
    for key in sorted(b):
        scale = max(np.abs(b[key]).max(), 1e-30)
        assert np.abs(a[key] - b[key]).max() <= tol * scale, key
    for which in (0, 1):
        for i in range(fb.num_chunks(which)):
            y = fb.dft(which, i)
            assert np.abs(fa.dft(which, i) - y).max() <= tol * max(np.abs(y).max(), 1e-30), ("flux", which, i)
    for i in range(db.num_chunks()):
        y = db.dft(i)
        assert np.abs(da.dft(i) - y).max() <= tol * max(np.abs(y).max(), 1e-30), ("map", i)


@pytest.mark.parametrize("single", [False, True], ids=["f64", "f32"])
@pytest.mark.parametrize("poles", [0, 1, 2])
@pytest.mark.parametrize("tm", [True, False], ids=["tm", "te"])
@pytest.mark.parametrize("nx,ny,npml", [(13, 17, 3), (14, 46, 3), (15, 47, 3), (29, 93, 4), (30, 94, 0), (61, 150, 5)])
def test_tile_edges(gpu_lib, oracle_lib, nx, ny, npml, tm, poles, single):
    print(f"[step2d] {nx}x{ny} tm={tm} poles={poles} single={single}", flush=True)
    compare(gpu_lib, oracle_lib, (1, 2, 3, 9, 16, 27), single, nx=nx, ny=ny, tm=tm, poles=poles, npml=npml)


@pytest.mark.parametrize("tm", [True, False], ids=["tm", "te"])
def test_magnetic_wall_and_complex_fields(gpu_lib, oracle_lib, tm):
    print(f"[step2d] walls, complex, tm={tm}", flush=True)
    compare(gpu_lib, oracle_lib, (1, 21, 8), False, nx=33, ny=50, tm=tm, poles=1, npml=3, walls=True, real=False)
