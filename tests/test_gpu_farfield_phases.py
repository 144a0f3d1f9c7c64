"""Phases of the far-field kernel's frequency groups."""

import numpy as np
import pytest

from meep_amd.capi import Ez, X, Y, Z, fields, gaussian_src_time, structure

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nf,npts", [(3, 1), (5, 1), (5, 4200), (10, 2100), (7, 1)])
def test_groups_hold_each_frequencys_own_phase(gpu_lib, nf, npts):
    """Frequencies evenly spaced to a few ulps, far away: a group's fields are those of each
    frequency by itself.  Either phase carries the rounding of (cycles r), 2^-53 of 2 pi f r, the
    turned one a second of that size.  The second frequency is up to two ulps (2^-53) high, within
    what counts as even spacing: a phase that followed the first two frequencies alone would be off
    by up to 8 ulps of 2 pi r at the fifth."""
    print(f"[farfield] own phases nf={nf} npts={npts}", flush=True)
    d = 2.0 ** -5
    freqs = [0.5 + i * d for i in range(nf)]
    freqs[1] += (2 if nf <= 5 else 1) * 2.0 ** -53
    s = structure(gpu_lib, dim=3, size=(2.2, 2.2, 2.2), a=10, pml=[(q, side, 0.5) for q in (X, Y, Z) for side in (0, 1)])
    f = fields(s)
    cen = (1.1, 1.1, 0.9)
    f.add_volume_source(Ez, gaussian_src_time(0.6, 0.6, start_time=-4.0), cen, cen)
    box = [((0.8, 0.8, 1.4), (1.4, 1.4, 1.4), 1.0)]
    many = f.add_dft_near2far(box, np.asarray(freqs), decimation_factor=1)
    each = [f.add_dft_near2far(box, np.asarray([q]), decimation_factor=1) for q in freqs]
    f.step_n(80)
    r = 1e5
    if npts == 1:
        a = many.farfield((0.6 * r, 0.3 * r, 0.74 * r))
        b = np.concatenate([n.farfield((0.6 * r, 0.3 * r, 0.74 * r)) for n in each])
        a, b = np.asarray(a).reshape(-1), b.reshape(-1)
    else:  # points of a line
        lo, hi, res = (0.6 * r, 0.3 * r, 0.74 * r), (0.6 * r + npts - 1, 0.3 * r, 0.74 * r), 1.0
        a = many.get_farfields_array(lo, hi, res)[0]
        b = np.stack([n.get_farfields_array(lo, hi, res)[0][..., 0] for n in each], axis=-1)
    assert a.shape == b.shape and np.abs(b).max() > 0
    tol = 3 * 2 * np.pi * max(freqs) * r * 2.0 ** -53
    assert np.abs(a - b).max() <= tol * np.abs(b).max(), np.abs(a - b).max() / np.abs(b).max() / tol
