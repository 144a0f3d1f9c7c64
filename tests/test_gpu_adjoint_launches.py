"""The reverse step's fused launches: objective monitors on both sides of the 1024 points that one
block takes, with averages of one, two and four points, both polarisations.  The gradient against
central differences of the engine's own FP64 runs at the largest pixel and one other, 1e-6 of the
largest value (truncation 1e-10, cancellation 5e-11 J over the step)."""

import numpy as np
import pytest

from meep_amd.capi import Ex, Ey, Ez, Hz, adjoint, fields, gaussian_src_time, pml, structure

pytestmark = pytest.mark.gpu

STEPS = 150
DESIGN = ((1.5, 1.0, 0.0), (2.5, 2.0, 0.0))


def build(lib, comp, mons, lo, hi, chi=None):
    rng = np.random.default_rng(7)
    s = structure(lib, dim=2, size=(4.0, 3.2), a=10, pml=pml(0.5))
    for c in ([Ez] if comp == Ez else [Ex, Ey]):
        s.set_chi1inv(c, 1.0 / rng.uniform(1.0, 4.0, size=s.shape))
    if chi is not None:
        s.set_chi1inv(comp, chi)
    f = fields(s)
    f.use_real_fields()
    f.add_volume_source(Ez if comp == Ez else Hz, gaussian_src_time(0.8, 0.6, start_time=-3.0), (0.9, 1.4, 0), (0.9, 1.4, 0))
    return s, f, f.add_dft_fields(mons, lo, hi, [0.7, 0.9], decimation_factor=1)


@pytest.mark.parametrize("comp,mons", [(Ez, [Ez]), (Ex, [Ex, Ey])], ids=["tm", "te"])
@pytest.mark.parametrize("lo,hi", [((3.0, 1.0, 0), (3.0, 1.0, 0)), ((0.6, 0.2, 0), (3.8, 3.1, 0)), ((0, 0, 0), (4.0, 3.2, 0))],
                         ids=["point", "near1024", "cell"])
def test_gradient(gpu_lib, comp, mons, lo, hi):
    print(f"[adjoint launches] comp={comp} {lo} {hi}", flush=True)

    def value(chi):
        _, f, mon = build(gpu_lib, comp, mons, lo, hi, chi)
        f.step_n(STEPS)
        return sum(float(np.sum(np.abs(mon.dft(i)) ** 2)) for i in range(mon.num_chunks()))

    s, f, mon = build(gpu_lib, comp, mons, lo, hi)
    adj = adjoint(f, mon, comp, *DESIGN)
    f.step_n(STEPS)
    g = adj.gradient()
    chi = s.get_chi1inv(comp)
    top = np.abs(g).max()
    assert top > 0
    for i, j in (np.unravel_index(np.argmax(np.abs(g)), g.shape), (2, 3)):
        at = (adj.box_lo[0] + i, adj.box_lo[1] + j)
        h = 1e-5 * chi[at]
        vals = []
        for sign in (1, -1):
            c2 = chi.copy()
            c2[at] += sign * h
            vals.append(value(c2))
        assert abs(g[i, j] - (vals[0] - vals[1]) / (2 * h)) <= 1e-6 * top
