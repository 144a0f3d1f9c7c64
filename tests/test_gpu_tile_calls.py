"""The multi-step kernel of 2D chunks as programs reach it: scenarios with no kernel forced, calls
of changing lengths with single steps, new sources and new monitors between them, and batches of
2D members alone.  Against the oracle, at the bounds of test_gpu_parity.py (1e-10 of each array's
maximum in FP64, 1e-4 in FP32), and batches against single steps too."""

import numpy as np
import pytest

from meep_amd.capi import (K_TILE2D, Ex, Ey, Ez, Hz, X, Y, batch, fields, gaussian_src_time, linspace, pml, structure)
from scenarios import SCENARIOS, state
from test_gpu_step2d import build

pytestmark = pytest.mark.gpu


def same(a, b, single, what):
    tol = 1e-4 if single else 1e-10
    assert set(a) == set(b), (what, sorted(set(a) ^ set(b)))
    for key in sorted(b):
        scale = max(np.abs(b[key]).max(), 1e-30)
        assert np.abs(a[key] - b[key]).max() <= tol * scale, (what, key)


def accumulated(mon):
    """Every accumulator array of a flux or map monitor."""
    if hasattr(mon, "flux"):
        return {(w, i): mon.dft(w, i) for w in (0, 1) for i in range(mon.num_chunks(w))}
    return {i: mon.dft(i) for i in range(mon.num_chunks())}


def tile_launches(f, call):
    f.set_kernel_timing(True)
    f.reset_kernel_timing()
    call()
    n = f.kernel_timing(K_TILE2D)[1]
    f.set_kernel_timing(False)
    return n


# whether the kernel takes the scenario (not with conductivity or periodic halos)
PLAIN_2D = {"waveguide_2d": True, "metal_magnetic_2d_te": True, "conductive_2d_tm": False, "zone_edge_2d": False}


@pytest.mark.parametrize("single", [False, True], ids=["f64", "f32"])
@pytest.mark.parametrize("name", sorted(PLAIN_2D))
def test_scenarios_with_no_kernel_forced(gpu_lib, oracle_lib, name, single):
    builder, nsteps = SCENARIOS[name]
    print(f"[tile] {name} single={single}", flush=True)
    sg, fg, mg = builder(gpu_lib, single=single)
    assert (tile_launches(fg, lambda: fg.step_n(nsteps)) > 0) == PLAIN_2D[name]
    so, fo, mo = builder(oracle_lib, single=single)
    fo.step_n(nsteps)
    same(state(fg, sg, 2), state(fo, so, 2), single, name)
    for x, y in zip(mg, mo):
        same(accumulated(x), accumulated(y), single, name)


@pytest.mark.parametrize("single", [False, True], ids=["f64", "f32"])
@pytest.mark.parametrize("poles", [0, 1, 2])
@pytest.mark.parametrize("tm", [True, False], ids=["tm", "te"])
def test_calls_of_changing_lengths(gpu_lib, oracle_lib, tm, poles, single):
    """Single steps between calls swap P and P_prev, short calls make short launches, a new source
    or monitor changes the plan in mid-run."""
    print(f"[tile] calls tm={tm} poles={poles} single={single}", flush=True)
    calls = (1, 24, 2, 1, 3, 1, 1, 17, "source", 4, 1, 8, "monitor", 40, 5, 1, 2)
    out = []
    for lib in (gpu_lib, oracle_lib):
        s, f, fl, df = build(lib, 33, 70, tm, poles, single)
        mons = [fl, df]
        for n in calls:
            if n == "source":
                f.add_volume_source(Ez if tm else Ex, gaussian_src_time(0.7, 0.5, start_time=f.time() - 6.0), (1.4, 2.0, 0), (1.9, 2.3, 0))
            elif n == "monitor":
                mons.append(f.add_dft_flux(Y, (0.5, 4.1, 0), (2.8, 4.1, 0), linspace(0.5, 0.7, 2), decimation_factor=2))
            elif lib is gpu_lib:
                took = tile_launches(f, lambda: f.step_n(n))
                assert took > 0 if n > 1 else took == 0, (n, took)
            else:
                f.step_n(n)
        out.append((state(f, s, 2), [accumulated(m) for m in mons]))
    (a, ma), (b, mb) = out
    same(a, b, single, "state")
    for k, (x, y) in enumerate(zip(ma, mb)):
        same(x, y, single, k)


def members(lib, single):
    """2D cells of both polarisations with 0, 1 and 2 poles, one with complex fields, each with a
    flux line; the second is one odd number of steps ahead."""
    out = []
    for k, (tm, poles, real) in enumerate([(True, 0, True), (False, 1, True), (True, 2, True), (False, 0, False), (True, 1, True)]):
        size = (3.1 + 0.7 * k, 6.4 - 0.9 * k)
        rng = np.random.default_rng(50 + k)
        s = structure(lib, dim=2, size=size, a=10, pml=pml(0.4)[:4], single=single)
        ele = [Ez] if tm else [Ex, Ey]
        for c in ele:
            s.set_chi1inv(c, 1.0 / rng.uniform(1.0, 6.0, size=s.shape))
        if poles > 0:
            s.add_susceptibility(lambda x, y, z: 1.2 if 0.8 < x < 2.0 else 0.0, 1.0, 0.1, drude=True)
        if poles > 1:
            s.add_susceptibility(lambda x, y, z: 0.5 + 0.2 * y if 0.8 < y < 2.0 else 0.0, 0.9, 0.05)
        f = fields(s)
        if real:
            f.use_real_fields()
        at = (0.45 * size[0], 0.5 * size[1], 0.0)
        f.add_volume_source(Ez if tm else Hz, gaussian_src_time(0.5 + 0.03 * k, 0.6, start_time=-5.0), at, at, 1.0 + 0.5j)
        fl = f.add_dft_flux(X, (0.7 * size[0], 0.5, 0), (0.7 * size[0], size[1] - 0.5, 0), linspace(0.4, 0.8, 3 + k), decimation_factor=1)
        out.append((s, f, [fl]))
    out[1][1].step_n(7)
    return out


def drive(sims, step):
    """80 steps, calls of 2, 3, 7 and 40 with steps of single members and a late monitor between."""
    step(80)
    for n in (2, 3):
        step(n)
    sims[1][1].step()
    sims[2][1].step_n(3)
    step(7)
    s, f, mons = sims[2]
    mons.append(f.add_dft_flux(Y, (1.0, 2.5, 0), (2.4, 2.5, 0), linspace(0.5, 0.7, 2), decimation_factor=1))
    sims[0][1].add_volume_source(Ez, gaussian_src_time(0.6, 0.5, start_time=sims[0][1].time() - 5.0), (1.1, 1.5, 0), (1.4, 1.9, 0))
    step(2)
    step(70)
    sims[4][1].step_n(21)
    step(40)


def test_batches_of_2d_members(gpu_lib, oracle_lib):
    print("[tile] batch against the oracle", flush=True)
    together = members(gpu_lib, False)
    b = batch([f for _, f, _ in together], use_graph=False, autotune=False)
    drive(together, b.step_n)
    ref = members(oracle_lib, False)
    drive(ref, lambda n: [f.step_n(n) for _, f, _ in ref])
    for k, ((s1, f1, m1), (s2, f2, m2)) in enumerate(zip(together, ref)):
        assert f1.t == f2.t
        same(state(f1, s1, 2), state(f2, s2, 2), False, k)
        for x, y in zip(m1, m2):
            same(accumulated(x), accumulated(y), False, k)


@pytest.mark.parametrize("single", [False, True], ids=["f64", "f32"])
def test_batches_of_2d_members_against_single_steps(gpu_lib, single, monkeypatch):
    """The same against the chunks stepped alone by the one-step kernels, at the bounds of
    test_gpu_batch.py (1e-11, FP32 1e-5).  In FP32 the oracle is no sharper reference here: a
    Drude polarisation sums the rounding of every step, and the FP32 oracle's is 2.4e-4 of the
    largest value from the FP64 oracle's (so is the engine's: 2.3e-4)."""
    print(f"[tile] batch against single steps single={single}", flush=True)
    together = members(gpu_lib, single)
    b = batch([f for _, f, _ in together], use_graph=False, autotune=False)
    drive(together, b.step_n)
    monkeypatch.setenv("MEEP_AMD_NO_TILE2D", "1")
    alone = members(gpu_lib, single)
    drive(alone, lambda n: [f.step_n(n) for _, f, _ in alone])
    tol = 1e-5 if single else 1e-11
    for k, ((s1, f1, m1), (s2, f2, m2)) in enumerate(zip(together, alone)):
        assert f1.t == f2.t
        a, c = state(f1, s1, 2), state(f2, s2, 2)
        assert set(a) == set(c)
        for x, y in [(a, c)] + [(accumulated(x), accumulated(y)) for x, y in zip(m1, m2)]:
            for key in y:
                assert np.abs(x[key] - y[key]).max() <= tol * max(np.abs(y[key]).max(), 1e-30), (k, key)
