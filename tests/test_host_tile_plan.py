"""When the tile kernel's plan of a 2D chunk is built, on the CPU build of tests/host_mock
(allocations and tile launches are counted; no kernel runs)."""

import ctypes

import numpy as np
import pytest

from meep_amd import capi
from meep_amd.capi import Ez, fields, gaussian_src_time, structure


@pytest.fixture(scope="module")
def host_lib():
    from host_mock import build
    lib = capi.bind(ctypes.CDLL(build.build()))
    lib.mock_malloc_count.restype = lib.mock_step2d_launches.restype = ctypes.c_long
    return lib


def cell(lib, npole=1, nx=40, ny=60):
    s = structure(lib, dim=2, size=(nx / 10, ny / 10), a=10, pml=capi.pml(0.3)[:4])
    s.set_chi1inv(Ez, np.full(s.shape, 0.5))
    for q in range(npole):
        s.add_susceptibility(lambda x, y, z: 1.0 if x < 2.0 else 0.0, 1.0 + q, 0.1)
    f = fields(s)
    f.use_real_fields()
    f.add_volume_source(Ez, gaussian_src_time(0.6, 0.6), (1.5, 2.0, 0), (1.5, 2.0, 0))
    f.add_dft_fields([Ez], (0, 0, 0), (nx / 10, ny / 10, 0), np.linspace(0.4, 0.8, 3), decimation_factor=1)
    return s, f


def counted(lib, call):
    a, t = lib.mock_malloc_count(), lib.mock_step2d_launches()
    call()
    return lib.mock_malloc_count() - a, lib.mock_step2d_launches() - t


def test_steps_alone_between_calls_keep_the_plan(host_lib):
    """A step taken alone swaps P and P_prev: the plan holds both orders.  What is allocated a
    call is its source rows."""
    s, f = cell(host_lib)
    f.step_n(40)
    f.step_n(40)
    _, base = counted(host_lib, lambda: f.step_n(8))
    assert base > 0
    for _ in range(3):
        f.step()
        for n in (2, 3, 8, 17):
            made, launches = counted(host_lib, lambda: f.step_n(n))
            assert made <= 2 and launches > 0, n


def test_new_sources_keep_buffers_and_monitor_tables(host_lib):
    s, f = cell(host_lib)
    f.step_n(40)
    for _ in range(3):
        f.add_volume_source(Ez, gaussian_src_time(0.5, 0.6), (2.5, 2.0, 0), (2.5, 2.0, 0))
        made, launches = counted(host_lib, lambda: f.step_n(4))
        assert made <= 5 and launches > 0  # source sets and rows, arguments


def test_a_short_first_call_steps_one_by_one(host_lib):
    """The plan is built once the steps asked for since the last change are worth it."""
    s, f = cell(host_lib)
    assert counted(host_lib, lambda: f.step_n(3))[1] == 0
    for _ in range(20):
        launches = counted(host_lib, lambda: f.step_n(3))[1]
    assert launches > 0
    f.add_dft_fields([Ez], (0, 0, 0), (1.0, 1.0, 0), [0.5], decimation_factor=1)
    assert counted(host_lib, lambda: f.step_n(3))[1] == 0
    assert counted(host_lib, lambda: f.step_n(60))[1] > 0


def test_a_batch_and_a_member_alone_keep_both_plans(host_lib):
    sims = [cell(host_lib, npole=q % 2, nx=40 + 9 * q) for q in range(3)]
    b = capi.batch([f for _, f in sims], use_graph=False, autotune=False)
    b.step_n(80)
    f = sims[1][1]
    f.step_n(60)
    f.step()
    b.step_n(4)
    for _ in range(2):
        f.step()  # swaps P and P_prev of this member
        made, launches = counted(host_lib, lambda: f.step_n(4))
        assert made <= 2 and launches > 0
        assert counted(host_lib, lambda: b.step_n(4))[1] > 0


def test_scenarios_plan_with_no_kernel_forced(host_lib):
    """Every scenario's default plan validates, the tile kernel's where it takes the cell."""
    from scenarios import SCENARIOS
    from test_gpu_tile_calls import PLAIN_2D
    for name in sorted(SCENARIOS):
        for single in (False, True):
            s, f, _ = SCENARIOS[name][0](host_lib, single=single)
            launches = counted(host_lib, lambda: f.step_n(30))[1]
            f.step()
            assert f.t == 31 and (launches > 0) == PLAIN_2D.get(name, False), name


def test_batches_of_2d_members_take_the_tile_kernel(host_lib):
    import test_gpu_tile_calls as TC
    sims = TC.members(host_lib, False)
    b = capi.batch([f for _, f, _ in sims], use_graph=False, autotune=False)
    seen = []
    TC.drive(sims, lambda n: seen.append((n, counted(host_lib, lambda: b.step_n(n))[1])))
    took = {n: t for n, t in seen}
    assert all(took[n] > 0 for n in (80, 3, 7, 70, 40)), seen


def test_a_first_short_call_makes_few_allocations(host_lib):
    """Beside the chunks' rings of deferred values and the source rows: nothing while the steps and
    chunks are few, one allocation for the grouped launches' tables after that."""
    s = structure(host_lib, dim=3, size=(2.0, 1.8, 1.6), a=8)
    f = fields(s)
    f.use_real_fields()
    f.add_volume_source(Ez, gaussian_src_time(0.6, 0.6), (1.0, 0.9, 0.8), (1.0, 0.9, 0.8))
    fl = [f.add_dft_flux(d, (0.4, 0.4, 0.4), hi, [0.5, 0.6], decimation_factor=1)
          for d, hi in ((0, (0.4, 1.4, 1.2)), (1, (1.6, 0.4, 1.2)), (2, (1.6, 1.4, 0.4)))]
    f.step()
    chunks = sum(m.num_chunks(w) for m in fl for w in (0, 1))
    assert counted(host_lib, lambda: f.step_n(2))[0] <= chunks + 1
    assert counted(host_lib, lambda: f.step_n(40))[0] <= 2


def test_a_batch_builds_its_members_plans_together(host_lib):
    """Second buffers and monitor tables of all members are one allocation each: what building costs
    does not grow with the members (a member's own rings of deferred values apart)."""
    made = []
    for count in (2, 12):
        sims = [cell(host_lib, npole=q % 2, nx=40 + 3 * q) for q in range(count)]
        b = capi.batch([f for _, f in sims], use_graph=False, autotune=False)
        b.step_n(2)  # the first step and the one-step plan
        n, launches = counted(host_lib, lambda: b.step_n(40))
        assert launches > 0
        made.append(n)
    assert made[0] == made[1], made
