"""What the host code does when the device runs out of memory, on the CPU build of
tests/host_mock: an allocation of a chosen call fails, and the calls after it are checked."""

import ctypes

import numpy as np
import pytest

from meep_amd import capi
from meep_amd.capi import Ez, MeepError, fields, gaussian_src_time, structure


@pytest.fixture(scope="module")
def host_lib():
    from host_mock import build
    lib = capi.bind(ctypes.CDLL(build.build()))
    lib.mock_fail_malloc.argtypes = [ctypes.c_long]
    lib.mock_set_free.argtypes = [ctypes.c_size_t]
    lib.mock_malloc_count.restype = lib.mock_step2d_launches.restype = ctypes.c_long
    return lib


def test_far_fields_after_a_failed_allocation(host_lib):
    """A far-field call whose scratch cannot be allocated raises; the next one allocates it (the
    scratch outlives a call, and a launch with a buffer that was never allocated would write
    through a null pointer)."""
    for after in range(20):
        s = structure(host_lib, dim=2, size=(3.0, 2.5), a=10, pml=[(d, side, 0.5) for d in (0, 1) for side in (0, 1)])
        f = fields(s)
        f.add_volume_source(Ez, gaussian_src_time(0.7, 0.6), (1.4, 1.2, 0), (1.4, 1.2, 0))
        n2f = f.add_dft_near2far([((0.9, 1.8, 0), (2.1, 1.8, 0), 1.0)], [0.6, 0.7], decimation_factor=1)
        f.step_n(3)
        host_lib.mock_fail_malloc(after)
        failed = False
        try:
            n2f.get_farfields_array((-2.0, 5.0, 0), (5.0, 5.0, 0), 2.0)
        except MeepError as e:
            assert "far-field launch" not in str(e)
            failed = True
        host_lib.mock_fail_malloc(-1)
        out, _ = n2f.get_farfields_array((-2.0, 5.0, 0), (5.0, 5.0, 0), 2.0)
        assert np.all(np.isfinite(out))
        n2f.farfield((1.5, 9.0, 0))
        if not failed:
            break
    assert after >= 2 and not failed  # some allocation was made to fail, and the last pass reached none


def plain_2d(lib, nx=40, ny=60):
    s = structure(lib, dim=2, size=(nx / 10, ny / 10), a=10, pml=capi.pml(0.3)[:4])
    s.set_chi1inv(Ez, np.full(s.shape, 0.5))
    s.add_susceptibility(lambda x, y, z: 1.0 if x < 2.0 else 0.0, 1.0, 0.1)
    f = fields(s)
    f.use_real_fields()
    f.add_volume_source(Ez, gaussian_src_time(0.6, 0.6), (1.5, 2.0, 0), (1.5, 2.0, 0))
    f.add_dft_flux(0, (2.5, 1.0, 0), (2.5, 5.0, 0), np.linspace(0.4, 0.8, 3), decimation_factor=1)
    f.step()
    return s, f


def _raised(lib):
    """How many of the allocations of a step_n call raise when they fail; the call after one that
    raised, and the steps after one that did not, always go on."""
    n = 0
    for after in range(60):
        s, f = plain_2d(lib)
        lib.mock_fail_malloc(after)
        before = lib.mock_malloc_count()
        try:
            f.step_n(16)
            assert f.t == 17
        except MeepError as e:
            assert "internal" not in str(e)
            n += 1
        made = lib.mock_malloc_count() - before
        lib.mock_fail_malloc(-1)
        t = f.t
        f.step_n(16)
        f.step()
        assert f.t == t + 17
        if made <= after:
            return n
    raise AssertionError("every pass ran out of memory")


def test_second_buffers_that_do_not_fit(host_lib, monkeypatch):
    """A 2D chunk whose second buffers or tile tables cannot be allocated steps one by one: no
    allocation raises that does not raise without the tile kernel."""
    monkeypatch.setenv("MEEP_AMD_NO_TILE2D", "1")
    plain = _raised(host_lib)
    monkeypatch.delenv("MEEP_AMD_NO_TILE2D")
    assert _raised(host_lib) <= plain


def _allocations(lib, call):
    before = lib.mock_malloc_count()
    call()
    return lib.mock_malloc_count() - before


def test_second_buffers_leave_memory_free(host_lib, monkeypatch):
    """With less than an eighth of the device's memory left the chunk takes no second buffers."""
    host_lib.mock_set_free(36 << 30)
    try:
        s, f = plain_2d(host_lib)
        short = _allocations(host_lib, lambda: f.step_n(16))
    finally:
        host_lib.mock_set_free(256 << 30)
    s, f = plain_2d(host_lib)
    ample = _allocations(host_lib, lambda: f.step_n(16))
    monkeypatch.setenv("MEEP_AMD_NO_TILE2D", "1")
    s, f = plain_2d(host_lib)
    assert short == _allocations(host_lib, lambda: f.step_n(16)) < ample


@pytest.mark.parametrize("short", [False, True], ids=["3d_member", "memory"])
def test_batch_that_the_tile_kernel_does_not_take(host_lib, monkeypatch, short):
    """A batch with a member that the tile kernel does not take, or without the memory for its
    second buffers, steps all of its members one by one; no member allocates second buffers
    that the batch then does not use."""
    def run():
        sims = [plain_2d(host_lib, 40 + 7 * q, 50) for q in range(3)]
        if not short:
            s = structure(host_lib, dim=3, size=(1.2, 1.0, 1.0), a=10)
            f = fields(s)
            f.add_volume_source(Ez, gaussian_src_time(0.6, 0.6), (0.5, 0.5, 0.5), (0.5, 0.5, 0.5))
            f.step()
            sims.append((s, f))
        b = capi.batch([f for _, f in sims], use_graph=False, autotune=False)
        n = _allocations(host_lib, lambda: b.step_n(12))
        assert all(f.t == 13 for _, f in sims)
        return n
    if short:
        host_lib.mock_set_free(36 << 30)
    try:
        got = run()
    finally:
        host_lib.mock_set_free(256 << 30)
    monkeypatch.setenv("MEEP_AMD_NO_TILE2D", "1")
    assert got == run()


@pytest.mark.parametrize("interval", [0, 20], ids=["history", "checkpoints"])
def test_recording_that_runs_out_of_memory(host_lib, interval):
    """The tile kernel's state is where every reader looks after an even number of launches: an
    allocation of the reverse mode's recording that fails leaves it there, and the fields go on."""
    import adjoint_cases as AC
    for after in range(400):
        s, f, mon = AC.build(host_lib, AC.rho_grid())
        adj = capi.adjoint(f, mon, Ez, AC.DESIGN[0], AC.DESIGN[1], checkpoint_interval=interval)
        f.step_n(9)
        host_lib.mock_fail_malloc(after)
        before, launches = host_lib.mock_malloc_count(), host_lib.mock_step2d_launches()
        failed = False
        try:
            f.step_n(700 if interval == 0 else 60)
        except MeepError as e:
            assert "internal" not in str(e)
            failed = True
        made = host_lib.mock_malloc_count() - before
        host_lib.mock_fail_malloc(-1)
        assert (host_lib.mock_step2d_launches() - launches) % 2 == 0, after
        f.step_n(30)
        adj.gradient()
        if made <= after:
            break
    assert not failed and after >= 2
