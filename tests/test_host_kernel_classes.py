"""The kernel-timing classes, on the CPU build of tests/host_mock (launches are counted)."""

import ctypes

import pytest

from meep_amd import capi
from meep_amd.capi import Ez, fields, gaussian_src_time, structure


@pytest.fixture(scope="module")
def host_lib():
    from host_mock import build
    lib = capi.bind(ctypes.CDLL(build.build()))
    lib.mock_fast_launches.restype = lib.mock_step2d_launches.restype = ctypes.c_long
    return lib


def cell(lib):
    s = structure(lib, dim=2, size=(6.0, 5.0), a=10, pml=capi.pml(0.5)[:4])
    f = fields(s)
    f.use_real_fields()
    f.add_volume_source(Ez, gaussian_src_time(0.6, 0.6), (3.0, 2.0, 0), (3.0, 2.0, 0))
    f.step()
    return s, f


def classes(f, *which):
    return [f.kernel_timing(k)[1] for k in which]


def test_the_interior_class_times_the_interior_alone(host_lib):
    """One step: an interior launch a phase in the interior classes and the slabs' launch beside it
    (without timing they are one launch)."""
    s, f = cell(host_lib)
    before = host_lib.mock_fast_launches()
    f.step()
    assert host_lib.mock_fast_launches() - before == 2
    f.set_kernel_timing(True)
    f.reset_kernel_timing()
    before = host_lib.mock_fast_launches()
    f.step()
    assert host_lib.mock_fast_launches() - before == 4
    assert classes(f, capi.K_STEP_BH, capi.K_STEP_DE, capi.K_BH_INTERIOR, capi.K_DE_INTERIOR) == [1, 1, 1, 1]


def test_steps_of_the_tile_kernel_are_a_class_of_their_own(host_lib):
    s, f = cell(host_lib)
    f.step_n(40)
    f.set_kernel_timing(True)
    f.reset_kernel_timing()
    before = host_lib.mock_step2d_launches()
    f.step_n(32)
    tiles = host_lib.mock_step2d_launches() - before
    assert tiles == 4
    assert classes(f, capi.K_TILE2D, capi.K_STEP_BH, capi.K_STEP_DE, capi.K_DE_INTERIOR) == [tiles, 0, 0, 0]
    with pytest.raises(capi.MeepError):
        f.kernel_timing(capi.K_TILE2D + 1)
