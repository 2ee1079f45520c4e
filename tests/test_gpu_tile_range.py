"""The map stage above 12000 tiles, where the host waits for the tile range and launches just its workgroups (the tests of
small grids launch every tile): a band out of the box's reach, for which nothing is launched, and a narrow band, whose maps
from the handle's stream equal, bit for bit under the deterministic scatter, those of a captured graph, which launches every
tile."""
import math

import numpy as np
import pytest

import crime_amd
from conftest import small_params

pytestmark = pytest.mark.gpu

STAGES = ("ms_maps_clear", "ms_pixelize", "ms_total")


@pytest.mark.parametrize("det", [0, 1])
def test_band_out_of_reach_above_the_range_wait(cfgdir, det):
    par = small_params(cfgdir, f"reach192_{det}", n_grid=192, n_side=16, n_nu=8, nu_lo=300.0, nu_hi=320.0, l_box=600.0,
                       precision="single", extra=dict(deterministic=det))
    with crime_amd.GetHI(par) as gh:
        for run in (gh.run, gh.mk_T_maps):
            st = run()
            assert all(math.isfinite(st[k]) and 0 <= st[k] < 1e3 for k in STAGES), st
            assert st["ms_maps_clear"] + st["ms_pixelize"] <= st["ms_total"] * (1 + 1e-9)
            assert not gh.maps(np.float64).any()


@pytest.mark.parametrize("precision", ["single", "double"])
def test_range_launch_equals_full_launch(cfgdir, precision):
    par = small_params(cfgdir, f"range192_{precision}", n_grid=192, n_side=32, n_nu=8, nu_lo=1330.0, nu_hi=1350.0,
                       l_box=900.0, precision=precision, extra=dict(deterministic=1))
    with crime_amd.GetHI(par) as gh:
        st = gh.run()
        assert all(math.isfinite(st[k]) and st[k] >= 0 for k in STAGES)
        own = gh.maps(np.float64)
        ref = gh.reference_maps()
        with crime_amd.Batch([gh], n_streams=1) as batch:
            for _ in range(3):
                batch.run()
                assert np.array_equal(gh.maps(np.float64), own)
    assert 0 < np.count_nonzero(own) and np.array_equal(own != 0, ref != 0)
    assert np.abs(own - ref).max() < (1e-6 if precision == "single" else 1e-12) * np.abs(ref).max()
