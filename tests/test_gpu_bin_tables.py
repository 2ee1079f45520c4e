"""The map stage's LDS tables where a tile's samples occupy far more bins than a table holds (sums that find no slot go
to the maps), about as many, and few: every table against the FP64 maps scattered without one.  FP64 maps differ by the
order of at most 2^12 additions per bin (1e-12), FP32 maps by FP32 rounding (2e-5 of the largest, as elsewhere);
the fixed-point maps of every table are the same bits."""
import numpy as np
import pytest

import crime_amd
from conftest import small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["single", "double", "deterministic"])
@pytest.mark.parametrize("nside, sub, l_box", [(512, 4, 6000.0), (512, 0, 6000.0), (128, 3, 3000.0), (16, 3, 600.0)])
def test_tables_against_plain_scatter(cfgdir, kind, nside, sub, l_box):
    par = small_params(cfgdir, f"bins_{kind}_{nside}_{sub}", n_grid=32, n_side=nside, n_subcell=sub, l_box=l_box,
                       precision="single" if kind == "single" else "double",
                       extra=dict(deterministic=1) if kind == "deterministic" else None)
    with crime_amd.GetHI(par) as gh:
        first = None
        for v in range(4):
            gh.set_schedule([0, 0, 0, v])
            gh.run()
            m = gh.maps(np.float64)
            if kind == "deterministic":
                first = m if first is None else first
                assert np.array_equal(m, first), v
                continue
            ref = gh.reference_maps()
            assert np.count_nonzero(ref) > 100
            if kind == "double":
                assert np.all(np.abs(m - ref) <= 1e-12 * np.abs(ref)), v
            else:
                assert np.array_equal(m != 0, ref != 0)
                assert np.abs(m - ref).max() < 2e-5 * np.abs(ref).max(), v
