"""Point sources in fine pixels: the FP32 pixel screen's margins are fractions of a pixel that grow with Nside, so the
pixels of some 1e5 sources against the oracle's at the production Nside and beyond (counts exactly, the per-pixel terms to
1e-12 of their largest, the bars of test_gpu_psources.py)."""
import numpy as np
import pytest

import crime_amd
import oracle
from conftest import small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_side, n_grid, l_box", [(256, 32, 350.0), (512, 48, 350.0), (1024, 32, 400.0), (1000, 24, 300.0)])
def test_pixels_vs_oracle(cfgdir, n_side, n_grid, l_box):
    par = small_params(cfgdir, f"pspix_{n_side}", precision="double", n_grid=n_grid, n_side=n_side, n_nu=2, l_box=l_box)
    with crime_amd.GetHI(par) as gh:
        gh.run()
        st = gh.mk_psources_maps()
        a, b = gh.ps_pixel_sums()
        dens = gh.grid(crime_amd.GRID_DENS).ravel()
        dz = gh.grid(crime_amd.GRID_DZRSD).ravel()
        s2, _ = gh.sigma2()
    _, ra, rb, total = oracle.psources(par.desc(), dens, dz, s2, with_maps=False)
    print(f"\nNside {n_side}: {total} sources in {np.count_nonzero(ra)} pixels", flush=True)
    assert st["n_sources"] == total and total > 30000
    assert np.array_equal(a > 0, ra > 0)
    assert np.abs(a - ra).max() < 1e-12 * np.abs(ra).max()
    assert np.abs(b - rb).max() < 1e-12 * np.abs(rb).max()
