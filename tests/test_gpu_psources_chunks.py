"""Point sources at the edges of the kernel's chunks of 512 sources per tile: cells that hold several chunks,
tiles that hold a handful of sources or none, grids that end inside a tile; against the oracle on the GPU's own
fields (the bars of test_gpu_psources.py: the number of sources exactly, the per-pixel terms to 1e-12)."""
import numpy as np
import pytest

import crime_amd
import oracle
from conftest import small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_grid, n_side, l_box", [(8, 4, 700.0), (12, 16, 500.0), (48, 32, 150.0), (24, 7, 900.0)])
def test_psources_chunks_vs_oracle(cfgdir, n_grid, n_side, l_box):
    par = small_params(cfgdir, f"psc_{n_grid}", precision="double", n_grid=n_grid, n_side=n_side, n_nu=8, l_box=l_box)
    with crime_amd.GetHI(par) as gh:
        gh.run()
        st = gh.mk_psources_maps()
        a, b = gh.ps_pixel_sums()
        dens = gh.grid(crime_amd.GRID_DENS).ravel()
        dz = gh.grid(crime_amd.GRID_DZRSD).ravel()
        s2, _ = gh.sigma2()
    _, ra, rb, total = oracle.psources(par.desc(), dens, dz, s2, with_maps=False)
    print(f"\n{n_grid}^3, box {l_box}: {total} sources, {total / n_grid ** 3:.2f} per cell", flush=True)
    assert st["n_sources"] == total
    assert np.abs(a - ra).max() < 1e-12 * np.abs(ra).max()
    assert np.abs(b - rb).max() < 1e-12 * np.abs(rb).max()
    assert np.array_equal(a > 0, ra > 0)
