"""The accuracy of a point source's two terms.  In a pixel with one source the ratio of the terms is 10 x^-0.65,
x = (1 + z) / 1000, whatever the source's luminosity and distance: each term is a power good to one rounding and at most
three products, so the ratio's distance from the oracle's gathers some ten roundings, each of rms 2^-53 / sqrt(3) at
most: 2.0e-16 in all.  Powers written as exponentials of a logarithm's multiple (ln x = -6.8, whose own rounding is 8 times
that of a number near 1) double it."""
import numpy as np
import pytest

import crime_amd
import oracle
from conftest import small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_side", [64, 256])
def test_ratio_of_the_terms(cfgdir, n_side):
    par = small_params(cfgdir, f"sed_{n_side}", precision="double", n_grid=32, n_side=n_side, n_nu=4,
                       l_box={64: 150.0, 256: 300.0}[n_side])
    with crime_amd.GetHI(par) as gh:
        gh.run()
        gh.mk_psources_maps()
        a, b = gh.ps_pixel_sums()
        dens = gh.grid(crime_amd.GRID_DENS).ravel()
        dz = gh.grid(crime_amd.GRID_DZRSD).ravel()
        s2, _ = gh.sigma2()
    _, ra, rb, total = oracle.psources(par.desc(), dens, dz, s2, with_maps=False)
    # most pixels hold one source; in those of several the ratio is a mean of theirs
    hit = np.flatnonzero(ra > 0)
    assert np.array_equal(hit, np.flatnonzero(a > 0))
    err = (b[hit] / a[hit]) / (rb[hit] / ra[hit]) - 1.0
    rms = np.sqrt(np.mean(err ** 2))
    print(f"\n{total} sources in {hit.size} pixels: rms {rms:.2e}, largest {np.abs(err).max():.2e}", flush=True)
    assert rms < 2.0e-16
