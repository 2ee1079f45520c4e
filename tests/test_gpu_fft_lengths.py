"""The field stage at every kind of line length: 2^a lines, whose threads have equal shares, and 3 2^a lines, whose
threads have one butterfly more or less, from one thread per line up; against the oracle on the same Philox modes.
Bars: FP64 1e-12 of each field's largest value; FP32 1e-5 of its rms (those of test_gpu_parity.py)."""
import numpy as np
import pytest

import crime_amd
import oracle
from conftest import small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8, 12, 16, 24, 48, 64, 96, 192])
@pytest.mark.parametrize("precision", ["double", "single"])
def test_fields_vs_oracle(cfgdir, n, precision):
    par = small_params(cfgdir, f"fft_{n}_{precision}", n_grid=n, precision=precision, n_side=4, n_nu=4)
    dens, vpot, s2, _ = oracle.fields(par.desc())
    with crime_amd.GetHI(par) as gh:
        st = gh.create_d_and_vr_fields()
        got = {crime_amd.GRID_DENS: dens, crime_amd.GRID_VPOT: vpot}
        for which, ref in got.items():
            err = np.abs(gh.grid(which) - ref).max()
            assert err < (1e-12 * np.abs(ref).max() if precision == "double" else 1e-5 * np.sqrt(np.mean(ref ** 2)))
        assert abs(st["sigma2_gauss"] - s2) < (1e-12 if precision == "double" else 1e-5) * s2
