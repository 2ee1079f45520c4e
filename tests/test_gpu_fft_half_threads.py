"""The field stage where FP32 lines take half the threads of FP64 ones (3 2^7 elements and more): FP32 fields against
FP64 fields of the same modes, in runs of cells at the start, the middle and the end of the box, and sigma^2.
Bar: 1e-5 of the field's rms, that of the FP32 fields against the oracle (test_gpu_fft_lengths.py)."""
import numpy as np
import pytest

import crime_amd
from conftest import small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [384, 768])
def test_fp32_fields_vs_fp64(cfgdir, n):
    m = 4 * n * n
    starts = (0, n ** 3 // 2 - 12345, n ** 3 - m)
    got, s2 = {}, {}
    for precision in ("double", "single"):
        par = small_params(cfgdir, f"half_{n}_{precision}", n_grid=n, precision=precision, n_side=4, n_nu=4)
        with crime_amd.GetHI(par) as gh:
            s2[precision] = gh.create_d_and_vr_fields()["sigma2_gauss"]
            got[precision] = [[gh.grid_range(w, c, m) for c in starts]
                              for w in (crime_amd.GRID_DENS, crime_amd.GRID_VPOT)]
    for ref, f in zip(got["double"], got["single"]):
        rms = np.sqrt(np.mean(np.concatenate(ref) ** 2))
        assert rms > 0
        for a, b in zip(ref, f):
            assert np.abs(a - b).max() < 1e-5 * rms
    assert abs(s2["single"] - s2["double"]) < 1e-5 * s2["double"]
