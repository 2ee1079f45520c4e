"""P(k)'s kz pass of columns and mirrors at the edges of its tiles: grids of one radix pass, columns that no full tile
divides (12, 24), the shortest and longer lines, and more shells than the smaller LDS histogram holds.

Bars as in test_gpu_power.py: counts exact, mean |k| to 1e-12, P to 1e-10 (FP64) or 1e-4 (FP32) of numpy's.  Shells
narrower than the fundamental mode hold as few as 6 modes, whose power can be a tenth of the mean that the FP32 bar
is relative to: 1e-3 there.
"""
import numpy as np
import pytest

import crime_amd
import oracle
from conftest import small_params
from pk_ref import pk_numpy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,prec,width", [(8, "double", 1.0), (12, "double", 1.0), (12, "single", 1.0), (16, "double", 1.0),
                                          (24, "single", 1.0), (64, "double", 0.1), (64, "single", 0.1),
                                          (128, "double", 1.0), (192, "single", 0.25), (192, "single", 3.0)])
def test_pk_column_pairs(cfgdir, n, prec, width):
    par = small_params(cfgdir, f"pkcol_{n}_{prec}_{width}", n_grid=n, precision=prec, l_box=800.0)
    d = par.desc()
    w = width * 2 * np.pi / d.l_box
    nb = int(np.ceil(np.sqrt(3.0) * n / 2 / width)) + 1
    with crime_amd.GetHI(par) as gh:
        gh.create_d_and_vr_fields()
        k, pk, cnt = gh.power_spectrum(nb, w)
    ek, epk, ecnt = pk_numpy(oracle.fields(d)[0], d.l_box, nb, w)
    assert cnt.sum() == n ** 3
    assert np.array_equal(cnt, ecnt)
    assert np.allclose(k, ek, rtol=1e-12, atol=0)
    sel = ecnt > 0
    sel[0] = False   # holds k = 0, the rounding of a zero mean
    err = np.abs(pk[sel] - epk[sel]) / epk[sel]
    assert err.max() < (1e-10 if prec == "double" else 1e-4 if width >= 1 else 1e-3)
