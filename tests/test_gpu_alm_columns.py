"""The widths of the alm GEMM's column tiles on both sides of their lines: one tile of up to five blocks of 16 columns (half a
block per map), or six from 800 l on; narrow tiles below 1024 rings, wide ones from there on.  A map's alms are the same bits
in every width and in a call of its own: each is one chain of products over the rings."""
import numpy as np
import pytest
import torch

import crime_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, nside, lmax", [(40, 24, 71), (41, 24, 71), (48, 208, 799), (48, 208, 800), (49, 208, 800),
                                            (64, 100, 140), (80, 24, 71), (96, 24, 71), (97, 24, 71), (128, 32, 60),
                                            (160, 24, 71), (200, 24, 71), (49, 500, 40), (49, 512, 40), (72, 512, 40),
                                            (80, 512, 40), (96, 512, 40)])
def test_widths_agree(n, nside, lmax):
    g = torch.Generator(device="cuda")
    g.manual_seed(n + nside)
    m = torch.randn((n, 12 * nside ** 2), generator=g, device="cuda", dtype=torch.float32)
    torch.cuda.synchronize()
    with crime_amd.Sht(nside, lmax, max_maps=n) as sh:
        alm = sh.map2alm_device(m.data_ptr(), n, False)
    with crime_amd.Sht(nside, lmax, max_maps=1) as one:
        for t in (0, n // 3, n - 1):
            ref = one.map2alm_device(m[t].data_ptr(), 1, False)[0]
            assert np.abs(ref).max() > 0 and np.array_equal(alm[t], ref), t
