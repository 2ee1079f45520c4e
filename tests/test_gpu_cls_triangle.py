"""Cross spectra of 65 to 256 maps on both sides of the lines between their two kernels (80 maps from 48 l, 128 from 160,
256 from 176, ...), with several groups of 16 l for each XCD, a last group that is not whole, and several sets; every
[a][b][l] against sums over the alms, to 1e-13 of the largest value (the bar of test_gpu_sht_tiles.py).

The smaller spectra do not pay for the larger ones' kernel: those of 256 maps at 48 l, a sixteenth of the products at
192 l, take at most a third of their time (a half, with one workgroup to an l)."""
import numpy as np
import pytest
import torch

import crime_amd

pytestmark = pytest.mark.gpu


def maps_of(n, nside, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    m = torch.randn((n, 12 * nside ** 2), generator=g, device="cuda", dtype=torch.float64)
    torch.cuda.synchronize()
    return m


def cross(alm, lmax):
    out = np.zeros((len(alm), len(alm), lmax + 1))
    for l in range(lmax + 1):
        a = alm[:, [crime_amd.alm_index(l, m, lmax) for m in range(l + 1)]]
        x = np.concatenate([a[:, :1].real, np.sqrt(2.0) * a[:, 1:].real, np.sqrt(2.0) * a[:, 1:].imag], axis=1)
        out[:, :, l] = x @ x.T / (2 * l + 1.0)
    return out


@pytest.mark.parametrize("n, lmax", [(65, 46), (65, 47), (80, 150), (81, 79), (112, 95), (128, 158), (128, 159), (129, 127),
                                     (160, 143), (177, 191), (208, 159), (256, 174), (256, 175)])
def test_cross_spectra(n, lmax):
    m = maps_of(n, 48, n + lmax)
    with crime_amd.Sht(48, lmax, max_maps=n) as sh:
        alm = sh.map2alm_device(m.data_ptr(), n, True)
        cl = sh.anafast_device(m.data_ptr(), n, True)
    want = cross(alm, lmax)
    assert np.abs(cl - want).max() < 1e-13 * np.abs(want).max()
    assert np.array_equal(cl, cl.transpose(1, 0, 2))


@pytest.mark.parametrize("nsets, mps, lmax", [(2, 66, 130), (3, 100, 47), (3, 100, 111), (2, 200, 160)])
def test_sets_of_many_maps(nsets, mps, lmax):
    nside = 48
    m = maps_of(nsets * mps, nside, lmax)
    step = 8 * mps * 12 * nside ** 2
    with crime_amd.Sht(nside, lmax, max_maps=nsets * mps) as sh:
        alm = sh.map2alm_device(m.data_ptr(), nsets * mps, True)
        cl = sh.cls_sets_device([m.data_ptr() + step * s for s in reversed(range(nsets))], mps, True)
    for s in range(nsets):
        want = cross(alm[s * mps:(s + 1) * mps], lmax)
        assert np.abs(cl[nsets - 1 - s] - want).max() < 1e-13 * np.abs(want).max()


def test_few_l_take_little_time():
    m = maps_of(256, 64, 1)
    ms = {}
    for lmax in (47, 191):
        with crime_amd.Sht(64, lmax, max_maps=256) as sh:
            t = []
            for _ in range(8):
                sh.anafast_device(m.data_ptr(), 256, True, to_host=False)
                t.append(sh.stats()["ms_cls"])
            ms[lmax] = min(t)
    assert 3 * ms[47] < ms[191], ms
