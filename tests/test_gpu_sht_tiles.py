"""Edges of the analysis products: GEMM tiles of 1 to 6 column blocks of 16 (half a block per 8 maps) and of 64 or
128 rows, the triangle of cross spectra for 65 to 256 maps beside the 64 x 64 tiles outside that range, and spectra
of listed pairs, for which only the named maps are transformed.

A map's alms do not depend on the maps beside it: every call agrees with single-map calls and with sums over
their alms to the rounding of FP64 sums of at most 2 Nside ring terms (alms) or 2 lmax products (C_l): 1e-13 of
the largest value.
"""
import numpy as np
import pytest
import torch

import crime_amd

pytestmark = pytest.mark.gpu


def maps_of(n, nside, seed):
    return np.random.default_rng(seed).normal(size=(n, 12 * nside ** 2))


def cross(alm, lmax):
    """C_l of every pair from alms (n, nalm) in he_indexlm order."""
    out = np.zeros((len(alm), len(alm), lmax + 1))
    for m in range(lmax + 1):
        a = alm[:, [crime_amd.alm_index(l, m, lmax) for l in range(m, lmax + 1)]]
        w = 1.0 if m == 0 else 2.0
        out[:, :, m:] += w * np.einsum("al,bl->abl", a.real, a.real) + w * np.einsum("al,bl->abl", a.imag, a.imag)
    return out / (2 * np.arange(lmax + 1) + 1.0)


@pytest.mark.parametrize("n, nside, lmax", [(1, 48, 143), (7, 96, 200), (8, 12, 35), (9, 12, 30), (41, 16, 47),
                                            (64, 12, 35), (65, 12, 35), (100, 9, 20), (200, 8, 23), (256, 4, 11),
                                            (257, 4, 11)])
def test_alms_and_spectra_of_many_maps(n, nside, lmax):
    maps = maps_of(n, nside, n)
    with crime_amd.Sht(nside, lmax, max_maps=1) as one:
        ref = np.concatenate([one.map2alm(m) for m in maps])
    with crime_amd.Sht(nside, lmax, max_maps=n) as sh:
        alm = sh.map2alm(maps)
        cl = sh.anafast(maps)
    assert np.abs(alm - ref).max() < 1e-13 * np.abs(ref).max()
    want = cross(ref, lmax)
    assert np.abs(cl - want).max() < 1e-13 * np.abs(want).max()
    assert np.array_equal(cl, cl.transpose(1, 0, 2))


@pytest.mark.parametrize("fp64", [False, True])
@pytest.mark.parametrize("pairs", [[(3, 3)], [(0, 7), (7, 0), (5, 5)], [(a, a) for a in range(9)], [(8, 1), (2, 8)]])
def test_pairs_transform_the_named_maps(pairs, fp64):
    nside, n = 16, 9
    m = torch.from_numpy(maps_of(n, nside, 3)).to("cuda", torch.float64 if fp64 else torch.float32)
    torch.cuda.synchronize()
    with crime_amd.Sht(nside, max_maps=n) as sh:
        full = sh.anafast_device(m.data_ptr(), n, fp64)
        got = sh.cls_pairs_device(m.data_ptr(), n, fp64, pairs)
        with pytest.raises(crime_amd.CrimeError):
            sh.cls_pairs_device(m.data_ptr(), n + 1, fp64, pairs)
    want = np.stack([full[a, b] for a, b in pairs])
    assert np.abs(got - want).max() < 1e-13 * np.abs(full).max()
