"""Emulator.predict (crime_mlp_predict: encoding, networks and sinh in one call) against the same steps one by one
(predict_y, then numpy's sinh and the scale), on both sides of its limits: calls whose kernels read the host's inputs
(up to 4096 rows), chunks, rings of chunks, ensembles, and inputs that are not a plain FP64 array.  The networks'
outputs are the same bits; sinh of numpy's FP32 library and of the device's FP64 differ by at most 4 ulp (5e-7),
the product rounds once on each side: 6e-7."""
import numpy as np
import pytest

import crime_amd.emulator as em

pytestmark = pytest.mark.gpu


def emulator(nets, max_batch):
    spec = em.MockSpec()
    x = em.features(em.latin_hypercube(64, 1), spec)
    dnu = (spec.nu_hi - spec.nu_lo) / spec.n_nu
    enc = em.encode(x, dnu)
    mlps = []
    for k in range(nets):
        m = em.Mlp(max_batch=max_batch)
        m.set_params(em.init_params(20 + k))
        mlps.append(m)
    return em.Emulator(mlps, enc.mean(axis=0), enc.std(axis=0), 7.0, 1.5, 2e-7, dnu), x


@pytest.mark.parametrize("nets, max_batch, n", [(1, 65536, 1), (1, 65536, 256), (1, 65536, 4096), (1, 65536, 4097),
                                                (1, 65536, 65537), (1, 65536, 400001), (1, 512, 513),
                                                (1, 8192, 100000), (3, 1024, 700), (3, 1024, 5000)])
def test_predict_equals_its_steps(nets, max_batch, n):
    emu, x = emulator(nets, max_batch)
    try:
        rng = np.random.default_rng(n)
        x = x[rng.integers(0, len(x), n)] * (1 + 1e-3 * rng.normal(size=(n, 8)))
        want = np.sinh(emu.predict_y(x)) * np.float32(emu.scale)
        for _ in range(2):
            got = emu.predict(x)
            assert got.shape == (n,) and got.dtype == np.float32
            assert np.all(np.abs(got - want) <= 6e-7 * np.abs(want))
        assert np.array_equal(emu.predict(x[:n // 2 + 1]), got[:n // 2 + 1])
        # other layouts and types go through the separate steps
        assert np.allclose(emu.predict(np.asfortranarray(x)), got, rtol=6e-7, atol=0)
        assert np.allclose(emu.predict(x.astype(np.float32)), emu.predict(x.astype(np.float32).astype(np.float64)),
                           rtol=6e-7, atol=0)
    finally:
        emu.close()
