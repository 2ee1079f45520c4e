"""Emulator.predict over the sizes of a call: on both sides of every limit of its parts, of the pinned memory a handle
keeps and of the ring, and the cost of a handle's first longer call.

A row's spectrum does not depend on the call it is part of (the same products in the same order), so any call agrees
bit for bit with calls of 1000 rows.  The first call of a handle finds its memory: over several new handles the
fastest takes at most twice the fastest repeated one (memory pinned inside the call took it to four or five times)."""
import time

import numpy as np
import pytest

import crime_amd.emulator as em

pytestmark = pytest.mark.gpu


def emulator(nets, max_batch):
    mlps = []
    for k in range(nets):
        m = em.Mlp(max_batch=max_batch)
        m.set_params(em.init_params(30 + k))
        mlps.append(m)
    return em.Emulator(mlps, np.zeros(8), np.ones(8), 1.0, 0.1, 2e-7, 1.5625)


def inputs(n):
    rng = np.random.default_rng(n)
    x = rng.uniform(-1.0, 1.0, size=(n, 8))
    x[:, 6] += x[:, 5]
    return x


@pytest.mark.parametrize("nets, max_batch, sizes", [
    (1, 65536, (16384, 16385, 24576, 24577, 65537, 98304, 98305, 300001, 5000)),
    (1, 64, (64, 65, 4100, 24577, 98305, 70)),
    (2, 64, (64, 65, 4100, 24577)),
    (3, 65536, (4096, 4097, 24576, 24577, 65537)),
    (2, 1024, (1025, 98305)),
])
def test_sizes_agree(nets, max_batch, sizes):
    emu = emulator(nets, max_batch)
    try:
        for n in sizes:
            x = inputs(n)
            got = emu.predict(x)
            parts = np.concatenate([emu.predict(x[i:i + 1000]) for i in range(0, n, 1000)])
            assert np.isfinite(got).all() and np.array_equal(got, parts), n
    finally:
        emu.close()


@pytest.mark.parametrize("n", [5000, 16384])
def test_first_call_finds_its_memory(n):
    x = inputs(n)

    def timed(emu):
        t0 = time.perf_counter()
        emu.predict(x)
        return time.perf_counter() - t0

    first, again = [], []
    for _ in range(8):
        emu = emulator(1, 65536)
        try:
            first.append(timed(emu))
            again.extend(timed(emu) for _ in range(5))
        finally:
            emu.close()
    assert min(first) <= 2.0 * min(again), (min(first), min(again))
