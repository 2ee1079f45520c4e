"""A prediction from a closed emulator is refused by the library (CrimeError, EINVAL) whether its array is a
plain FP64 one, which goes to the library in one call, or takes the separate steps."""
import numpy as np
import pytest

import crime_amd
import crime_amd.emulator as em
from crime_amd import _ffi


@pytest.mark.parametrize("nets, dtype", [(1, np.float64), (1, np.float32), (2, np.float64)])
def test_closed_emulator_is_refused(nets, dtype):
    emu = em.Emulator.__new__(em.Emulator)
    emu.mlps = []
    for _ in range(nets):
        m = em.Mlp.__new__(em.Mlp)
        m._lib, m._h = _ffi.gpu_lib(), None
        emu.mlps.append(m)
    emu.mlp = emu.mlps[0]
    emu.scale, emu.dnu, emu._z = 1.0, 1.0, None
    with pytest.raises(crime_amd.CrimeError) as e:
        emu.predict(np.zeros((4, 8), dtype))
    assert e.value.rc == -1
