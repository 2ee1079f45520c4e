"""The hidden units' activation is decided from the hardware's exponential and reciprocal with a margin, and its quotient
written out: over every FP32 value the BF16 result and the quotient are those of the plain formula."""
import pytest

from crime_amd.emulator import Mlp

pytestmark = pytest.mark.gpu


def test_every_float():
    with Mlp(max_batch=64) as net:
        assert net.silu_check() == (0, 0)
