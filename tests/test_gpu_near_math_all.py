"""The cheaper reciprocal, quotient, root and x / pi of the target function against the IEEE forms, bit
for bit, operand by operand on the device: all reciprocals, roots and quotients by pi of their ranges,
a sample of the 2^46 pairs of mantissas for the quotient (the probe counts all of them in 23 s), and
operands spread over the ranges with their ends."""
import ctypes as C
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu

LIB = Path(__file__).resolve().parent.parent / "restir-vulkan_amd" / "probe" / "near_math.so"


@pytest.fixture(scope="module")
def probe():
    lib = C.CDLL(str(LIB))
    for name in ("near_rcp", "near_over_pi", "near_sqrt", "near_div", "near_range"):
        getattr(lib, name).restype = C.c_int64
    lib.near_div.argtypes = [C.c_uint32, C.c_uint32]
    lib.near_range.argtypes = [C.c_uint32]
    return lib


@pytest.mark.parametrize("what", ["near_rcp", "near_over_pi", "near_sqrt"])
def test_every_operand(probe, what):
    assert getattr(probe, what)() == 0


@pytest.mark.parametrize("a0", [0, 1 << 21, 0x3504f3, 0x7ff000])  # both ends and around sqrt(2)
def test_quotients_of_mantissas(probe, a0):
    assert probe.near_div(a0, 1 << 12) == 0


def test_operands_over_their_ranges(probe):
    assert probe.near_range(64) == 0
