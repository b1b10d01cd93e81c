"""The contact law's root and quotients against sqrtf and the division, bit
for bit: every float for the root, random and hardest cases for quotients."""
import ctypes
from ctypes import c_int, c_uint32, c_uint64

import pytest

from demso_amd import build

pytestmark = pytest.mark.gpu

LOW, HIGH = 31 << 23, 223 << 23  # 2^-96, 2^96


@pytest.fixture(scope="module")
def check():
    lib = ctypes.CDLL(str(build.CHECK if build.CHECK.exists() else build.build_check()))
    lib.check_root.argtypes = [c_uint32, c_uint64, ctypes.POINTER(c_uint64 * 2)]
    lib.check_quotients.argtypes = [c_int, c_uint64, c_uint64, ctypes.POINTER(c_uint64 * 2)]

    def run(name, *args):
        out = (c_uint64 * 2)()
        assert getattr(lib, name)(*args, ctypes.byref(out)) == 0
        return list(out)

    return run


def test_root_of_every_float(check):
    assert check("check_root", 0, LOW) == [0, 0]
    assert check("check_root", LOW, HIGH - LOW + 1) == [0, 0]
    assert check("check_root", HIGH + 1, (1 << 32) - HIGH - 1) == [0, 0]  # to infinity, NaNs, negative floats


@pytest.mark.parametrize("hard", [0, 1])
def test_quotients(check, hard):
    assert check("check_quotients", hard, 12345, 1 << 31)[0] == 0
