"""Host rules of the list of the pores that need no GPU."""
import ctypes
import os
import re
import subprocess

import pytest

from initializator_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(_lib.LIB_PATH):
        subprocess.run(["make", "-C", os.path.join(ROOT, "initializator_amd", "csrc")], check=True,
                       stdout=subprocess.DEVNULL)
    return _lib.load()


def _internal(lib, name):
    """A function of namespace nmri by its name in the library's symbols."""
    out = subprocess.run(["nm", "-D", "--defined-only", _lib.LIB_PATH], check=True, capture_output=True, text=True).stdout
    return getattr(lib, re.search(rf"\b(_ZN4nmri{len(name)}{name}E\w*)", out).group(1))


def test_a_list_stays_inside_32_bit_byte_offsets(lib):
    """Every array of the list is read at slot * size in 32 bits: with velocity
    the largest is the 16-byte record, which wraps at 2^28 slots; without, three
    components.  (The slot past the last one is read too.)"""
    fit = _internal(lib, "pores_fit")
    fit.restype, fit.argtypes = ctypes.c_bool, [ctypes.c_uint64, ctypes.c_bool]
    assert not fit(64, True) and not fit(64, False)  # the empty group alone
    assert fit(128, True) and fit(128, False)
    for vel, size in ((True, 16), (False, 12)):
        wraps = (1 << 32) // size
        assert fit(wraps // 64 * 64 - 192, vel)
        for n in (wraps // 64 * 64, wraps // 64 * 64 + 64, 300_000_000 // 64 * 64 if vel else 360_000_000 // 64 * 64,
                  (1 << 32), (1 << 33) + 128):
            assert not fit(n, vel), (n, vel)
