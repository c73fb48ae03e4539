"""The Jacobi pairs' quotients and roots equal the IEEE operations (tests/cpp/plain_math_check.hip): they start from the
hardware's reciprocal and reciprocal root, whose approximations no document pins."""
import ctypes
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))


def test_quotients_and_roots_are_correctly_rounded_over_their_range():
    lib = os.path.join(HERE, "cpp", "libplain_math_check.so")
    if not os.path.exists(lib):
        subprocess.run(["make", "-C", os.path.dirname(lib), os.path.basename(lib)], check=True)
    counts = (ctypes.c_uint64 * 8)()
    assert ctypes.CDLL(lib).plain_math_check(counts) == 0
    binade = 1 << 23
    assert list(counts[0::2]) == [90 * binade + 1, 2 * (44 * binade + 1), 2 * (86 * binade + 1), 4 * 64 * binade]
    assert list(counts[1::2]) == [0, 0, 0, 0]
