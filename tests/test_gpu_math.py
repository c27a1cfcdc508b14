"""The tracing kernels' short forms of roots, reciprocal roots and texel
channels on every input, against fp64 (tests/cpp/device_math.hip)."""
import ctypes as C
import os

import pytest

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "quadray-engine_amd", "lib", "libqrcheck.so")


def test_short_forms_are_correctly_rounded(device):
    print("case every float through the short roots", flush=True)
    bad = (C.c_ulonglong * 6)()
    assert C.CDLL(LIB).qrcheck_math(bad) == 0
    assert dict(zip(("sqrt_mid", "root", "rsq", "unorm8", "near t0", "near"), bad)) == \
        dict.fromkeys(("sqrt_mid", "root", "rsq", "unorm8", "near t0", "near"), 0)
