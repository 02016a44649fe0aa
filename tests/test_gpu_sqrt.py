"""sqrt_rn (venusaur_amd/csrc/vz_device.h) equals the IEEE square root.

The kernels take the roots of sphere tests, of normalisation and of refraction
by sqrt_rn: v_rsq_f32 refined by one fma Newton-Raphson step for x in [2^-64,
2^64), sqrtf elsewhere.  The oracle calls sqrtf, so images stay bit-exact only
if the two agree on every input.  This runs the product's sqrt_rn over all of
that range (1,073,741,824 floats) and samples of the others, and also checks
that the comparison can fail: the unrefined product must differ somewhere.
"""
import ctypes as C
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "gpu_checks", "libsqrtcheck.so")


def _lib():
    if not os.path.exists(LIB):
        subprocess.run(["make", "-C", os.path.join(HERE, "gpu_checks")], check=True)
    lib = C.CDLL(LIB)
    lib.vz_check_sqrt_rn.restype = C.c_int
    lib.vz_check_sqrt_rn.argtypes = [C.POINTER(C.c_ulonglong), C.POINTER(C.c_uint32)]
    return lib


@pytest.mark.gpu
def test_sqrt_rn_equals_ieee_root_on_its_whole_range():
    print("case: sqrt_rn against sqrtf(x), x in [2^-64, 2^64) and samples outside", flush=True)
    out = (C.c_ulonglong * 5)()
    bad = (C.c_uint32 * 4)()
    assert _lib().vz_check_sqrt_rn(out, bad) == 0
    ref_diff, rn_diff, raw_diff, seen, expected = list(out)
    assert expected == 128 * (1 << 23) + (1 << 16) and seen == expected
    assert ref_diff == 0, "the root and the double-rounded reference disagree"
    assert rn_diff == 0, f"sqrt_rn differs from sqrtf(x) for {rn_diff} inputs, e.g. {[hex(b) for b in bad]}"
    assert raw_diff > 0, "the unrefined product never differed: the comparison checks nothing"
