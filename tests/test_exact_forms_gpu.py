"""The correctly rounded reciprocal, quotient and square root of the
integration kernels (mcx_internal.h: recip_rn, div_rn, sqrt_rn) equal IEEE's on
every operand that decides it, checked on the device by
tests/cpp/exact_forms_check (all reciprocals, all roots, all quotients near the
middle of two floats)."""
import subprocess

import pytest

from marching_cube_amd import build

pytestmark = pytest.mark.gpu


def test_exact_forms_equal_ieee():
    print("[case] reciprocal, quotient and root forms", flush=True)
    res = subprocess.run([build.EXACT_FORMS_BIN], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stderr
    f = res.stdout.split()
    vals = dict(zip(f[0::2], (int(x) for x in f[1::2])))
    assert vals["pairs"] > 90_000_000
    assert vals["recip_mismatch"] == vals["sqrt_mismatch"] == vals["div_mismatch"] == 0
