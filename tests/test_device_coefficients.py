"""The polynomial coefficients in csrc/device.hpp are those csrc/erfcx_fit.py makes (no GPU needed): the FP64 ones to the
last bit, the FP32 ones to 2 units in the last place (the fit runs in FP64 least squares)."""

import os
import re
import sys

import numpy as np
import pytest

pytest.importorskip("mpmath")
pytest.importorskip("scipy")

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pgm-md_amd", "csrc")
sys.path.insert(0, CSRC)

import erfcx_fit  # noqa: E402

NUMBER = r"-?\d+\.\d+(?:e[+-]\d+)?"


def _source():
    with open(os.path.join(CSRC, "device.hpp")) as f:
        return f.read()


def _table(name):
    body = re.search(r"struct %s \{.*?c\[\d+\] = \{(.*?)\}" % name, _source(), re.S).group(1)
    return [float(v) for v in re.findall(NUMBER, body)]


@pytest.mark.parametrize(
    "name,fit,bound", [("ErfcxD", erfcx_fit.fit_erfcx64, 1.1e-16), ("ExpD", erfcx_fit.fit_exp64, 4e-17)]
)
def test_fp64_tables(name, fit, bound):
    err, c = fit()
    assert _table(name) == c
    assert err < bound   # the polynomial in exact arithmetic


def test_fp32_coefficients():
    err, c = erfcx_fit.fit()
    body = re.search(r"float erfcxFast\(float x\) \{(.*?)return", _source(), re.S).group(1)
    have = np.array([float(v) for v in re.findall(r"(%s)f[;)]" % NUMBER, body) if v not in ("0.5", "1.0")], np.float32)
    assert len(have) == len(c) == 9
    np.testing.assert_array_almost_equal_nulp(have, c.astype(np.float32), 2)
    assert err < 2e-8
