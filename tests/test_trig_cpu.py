"""The device's bounded trigonometry (dtrig.h) compiled for the CPU: its fp64 values against numpy's, and the fp32
results it rounds to. Angles of whole warps with the neighbourhoods of multiples of pi/2, every quadrant and octant
of the arctangent with signed zeros, and arccosines up to both ends."""
import ctypes
import decimal
import math
import os
import re
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = """
#define PH_DEV inline
#include "dtrig.h"
extern "C" void trig(long n, const float* x, const float* y, double* s, double* c, double* a, double* ad, float* sf, float* cf, float* af, float* ac) {
    for (long i = 0; i < n; i++) {
        phd::sincos64(x[i], s + i, c + i);
        a[i] = phd::atan2_64(y[i], x[i]);
        ad[i] = x[i] >= -1 && x[i] <= 1 ? phd::acos64(x[i]) : 0;
        phd::sincos_cr(x[i], sf + i, cf + i);
        af[i] = phd::atan2_cr(y[i], x[i]);
        ac[i] = x[i] >= -1 && x[i] <= 1 ? phd::acos_cr(x[i]) : 0;
    }
}
"""


@pytest.fixture(scope="module")
def trig(tmp_path_factory):
    d = tmp_path_factory.mktemp("trig")
    (d / "t.cpp").write_text(SRC)
    so = d / "t.so"
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-I", os.path.join(ROOT, "photon_amd/csrc/hip"), str(d / "t.cpp"), "-o", str(so)],
                   check=True)
    lib = ctypes.CDLL(str(so))

    def run(x, y):
        x, y = np.ascontiguousarray(x, np.float32), np.ascontiguousarray(y, np.float32)
        out = [np.zeros(len(x), t) for t in [np.float64] * 4 + [np.float32] * 4]
        lib.trig(ctypes.c_long(len(x)), *[ctypes.c_void_p(v.ctypes.data) for v in [x, y] + out])
        return out

    return run


def _ulps64(got, want):
    return np.max(np.abs(got - want) / np.spacing(np.maximum(np.abs(want), 1e-300)))


def test_trigonometry_is_within_two_ulps_and_rounds_to_the_same_floats(trig):
    rng = np.random.default_rng(2)
    n = 400000
    x = rng.uniform(-2 * math.pi, 2 * math.pi, n).astype(np.float32)
    k = n // 4  # around multiples of pi/2
    x[:k] = (np.round(rng.uniform(-4, 4, k)) * (math.pi / 2) * (1 + rng.uniform(-1, 1, k) * 10.0 ** rng.uniform(-8, -2, k))).astype(np.float32)
    x[k:2 * k] = (rng.choice([-1.0, 1.0], k) * (1 - 10.0 ** rng.uniform(-8, 0, k))).astype(np.float32)
    x[2 * k:2 * k + 6] = [0.0, -0.0, 1.0, -1.0, math.pi, 2 * math.pi]
    y = rng.uniform(-1, 1, n).astype(np.float32)
    y[::7] = x[::7]
    y[1::7] *= np.float32(1e-6)
    y[2::701], y[3::701] = 0.0, -0.0
    s, c, a, ad, sf, cf, af, ac = trig(x, y)
    xd, yd = x.astype(np.float64), y.astype(np.float64)
    unit = np.abs(x) <= 1
    # Two ulps of ours (three for the arccosine), and half a one of the reference's.
    assert _ulps64(s, np.sin(xd)) <= 2.5 and _ulps64(c, np.cos(xd)) <= 2.5 and _ulps64(a, np.arctan2(yd, xd)) <= 2.5
    assert _ulps64(ad[unit], np.arccos(xd[unit])) <= 3.5
    for got, want in ((sf, np.sin(xd)), (cf, np.cos(xd)), (af, np.arctan2(yd, xd)), (ac[unit], np.arccos(xd[unit]))):
        assert np.array_equal(got, want.astype(np.float32))


def test_arctangent_of_signed_zeros_and_nan(trig):
    x = np.array([0.0, -0.0, 0.0, -0.0, -1.0, -1.0, 1.0, np.nan, 1.0, 0.0], np.float32)
    y = np.array([0.0, 0.0, -0.0, -0.0, 0.0, -0.0, -0.0, 1.0, np.nan, -2.0], np.float32)
    af = trig(x, y)[6]
    want = np.arctan2(y, x)
    assert np.array_equal(np.isnan(af), np.isnan(want))
    ok = ~np.isnan(want)
    assert np.array_equal(af[ok], want[ok]) and np.array_equal(np.signbit(af[ok]), np.signbit(want[ok]))


def test_the_arctangents_polynomial_is_as_close_as_it_says():
    """Its coefficients, read from the header, against the series of the arctangent in 50 digits: t + t z p(z) is within
    1.5e-18 of it for |t| <= tan(pi/8)."""
    text = open(os.path.join(ROOT, "photon_amd/csrc/hip/dtrig.h")).read()
    body = text[text.index("double atan2_64"):text.index("double a = __builtin_fma(t * z, p, t)")]
    coefficients = [decimal.Decimal(float.fromhex(c)) for c in re.findall(r"-?0x1\.[0-9a-f]+p-\d+", body)]
    assert len(coefficients) == 12
    with decimal.localcontext() as ctx:
        ctx.prec = 50
        end = decimal.Decimal(2).sqrt() - 1
        for k in range(0, 401):
            t = end * k / 400
            z = t * t
            p = decimal.Decimal(0)
            for c in coefficients:
                p = p * z + c
            want = sum((-1) ** j * t ** (2 * j + 1) / (2 * j + 1) for j in range(60))
            assert abs(t + t * z * p - want) < decimal.Decimal("1.5e-18"), k
