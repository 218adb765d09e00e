"""The FP64 arithmetic of the ion kernels (csrc/chy_device.h), compiled for the
host: the hardware's reciprocal and reciprocal square root are stood in for by
values 2^-24 off, which the refinements after them have to make up for.
Quotients and roots against IEEE division and square root, sine, cosine and
logarithm against 80-bit values at the arguments that occur, the 24-bit uniform
numbers (k + 1/2) 2^-24."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_SRC = """
#include "chy_device.h"
extern "C" {
void v_div_rn(long n, const double *a, const double *d, double *q)
{ for (long i = 0; i < n; i++) q[i] = chy::div_rn(a[i], d[i], 1.0 / d[i]); }
void v_div(long n, const double *a, const double *b, double *q)
{ for (long i = 0; i < n; i++) q[i] = chy::div_normal(a[i], b[i]); }
void v_sqrt(long n, const double *x, double *r) { for (long i = 0; i < n; i++) r[i] = chy::sqrt_normal(x[i]); }
void v_log(long n, const double *u, double *r) { for (long i = 0; i < n; i++) r[i] = chy::log_unit(u[i]); }
void v_sincos(long n, const double *u, double *s, double *c)
{ for (long i = 0; i < n; i++) chy::sincos2pi(u[i], s[i], c[i]); }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    d = tmp_path_factory.mktemp("device_math")
    (d / "m.hip").write_text(_SRC)
    subprocess.run([hipcc, "--offload-host-only", "-O2", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared",
                    "-I" + os.path.join(_ROOT, "collisional-hybrid_amd", "csrc"), "-I" + os.path.join(_ROOT, "include"),
                    str(d / "m.hip"), "-o", str(d / "m.so")], check=True, capture_output=True)
    return C.CDLL(str(d / "m.so"))


def _call(f, *args, outs=1):
    n = len(args[0])
    out = [np.empty(n) for _ in range(outs)]
    f(C.c_long(n), *[C.c_void_p(np.ascontiguousarray(a, np.float64).ctypes.data) for a in args],
      *[C.c_void_p(o.ctypes.data) for o in out])
    return out[0] if outs == 1 else out


def _u24():
    """Every 17th of the 2^24 arguments, and those around the quadrants, 1 and 0."""
    k = [np.arange(0, 1 << 24, 17)]
    k += [np.arange(-40, 40) + (q << 21) for q in range(9)]
    k = np.concatenate(k)
    return (k[(k >= 0) & (k < 1 << 24)] + 0.5) * 2.0 ** -24


def _check(got, ref, most, rate):
    """got within `most` ulps of the 80-bit ref, off the nearest double for at
    most `rate` of the values."""
    near = ref.astype(np.float64)
    ulp = np.spacing(np.abs(near))
    assert (np.abs(got.astype(np.longdouble) - ref) / ulp).max() <= most
    assert np.mean(got != near) <= rate


# spacings as runs have them, one ulp around powers of two, and full mantissas
def test_division_by_a_spacing_is_rounded_to_nearest(lib):
    rng = np.random.default_rng(1)
    n = 400000
    d = np.concatenate([rng.choice([0.05, 0.1, 1 / 3, 0.7, 1e-3, 12.8 / 256], n // 4), np.exp(rng.uniform(-20, 20, n // 4)),
                        np.nextafter(2.0 ** rng.integers(-8, 8, n // 4), 0), np.nextafter(2.0 ** rng.integers(-8, 8, n // 4), 9e9)])
    a = d * rng.uniform(0, 512, n)
    a[::3] = d[::3] * rng.integers(0, 512, len(a[::3]))
    a[1::7] = np.nextafter(a[1::7], 0)
    a[:4] = 0.0
    assert np.array_equal(_call(lib.v_div_rn, a, d), a / d)


# the exact remainder leaves a wrong last bit only where a quotient lies within
# 2^-24 of an ulp, or so, of a tie
def test_general_division_and_square_root(lib):
    rng = np.random.default_rng(2)
    n = 1000000
    a, b = rng.standard_normal((2, n)) * np.exp(rng.uniform(-60, 60, (2, n)))
    q, ref = _call(lib.v_div, a, b), a / b
    assert (np.abs(q - ref) <= np.spacing(np.abs(ref))).all() and np.mean(q != ref) <= 1e-5
    x = np.concatenate([np.exp(rng.uniform(-120, 120, n)), rng.uniform(0, 1, n), np.arange(1.0, 3000) ** 2])
    r, ref = _call(lib.v_sqrt, x), np.sqrt(x)
    assert (np.abs(r - ref) <= np.spacing(ref)).all() and np.mean(r != ref) <= 1e-5
    # zero, and what rounding leaves below it, clamp to zero
    assert np.array_equal(_call(lib.v_sqrt, np.array([0.0, -0.0, -2.0 ** -52])), np.zeros(3))


# the series' and the final addition's roundings are at most a quarter of an ulp
# beside the last rounding's half; the rates are those that the functions state
def test_sine_and_cosine(lib):
    u = np.concatenate([_u24(), [0.0, 0.125, 0.25, 0.5, 0.75, 1.0]])
    s, c = _call(lib.v_sincos, u, outs=2)
    angle = (2.0 * np.pi * u).astype(np.longdouble)  # the rounded product is the argument
    _check(s, np.sin(angle), 0.75, 0.0135)
    _check(c, np.cos(angle), 0.75, 0.0135)


def test_logarithm(lib):
    u = _u24()
    _check(_call(lib.v_log, u), np.log(u.astype(np.longdouble)), 0.75, 0.0085)
