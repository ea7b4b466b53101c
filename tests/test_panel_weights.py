"""The kernel's panel polynomials against its definition
exp(beta (sqrt(1 - (2 d / w)^2) - 1)) (src/kernel.rs:81-89) in long double:
the engine's own coefficients, evaluated as the kernels do (Horner with one
rounding a step, the even part plus and minus x times the odd part), over
every width, for the beta of upsampling factor 2 and for those of factors
from 1.1 to 64.  The largest weight error of a width may not exceed that of
the direct formula in the same precision, or a unit in the last place of 1
where that is larger (2^-52, 2^-23).
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

REPLAY = os.path.join(os.path.dirname(os.path.abspath(__file__)), "replay")
LD = np.longdouble


@pytest.fixture(scope="module")
def panels():
    subprocess.run(["make", "-s", "-C", REPLAY], check=True)
    L = ctypes.CDLL(os.path.join(REPLAY, "_build", "libtile_replay.so"))
    L.replay_panels.argtypes = [ctypes.c_int, ctypes.c_double, ctypes.c_int, ctypes.c_void_p,
                                ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p]

    def get(width, beta, f64):
        coef = (ctypes.c_double * 512)()
        odd, n = ctypes.c_int(), ctypes.c_int()
        even = L.replay_panels(width, beta, int(f64), coef, 512, ctypes.byref(odd),
                               ctypes.byref(n))
        assert n.value == (width - 1) // 2 * (even + odd.value)
        return np.asarray(coef[: n.value]).reshape(-1, even + odd.value), even
    return get


def _exact(d, w, beta):
    s = 2 * d / w
    return np.exp(LD(beta) * (np.sqrt(1 - s * s) - 1))


def _fma(a, b, c, real):
    wide = np.float64 if real is np.float32 else LD
    return (a.astype(wide) * b.astype(wide) + c.astype(wide)).astype(real)


def _horner(coef, x2, real):
    v = np.full(x2.shape, coef[-1], dtype=real)
    for c in coef[-2::-1]:
        v = _fma(v, x2, np.full(x2.shape, c, dtype=real), real)
    return v


def _errors(table, even, w, beta, real):
    """Largest error of the inner weights: (polynomials, direct formula)."""
    off = (np.linspace(-0.5, 0.5, 501) - 0.5 * (w - 1)).astype(real)
    x = off + real(0.5 * (w - 1))
    x2 = x * x
    poly = direct = 0.0
    for t in range(1, (w - 1) // 2 + 1):
        row = table[t - 1].astype(real)
        e, o = _horner(row[:even], x2, real), _horner(row[even:], x2, real)
        for cell, sx in ((t, x), (w - 1 - t, -x)):
            ref = _exact(off.astype(LD) + cell, w, beta)
            s = real(2) * (off + real(cell)) / real(w)
            plain = np.exp(real(beta) * (np.sqrt(real(1) - s * s) - real(1)))
            poly = max(poly, float(np.abs(_fma(sx, o, e, real) - ref).max()))
            direct = max(direct, float(np.abs(plain - ref).max()))
    return poly, direct


def _betas(w):
    yield {2: 2.20, 3: 2.26, 4: 2.38}.get(w, 2.30) * w
    for sigma in (1.1, 1.25, 1.5, 3.0, 4.0, 8.0, 64.0):
        yield 0.97 * np.pi * w * (1 - 1 / (2 * sigma))


@pytest.mark.parametrize("prec,width", [("f32", w) for w in range(3, 9)] +
                         [("f64", w) for w in range(3, 17)])
def test_panels_are_as_good_as_the_formula(panels, prec, width):
    real, ulp = (np.float64, 2.0 ** -52) if prec == "f64" else (np.float32, 2.0 ** -23)
    for beta in _betas(width):
        table, even = panels(width, beta, prec == "f64")
        poly, direct = _errors(table, even, width, beta, real)
        assert poly <= max(direct, ulp), (beta / width, poly, direct)
