"""The polynomial of the inference GELU (one_plus_erf in sur_lib.hip), evaluated
here in float32 with the coefficients of the source: GELU from it is no further
from the float64 value than with a correctly rounded float32 erf, on [-6, 6] and
over the float32 range, and the exponent stays positive and grows beyond the
fitted interval, so the tails go to z and to 0."""
import os
import re

import numpy as np
from scipy.special import erf, erfc, ndtr

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'frfs_amd', 'csrc', 'sur_lib.hip')
f32 = np.float32


def _coefficients():
    """Lowest power (u^1) first."""
    body = open(SRC).read().split('float one_plus_erf(float z) {')[1].split('return')[0]
    c = [float(v) for v in re.findall(r'(?:float a = |, u, )(-?[0-9.e+-]+)f', body)]
    assert len(c) == 10
    return c[::-1]


def _fma(a, b, c):
    return f32(a.astype(np.float64) * b.astype(np.float64) + np.float64(c))


def _exponent(c, u):
    a = np.full_like(u, f32(c[-1]))
    with np.errstate(over='ignore'):
        for k in range(len(c) - 2, -1, -1):
            a = _fma(a, u, f32(c[k]))
        return f32(a * u)


def _gelu_fit(c, z):
    e = f32(np.exp2(-_exponent(c, np.abs(z)).astype(np.float64)))
    return f32(f32(f32(0.5) * z) * np.where(z > 0, f32(2) - e, e).astype(f32))


def _gelu_erf(z):
    e = f32(erf(f32(z * f32(0.70710678118654752)).astype(np.float64)))
    return f32(f32(f32(0.5) * z) * f32(f32(1) + e))


def test_no_further_from_float64_than_with_erf():
    c = _coefficients()
    z = np.random.default_rng(0).uniform(-6, 6, 400000).astype(f32)
    ref = z.astype(np.float64) * ndtr(z.astype(np.float64))
    fit, old = (np.abs(g(z).astype(np.float64) - ref) for g in (lambda x: _gelu_fit(c, x), _gelu_erf))
    rms = [np.sqrt((e ** 2).mean()) for e in (fit, old)]
    print('rms', rms, 'max', fit.max(), old.max())
    assert rms[0] <= rms[1] and fit.max() <= old.max()


def test_tails():
    c = _coefficients()
    u = np.linspace(6.2, 200, 20000).astype(f32)
    q = _exponent(c, u)
    end = erfc(6.2 / np.sqrt(2))                       # of the fitted interval
    assert (q > -np.log2(end) - 1e-4).all() and (np.diff(q) >= 0).all()
    z = np.concatenate([np.geomspace(7, 3e38, 400), [np.finfo(f32).max]]).astype(f32)
    assert np.array_equal(_gelu_fit(c, z), z)
    assert (np.abs(_gelu_fit(c, -z)) <= 0.5 * 6.2 * end).all()
