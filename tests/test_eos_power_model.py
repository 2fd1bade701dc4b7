"""The short form of the EOS's power x**GAMMA (csrc/common.h pow_gamma) in a
host model: with the hardware's float log2 and exp2 off by two ulps either way
the double it rounds stays within 512 double ulps of the power, so that the
rounding test, which sends everything within 1024 of a float midpoint to pow,
leaves the rounded value unchanged."""
import numpy as np
import pytest

f32, f64, ext = np.float32, np.float64, np.longdouble
GAMMA = f64(f32(1.4))


def _fma(a, b, c):
    return (a.astype(ext) * b + c).astype(f64)


def _short_form(x, log_ulps, exp_ulps):
    t = np.log2(x.astype(f64)).astype(f32)
    t = t + f32(log_ulps) * np.spacing(t)
    s0 = np.exp2((f32(-0.2) * t).astype(f64)).astype(f32)
    s0 = (s0 + f32(exp_ulps) * np.spacing(s0)).astype(f64)
    X = x.astype(f64)
    s2 = s0 * s0
    s5 = (s2 * s2) * s0
    h = _fma(-X, s5, f64(1.0))
    s = _fma(s0 * h, _fma(h, f64(3.0 / 25.0), f64(0.2)), s0)
    z = t.astype(f64) * ((GAMMA - 1.4) * 0.69314718055994531)
    y7 = (X * X) * ((s * s) * s)
    return _fma(y7, _fma(f64(0.5) * z, z, z), y7)


@pytest.mark.skipif(np.finfo(ext).nmant < 63, reason="no extended precision")
def test_short_form_error_with_an_inexact_logarithm():
    rng = np.random.default_rng(4)
    x = np.concatenate([
        np.exp2(rng.uniform(-16.0, 4.0, 60000)),
        1.0 + rng.uniform(-1e-3, 1e-3, 20000),        # t near 0
        np.exp2(np.arange(-16.0, 4.5, 0.5))]).astype(f32)
    want = np.power(x.astype(ext), ext(GAMMA))
    worst = 0.0
    for lo in (-2, -1, 0, 1, 2):
        for ex in (-2, 0, 2):
            y = _short_form(x, lo, ex)
            err = np.abs(y.astype(ext) - want) / np.spacing(want.astype(f64))
            worst = max(worst, float(err.max()))
    assert 1.0 < worst < 512.0, worst
