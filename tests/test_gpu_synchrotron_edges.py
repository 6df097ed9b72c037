"""The synchrotron coefficients' roots, exponential and sine at the ends of
their ranges (transfer.py:30-86 of the reference): outside FP32's range of X the
library's roots, beyond |pitch| = 2^15 its sine; the cuts in X and Theta; zero,
negative, infinite and NaN inputs.

Tolerance: X carries a relative error of about 5 units of the last place, X^(1/3)
of 5/3 + 1, and exp(-X^(1/3)) that times X^(1/3) <= 650 where nothing
underflows: 650 * 2.7 * 2^-53 + 20 * 2^-53 < 2.1e-13 on either side, 5e-13.
"""
import itertools

import numpy as np
import pytest

import mahakala as ma
from oracle import mahakala_np as onp

pytestmark = pytest.mark.gpu


def _both(Ne, Th, B, pitch, nu, **kw):
    with np.errstate(all="ignore"):
        ref = [np.asarray(v) for v in onp.synchrotron_coefficients(Ne, Th, B, pitch, nu, **kw)]
    return [np.asarray(v) for v in ma.synchrotron_coefficients(Ne, Th, B, pitch, nu, **kw)], ref


@pytest.mark.parametrize("invariant", [True, False])
def test_wide_range_of_X(invariant):
    """X from 1e-45 to 2.7e8 (X^(1/3) = 650), through 1e-36, at ordinary angles and beyond 2^15."""
    kw = dict(invariant=invariant, rescale_nu=1 / 230e9) if invariant else dict(invariant=False)
    B, Th, Ne = 30.0, 10.0, 1e5
    for pitch in (0.5, 3.0, -2.0, 32767.0, 32769.0, 1e6):
        nus = 2.0 / 9.0 * B * onp.EE / (2 * np.pi * onp.ME * onp.CL) * Th ** 2 * abs(np.sin(pitch))
        nu = nus * np.concatenate([10.0 ** np.linspace(-45, 8.4, 700), 1e-36 * (1 + np.linspace(-1e-6, 1e-6, 41))])
        one = np.ones_like(nu)
        got, ref = _both(Ne * one, Th * one, B * np.sign(np.sin(pitch)) * one, pitch * one, nu, **kw)
        for g, r in zip(got, ref):
            ok = np.isfinite(r) & (np.abs(r) > 1e-290)
            assert ok.sum() > 300
            np.testing.assert_allclose(g[ok], r[ok], rtol=5e-13)


@pytest.mark.parametrize("invariant", [True, False])
def test_cuts_and_special_values(invariant):
    kw = dict(invariant=invariant, rescale_nu=1 / 230e9) if invariant else dict(invariant=False)
    v = list(itertools.product([0.0, 1e5], [0.0, 0.299, 0.3, 10.0, np.nan], [0.0, 1e-12, 30.0, -30.0, np.nan],
                               [0.0, 1.0, np.pi, -1.0, np.nan], [1e-3, 230e9, 1e18, np.nan]))
    got, ref = _both(*[np.array(x) for x in zip(*v)], **kw)
    for g, r in zip(got, ref):
        assert not np.isnan(g).any()
        zero = r == 0.0
        np.testing.assert_array_equal(g[zero], 0.0)
        ok = np.isfinite(r) & (np.abs(r) > 1e-290)
        np.testing.assert_allclose(g[ok], r[ok], rtol=5e-13)
