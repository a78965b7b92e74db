"""The angle from which a Rollett-Holm weight counts as exactly 1.0 is accepted on
one evaluation (cut * exp(-arg) <= 2^-55 at moderate arg and exponent) instead of
samples.  Restated here over the same glibc functions: wherever the rule accepts,
no angle above has another weight, and no pair at or below the matching |q0| has
one in the oracle."""
from __future__ import annotations

import math

import numpy as np
import pytest

from oracle import oracle as om
from score_amd import abi
from score_amd.synth import ParamsSpec

LAGB = 15.0 / 180.0 * math.pi


def _weight(cut, trans, n, theta):
    try:
        return 1.0 - cut * math.exp(-1.0 * trans * math.pow(theta / LAGB, n))
    except OverflowError:  # C's pow gives infinity there, so exp gives 0
        return 1.0


def _accepted(cut, trans, n):
    """theta_hi where the rule accepts, else None"""
    if _weight(cut, trans, n, math.pi) != 1.0 or _weight(cut, trans, n, 0.0) == 1.0:
        return None
    lo, hi = 0.0, math.pi
    for _ in range(200):
        mid = 0.5 * (lo + hi)
        lo, hi = (lo, mid) if _weight(cut, trans, n, mid) == 1.0 else (mid, hi)
    theta = hi + 0.2 / 180.0 * math.pi
    if theta >= 2.0 * math.acos(0.85):
        return None
    arg = trans * math.pow(theta / LAGB, n)
    ok = n <= 1000.0 and 2.0 <= arg <= 700.0 and cut * math.exp(-1.0 * arg) <= 2.0 ** -55
    return theta if ok else None


def _settings():
    rng = np.random.default_rng(7)
    yield 0.9, 5.0, 9.0
    for _ in range(400):
        yield 10.0 ** rng.uniform(-12, 6), 10.0 ** rng.uniform(-2, 2.5), 10.0 ** rng.uniform(-0.5, 3.2)


def test_accepted_settings_have_no_other_weight_above():
    seen = 0
    for cut, trans, n in _settings():
        theta = _accepted(cut, trans, n)
        if theta is None:
            continue
        seen += 1
        near = theta + np.arange(200) * 1e-9
        for t in (*near, *np.linspace(theta, math.pi, 400)):
            assert _weight(cut, trans, n, t) == 1.0, (cut, trans, n, t)
    assert seen >= 50 and _accepted(0.9, 5.0, 9.0) is not None


@pytest.mark.parametrize("cut,trans,n", [(0.9, 5.0, 9.0), (0.99, 5.0, 9.0), (1.0, 3.0, 4.0)])
def test_pairs_beyond_the_angle_have_weight_one(cut, trans, n):
    theta = _accepted(cut, trans, n)
    assert theta is not None
    omega_hi = math.cos(0.5 * theta)
    prm = ParamsSpec(mobility_model=abi.MOB_ROLLETTHOLM, rh_cut=cut, rh_trans=trans, rh_exponent=n)
    rng = np.random.default_rng(3)
    below = 0
    for p, q in rng.normal(size=(4000, 2, 4)):
        p, q = p / np.sqrt((p * p).sum()), q / np.sqrt((q * q).sum())
        if om.disori_omega(p, q) <= np.nextafter(omega_hi, 0.0):
            below += 1
            assert om.mobility_weight(prm, p, q) == 1.0
    assert below >= 100
