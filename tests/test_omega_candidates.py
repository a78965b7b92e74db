"""The device's disorientation takes three of Grimmer's 24 candidates (the largest
component, the two largest magnitudes added, all four magnitudes added); that this
is the largest |candidate| to the last bit rests on rounding being monotone and
symmetric.  Checked in the same double arithmetic against the oracle's 24."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import oracle as om


def _three(p, q):
    m = q * np.array([1.0, -1.0, -1.0, -1.0])
    a = m[0] * p[0] - m[1] * p[1] - m[2] * p[2] - m[3] * p[3]
    b = p[0] * m[1] + m[0] * p[1] + (m[2] * p[3] - m[3] * p[2])
    c = p[0] * m[2] + m[0] * p[2] + (-(m[1] * p[3]) + m[3] * p[1])
    d = p[0] * m[3] + m[0] * p[3] + (m[1] * p[2] - m[2] * p[1])
    v = np.abs(np.array([a, b, c, d]))
    s = np.sort(v)
    return max(s[3], (s[3] + s[2]) * (1.0 / np.sqrt(2.0)), (((v[0] + v[1]) + v[2]) + v[3]) * 0.5)


@pytest.mark.parametrize("kind", ["random", "near", "same", "coarse"])
def test_three_candidates_are_the_largest(kind):
    rng = np.random.default_rng(len(kind))
    for _ in range(3000):
        p, q = (x / np.sqrt((x * x).sum()) for x in rng.normal(size=(2, 4)))
        if kind == "near":
            q = p + 1e-7 * rng.normal(size=4)
        elif kind == "same":
            q = p.copy()
        elif kind == "coarse":
            p, q = np.round(p * 4) / 4, np.round(q * 4) / 4
        assert om.disori_omega(p, q) == _three(p, q)
