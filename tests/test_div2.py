"""The two-operation division of the FP64 update (divr2 in tmk_physics.hpp) and the host's check of
the constants it is used for (div2_exact in tmk_api.hip), in exact integer and rational arithmetic:
a rounding differs from the IEEE quotient only where the check says one does.
"""
import math
import random
from fractions import Fraction as F

import pytest

from tetemoko_amd import scenarios


def divr2(x, y):
    """fma(x, yh, RN(x yl)) with yh = RN(1/y), yl = RN(1/y - yh), each rounding exact."""
    yh = float(F(1) / F(y))
    yl = float(F(1) / F(y) - F(yh))
    return float(F(x) * F(yh) + F(float(F(x) * F(yl))))


def suspects(y):
    """The dividends div2_exact tries, as 53-bit integers: those whose quotient by y lies next to a
    midpoint, |2^p X - (2Q + 1) Y| <= 6."""
    Y = int(math.ldexp(math.frexp(y)[0], 53))
    k = (Y & -Y).bit_length() - 1
    out = []
    for p in (53, 54):
        for N in range(-6, 7):
            if N == 0 or k > 2 or N % (1 << k):
                continue
            M = 1 << (p - k)
            c = (-(N >> k) * pow(Y >> k, -1, M)) % M
            while c < 1 << 54:
                if c >= 1 << 53 and c & 1:
                    assert (c * Y + N) % (1 << p) == 0
                    X = (c * Y + N) >> p
                    if 1 << 52 <= X < 1 << 53 and (X >= Y) == (p == 53):
                        out.append(X)
                c += M
    return Y, out


def constants():
    rho = scenarios.G_MPA / (scenarios.CS * scenarios.CS)
    return {"rho": rho, "Zs": rho * scenarios.CS, "Zp": rho * scenarios.CP}


@pytest.mark.parametrize("name", ["rho", "Zs", "Zp"])
def test_the_material_divides_exactly(name):
    y = constants()[name]
    Y, X = suspects(y)
    assert all(divr2(float(x), float(Y)) == float(x) / float(Y) for x in X)
    r = random.Random(7)
    for _ in range(20000):
        x = r.uniform(-1, 1) * 10.0 ** r.randint(-30, 6)
        assert divr2(x, y) == x / y


def test_suspects_are_the_only_dividends_that_can_fail():
    """For divisors that do fail, every failing dividend found by search near the suspects' class is a
    suspect: dividends with the smallest remainders against a midpoint are exactly those of |N| small."""
    r = random.Random(3)
    failing = 0
    for _ in range(4000):
        y = r.uniform(1, 2)
        Y, X = suspects(y)
        bad = [x for x in X if divr2(float(x), float(Y)) != float(x) / float(Y)]
        failing += bool(bad)
        for x in r.sample(range(1 << 52, 1 << 53), 3):
            if divr2(float(x), float(Y)) != float(x) / float(Y):
                assert x in X
    assert failing > 0  # the check matters: some constants do fail


def test_a_material_that_fails():
    """The shear speed the GPU test of the other division uses (tests/test_gpu_step.py)."""
    y = scenarios.G_MPA / (3013.5 * 3013.5)
    Y, X = suspects(y)
    assert any(divr2(float(x), float(Y)) != float(x) / float(Y) for x in X)


def test_signed_zero_and_sign():
    y = constants()["Zp"]
    assert math.copysign(1.0, -0.0 * (1 / y) + -0.0) == -1.0
    for x in (3.7, -3.7, 1e-200, -1e-200):
        assert divr2(x, y) == x / y


@pytest.mark.parametrize("y", [3.0, 6.0])
def test_the_plastic_return_divides_exactly(y):
    """div3, div6: the low words are exact and every quotient rounds as the division does."""
    h, l = (1.0 / 3.0, 2.0 ** -54 / 3.0) if y == 3.0 else (0.5 / 3.0, 2.0 ** -55 / 3.0)
    assert h == 1.0 / y and l == float(F(1) / F(y) - F(h))
    assert not suspects(y)[1]
    r = random.Random(11)
    for x in [float(k) for k in range(-40, 41)] + [r.uniform(-1, 1) * 10.0 ** r.randint(-30, 12) for _ in range(20000)]:
        assert divr2(x, y) == x / y
