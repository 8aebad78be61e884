"""The library's own two-operation divisions -- div2_exact, the low words, divr2, divr, div3, div6, built
for the host from the sources (tests/sanitize/host_library.cpp) -- against exact rational arithmetic
(tests/test_div2.py): the flag that sends a material to the two operations is set exactly when every
dividend that could be misrounded is not, dividends that are misrounded are by divr2 and not by divr, and
the range of dividends that the comments state holds, from both sides of its limit.
"""
import math
import random
import subprocess
from fractions import Fraction as F

import pytest

from test_div2 import constants, divr2, suspects
from test_host_library import HERE, driver  # noqa: F401  (fixture)
from tetemoko_amd import scenarios


def ask(driver, lines):  # noqa: F811
    r = subprocess.run([driver, "division"], cwd=HERE, input="\n".join(lines) + "\n", capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]
    return [[float.fromhex(t) for t in row.split()] for row in r.stdout.splitlines()[:len(lines)]]


def div_line(b, xs):
    return " ".join(["div", b.hex(), str(len(xs))] + [x.hex() for x in xs])


def low(b):
    return float(F(1) / F(b) - F(1.0 / b))


def test_flag_and_failing_dividends(driver):  # noqa: F811
    r = random.Random(5)
    bs = [r.uniform(1, 2) * 2.0 ** r.randint(-30, 30) for _ in range(1500)]
    bs += list(constants().values()) + [1.0, 2.0, 3.0, 10.0, 0.0026700000000000001, math.nextafter(2.0, 1.0)]
    bs += [scenarios.G_MPA / (3013.5 * 3013.5)]
    cases = []
    for b in bs:
        Y, X = suspects(b)
        scale = b / Y  # a power of two
        assert math.frexp(scale)[0] == 0.5
        cases.append((b, [math.ldexp(x * scale, r.randint(-200, 200)) for x in X]))
    out = ask(driver, [div_line(b, xs) for b, xs in cases])
    flags = set()
    for (b, xs), row in zip(cases, out):
        bad = [x for x in xs if divr2(x, b) != x / b]
        assert bool(row[0]) == (not bad), b
        assert row[1] == 1.0 / b and row[2] == low(b)
        for x, two, full in zip(xs, row[3::2], row[4::2]):
            assert two == divr2(x, b) and full == x / b, (b, x)
        flags.add(bool(bad))
    assert flags == {True, False}


@pytest.mark.parametrize("b,want", [(0.0, 0), (-16.0, 0), (math.inf, 0), (math.nan, 0), (5e-324, 0)])
def test_divisors_that_keep_the_other_division(driver, b, want):  # noqa: F811
    assert ask(driver, [div_line(b, [])])[0][0] == want


def test_materials(driver):  # noqa: F811
    r = random.Random(9)
    mats = [(scenarios.CS, scenarios.CP, scenarios.G_MPA), (3013.5, scenarios.CP, scenarios.G_MPA)]
    mats += [(r.uniform(1500, 4000), r.uniform(4000, 7000), r.uniform(1e4, 5e4)) for _ in range(300)]
    out = ask(driver, [" ".join(["par"] + [float(v).hex() for v in m]) for m in mats])
    for m, (flag, rho, Zp, Zs, lrho, l2Zp, l2Zs) in zip(mats, out):
        assert lrho == low(rho) and l2Zp == 0.5 * low(Zp) and l2Zs == 0.5 * low(Zs)
        exact = True
        for b in (rho, Zp, Zs):
            Y, X = suspects(b)
            exact = exact and all(divr2(float(x), float(Y)) == float(x) / float(Y) for x in X)
        assert bool(flag) == exact, m
    assert out[0][0] == 1 and out[1][0] == 0


@pytest.mark.parametrize("name", ["rho", "Zs", "Zp"])
def test_range_of_dividends(driver, name):  # noqa: F811
    b = constants()[name]
    yl = low(b)
    limit = 2.0 ** -1022 / abs(yl)  # a yl is normal from here on
    assert limit < 1e-289
    r = random.Random(13)
    above = [limit * r.uniform(1, 4) * r.choice([-1, 1]) for _ in range(4000)] + [1.7e308 * min(1.0, b)]
    below = [limit * 10.0 ** r.uniform(-16, 0) for _ in range(4000)]
    row = ask(driver, [div_line(b, above + below + [0.0, -0.0, math.inf, math.nan])])[0][3::2]
    assert row[:len(above)] == [x / b for x in above]
    off = [abs(q - x / b) / math.ulp(x / b) for x, q in zip(below, row[len(above):])]
    assert max(off) <= 1.0
    zero, mzero, inf, nan = row[-4:]
    assert zero == 0.0 and mzero == 0.0 and math.copysign(1, zero) == 1
    assert math.copysign(1, mzero) == (-1 if yl > 0 else 1)
    assert (inf == math.inf if yl > 0 else math.isnan(inf)) and math.isnan(nan)


def test_thirds_and_sixths(driver):  # noqa: F811
    r = random.Random(17)
    xs = [r.uniform(-1, 1) * 10.0 ** r.randint(-289, 308) for _ in range(20000)]
    xs += [0.0, -0.0, math.inf, -math.inf, 1.7976931348623157e308]
    row = ask(driver, [" ".join(["third", str(len(xs))] + [x.hex() for x in xs])])[0]
    for x, a, b in zip(xs, row[::2], row[1::2]):
        assert (a, math.copysign(1, a)) == (x / 3.0, math.copysign(1, x / 3.0)), x
        assert (b, math.copysign(1, b)) == (x / 6.0, math.copysign(1, x / 6.0)), x
    tiny = [r.uniform(1, 2) * 10.0 ** r.uniform(-315, -291) for _ in range(4000)]
    row = ask(driver, [" ".join(["third", str(len(tiny))] + [x.hex() for x in tiny])])[0]
    assert max(abs(a - x / 3.0) / math.ulp(x / 3.0) for x, a in zip(tiny, row[::2])) <= 1.0
