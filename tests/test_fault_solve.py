"""The device's rate-and-state fault solve (rs_solve in tmk_physics.hpp) against the reference's
bracketed Newton iteration (RSNEWTON, RSIBCF.ChF:336-401; rs_newton), both built for the host from
the device header with the host compiler's arithmetic (tests/cpp/fault_solve.cpp).

Both stop within atol = 2.2e-12 of a zero residual, at the same iterate but for the rounding of the
residual: where the residual crosses atol one may take a step more, so the slip rates differ by at
most 2 atol / f'(V), f' = alpha / V + eta (beta V >> 1), plus the rounding of y = asinh(beta V) and of
exp(psi / a), a few units in the last place of y and psi / a.
"""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = "/opt/rocm/llvm/bin/clang++"
ZS, V0 = 2.67e-3 * 3464.0, 1e-6
ATOL = 2.220446e-12
EPS = 2.0 ** -52


@pytest.fixture(scope="module")
def solve(tmp_path_factory):
    cc = CLANG if os.path.exists(CLANG) else shutil.which("clang++")
    if cc is None:
        pytest.skip("the device header needs clang's address spaces")
    so = str(tmp_path_factory.mktemp("fs") / "fault_solve.so")
    subprocess.run([cc, "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off",
                    "-I" + os.path.join(HERE, "cpp", "host_stub"), "-I" + os.path.join(HERE, "..", "include"),
                    "-o", so, os.path.join(HERE, "cpp", "fault_solve.cpp")], check=True)
    lib = ctypes.CDLL(so)
    pd = ctypes.POINTER(ctypes.c_double)

    def run(reference, phi, psi, sn, a, guess):
        args = [np.ascontiguousarray(x, dtype=np.float64) for x in (phi, psi, sn, a)]
        V = np.array(guess, dtype=np.float64)
        tau = np.empty_like(V)
        lib.fault_solve(int(reference), len(V), ctypes.c_double(ZS), ctypes.c_double(V0),
                        *[x.ctypes.data_as(pd) for x in args], V.ctypes.data_as(pd), tau.ctypes.data_as(pd))
        return V, tau

    return run


def _draw(seed, n=20000):
    rng = np.random.default_rng(seed)
    a, sn, psi = rng.uniform(0.005, 0.03, n), rng.uniform(50, 150, n), rng.uniform(0.3, 1.0, n)
    Vt = 10.0 ** rng.uniform(-18, 1, n)
    beta = np.exp(psi / a) / (2 * V0)
    phi = sn * a * np.arcsinh(beta * Vt) + 0.5 * ZS * Vt
    return rng, a, sn, psi, Vt, phi


GUESSES = {
    "rest": lambda rng, Vt, phi: np.zeros_like(Vt),
    "near": lambda rng, Vt, phi: Vt * (1 + 1e-3 * rng.standard_normal(len(Vt))),
    "any": lambda rng, Vt, phi: 10.0 ** rng.uniform(-14, 0, len(Vt)),
    "off": lambda rng, Vt, phi: Vt * 10.0 ** rng.uniform(-3, 3, len(Vt)),
    "outside": lambda rng, Vt, phi: np.where(rng.uniform(size=len(Vt)) < 0.5, 10 * phi / ZS, -1.0),
    "wave": lambda rng, Vt, phi: rng.uniform(0, 0.05, len(Vt)),
}


@pytest.mark.parametrize("guess", list(GUESSES))
def test_same_iterate_as_the_reference(solve, guess):
    rng, a, sn, psi, Vt, phi = _draw(sorted(GUESSES).index(guess))
    g = GUESSES[guess](rng, Vt, phi)
    V, tau = solve(False, phi, psi, sn, a, g)
    Vr, taur = solve(True, phi, psi, sn, a, g)
    alpha = sn * a
    y = taur / alpha
    # a root beyond the bracket: the iterate is held at the top, to its rounding
    slope = alpha / Vr + 0.5 * ZS
    bound = 2 * ATOL / slope + 8 * EPS * Vr * (1 + y + psi / a) + 8 * EPS * phi / slope
    assert np.all(np.abs(V - Vr) <= bound), np.max(np.abs(V - Vr) / bound)
    assert np.all(np.abs(tau - taur) <= 2 * ATOL + 16 * EPS * np.abs(taur))
    # and the same iterate, not only the same root, but where the residual is at the tolerance
    same = np.abs(V - Vr) <= 0.1 * ATOL / slope + 8 * EPS * Vr * (1 + y + psi / a) + 8 * EPS * phi / slope
    assert np.mean(same) > 0.995, np.mean(same)


@pytest.mark.parametrize("phi,psi,sn,a,guess", [
    (0.0, 0.6, 120.0, 0.01, 0.0),             # no load
    (70.0, 0.6, -5.0, 0.01, 1e-3),            # tension
    (70.0, 0.6, 0.0, 0.01, 1e-3),
    (70.0, 7.0, 120.0, 0.01, 1e-3),           # psi / a beyond the range of exp
    (70.0, -8.0, 120.0, 0.01, 1e-3),
    (float("nan"), 0.6, 120.0, 0.01, 1e-3),
    (70.0, float("nan"), 120.0, 0.01, 1e-3),
    (70.0, 0.6, 120.0, 0.01, float("nan")),
    (float("inf"), 0.6, 120.0, 0.01, 1e-3),
    (90.0, 0.2, 30.0, 0.01, 1e-3),            # the root beyond the bracket
    (5.0, 0.01, 100.0, 0.05, 1e-3),           # asinh far from a logarithm
    (12.823156259813329, 0.7683850130948197, 118.41973249921107, 0.007390680190921246, 14.0),  # 100 iterations
])
def test_other_inputs_give_what_the_reference_gives(solve, phi, psi, sn, a, guess):
    args = [np.array([x]) for x in (phi, psi, sn, a, guess)]
    V, tau = solve(False, *args)
    Vr, taur = solve(True, *args)
    assert np.array_equal(np.isnan(V), np.isnan(Vr)) and np.array_equal(np.isnan(tau), np.isnan(taur))
    if np.isfinite(Vr[0]):
        assert abs(V[0] - Vr[0]) <= 1e-12 * abs(Vr[0])
    if np.isfinite(taur[0]):
        assert abs(tau[0] - taur[0]) <= 1e-12 * abs(taur[0])
