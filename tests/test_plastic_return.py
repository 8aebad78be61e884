"""The FP32 bulk's plastic return (plastic_flow_delta in tmk_physics.hpp), built for the host from the
device header, against the same expressions in NumPy float32, where every operation rounds to nearest:
the same bits, so no operation of the return is less exact than an FP32 one.  (The host stand-in rounds
the hardware's estimates as coarsely as the hardware may.)
"""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = "/opt/rocm/llvm/bin/clang++"
f = np.float32


@pytest.fixture(scope="module")
def ret(tmp_path_factory):
    cc = CLANG if os.path.exists(CLANG) else shutil.which("clang++")
    if cc is None:
        pytest.skip("the device header needs clang's address spaces")
    so = str(tmp_path_factory.mktemp("pr") / "plastic_return.so")
    subprocess.run([cc, "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off",
                    "-I" + os.path.join(HERE, "cpp", "host_stub"), "-I" + os.path.join(HERE, "..", "include"),
                    "-o", so, os.path.join(HERE, "cpp", "plastic_return.cpp")], check=True)
    lib = ctypes.CDLL(so)
    pf = ctypes.POINTER(ctypes.c_float)

    def run(ns, k, dt, s):
        k, s = np.ascontiguousarray(k, f), np.array(s, f)
        lib.plastic_return(ns, len(s), k.ctypes.data_as(pf), ctypes.c_float(dt), s.ctypes.data_as(pf))
        return s

    return run


def expected(ns, k, dt, s):
    dxx, dyy, dzz, dxy, dxz, dyz, lam, gam = s.T.copy()
    md = (dxx + dyy + dzz) * f(1.0 / 3.0)
    exx, eyy, ezz = (dxx - md) + k[1], (dyy - md) + k[2], (dzz - md) + k[3]
    sxy, sxz, syz = dxy + k[4], dxz + k[5], dyz + k[6]
    J2 = f(0.5) * (exx * exx + eyy * eyy + ezz * ezz) + sxy * sxy
    if ns == 3:
        J2 = J2 + sxz * sxz + syz * syz
    ys = np.maximum(-k[7] * (md + k[0]) + (k[8] + gam * k[9]), f(0))
    tau = np.sqrt(J2)
    pl = (tau - ys) / (f(dt) * k[10] + k[11])
    dl = f(dt) * pl
    g, dm = dl * k[13] / tau, dl * k[12]
    new = [dxx - (dm + g * exx), dyy - (dm + g * eyy), dzz - (dm + g * ezz), dxy - g * sxy,
           dxz - g * sxz if ns == 3 else dxz, dyz - g * syz if ns == 3 else dyz, pl, gam + dl]
    old = [dxx, dyy, dzz, dxy, dxz, dyz, np.zeros_like(lam), gam]
    yields = J2 > ys * ys
    return np.where(yields[:, None], np.array(new).T, np.array(old).T), yields


@pytest.mark.parametrize("ns", [2, 3])
@pytest.mark.parametrize("eta", [0.0, 0.03])
def test_every_operation_rounds_to_nearest(ret, ns, eta):
    G, lam = 32038.0, 32038.0
    K, mu, beta, h, dt = lam + 2 * G / 3, 0.6, 0.3, 0.0, 3.75e-3
    k = np.array([-120.0, 0, 0, 0, 70.0, 0, 0, mu, 1.0, 0.01, h + G + mu * beta * K, eta * G, beta * K, G], f)
    rng = np.random.default_rng(5)
    s = np.zeros((20000, 8), f)
    s[:, :6] = rng.uniform(-1, 1, (len(s), 6)) * 10.0 ** rng.uniform(-3, 2, (len(s), 1))
    if ns == 2:
        s[:, 4:6] = 0
    s[:, 7] = rng.uniform(0, 1e-2, len(s))
    want, yields = expected(ns, k, dt, s)
    got = ret(ns, k, dt, s)
    assert 1000 < np.count_nonzero(yields) < len(s) - 1000
    assert np.array_equal(got, want)
