"""The device's fault faces (rs_fault, sw_fault in tmk_physics.hpp), built for the host from the device
header: the velocities that a face's tractions divide by an impedance to give are IEEE quotients for every
state, from tractions near the smallest number to infinite ones (SWFAULTBCF, SWIBCF.ChF:79-267;
RSFAULTBCF, RSIBCF.ChF:158-323), as NumPy gives them for the same operations.
"""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = "/opt/rocm/llvm/bin/clang++"
ZP, ZS = 2.67e-3 * 6000.0, 2.67e-3 * 3464.0


@pytest.fixture(scope="module")
def faces(tmp_path_factory):
    cc = CLANG if os.path.exists(CLANG) else shutil.which("clang++")
    if cc is None:
        pytest.skip("the device header needs clang's address spaces")
    so = str(tmp_path_factory.mktemp("ff") / "fault_faces.so")
    subprocess.run([cc, "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off",
                    "-I" + os.path.join(HERE, "cpp", "host_stub"), "-I" + os.path.join(HERE, "..", "include"),
                    "-o", so, os.path.join(HERE, "cpp", "fault_faces.cpp")], check=True)
    lib = ctypes.CDLL(so)
    pd, d = ctypes.POINTER(ctypes.c_double), ctypes.c_double

    def run(sw, w, a, b, L, tau0, state):
        w = np.ascontiguousarray(w, dtype=np.float64)
        out = np.empty((len(w), 6, 2))
        lib.fault_faces(int(sw), len(w), d(ZP), d(ZS), d(1e-6), d(a), d(b), d(L), d(tau0), d(state),
                        w.ctypes.data_as(pd), out.ctypes.data_as(pd))
        return out

    return run


def _states():
    rng = np.random.default_rng(3)
    w = rng.uniform(-1, 1, (4000, 6, 2)) * 10.0 ** rng.uniform(-2, 2, (4000, 1, 1))
    tiny = rng.uniform(-1, 1, (2000, 6, 2)) * 10.0 ** rng.uniform(-315, -280, (2000, 1, 1))
    huge = rng.uniform(-1, 1, (50, 6, 2))
    huge[:, 3] = 1.7e308 * np.where(huge[:, 3] < 0, -1.0, 1.0)  # normal tractions whose sum overflows
    inf = rng.uniform(-1, 1, (50, 6, 2))
    inf[:, 1, 0] = np.inf
    return np.concatenate([w, tiny, huge, inf])


@pytest.mark.parametrize("sw", [False, True])
def test_velocities_are_quotients(faces, sw):
    w = _states()
    w[:6000, 3] -= np.where(np.arange(6000) < 4000, 120.0, 0.0)[:, None]  # compression but for the tiny states
    o = faces(sw, w.reshape(len(w), 12), *((0.677, 0.525, 0.4, 75.0, 0.1) if sw else (0.012, 0.016, 0.02, 70.0, 0.7)))
    vx, vy, vz, syy, sxy, syz = (w[:, k] for k in range(6))
    with np.errstate(all="ignore"):
        p1, p2 = -syy[:, 0] - ZP * vy[:, 0], syy[:, 1] - ZP * vy[:, 1]
        q1, q2 = -sxy[:, 0] - ZS * vx[:, 0], sxy[:, 1] - ZS * vx[:, 1]
        for s in range(2):
            np.testing.assert_array_equal(o[:, 1, s], -((p1 + p2) / 2.0 / ZP))
        np.testing.assert_array_equal(o[:, 0, 0], -((o[:, 4, 0] + q1) / ZS))
        if sw:
            np.testing.assert_array_equal(o[:, 0, 1], (o[:, 4, 1] - q2) / ZS)
            r1, r2 = -syz[:, 0] - ZS * vz[:, 0], syz[:, 1] - ZS * vz[:, 1]
            np.testing.assert_array_equal(o[:, 2, 0], -((o[:, 5, 0] + r1) / ZS))
            np.testing.assert_array_equal(o[:, 2, 1], (o[:, 5, 1] - r2) / ZS)
    assert np.any(np.isinf(o[:, 1]))
