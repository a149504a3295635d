"""The closed-form cell recovery of the stage kernels (gpu-vah_amd/csrc/vah_face.h,
compiled for the host from the same header) against the oracle's
getInferredVariables (EnergyMomentumTensor.cpp:74-197) from the same start."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from tests.test_face_speed import _state
from tests.test_oracle_math import conserved_from_primitives, p

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-vah_amd", "csrc")

SRC = r'''
#define __host__
#define __device__
#include FACE_H
// 1 when the closed form applies; v: e, u^tau, u^x, u^y, u^eta
extern "C" int cell(double t, const double *q, double u0, double *v) {
    const vah::FaceStart s = vah::face_start(u0 * u0);
    double M[4];
    for (int m = 0; m < 4; ++m) M[m] = q[m] - q[5 + m];
    vah::CellRoot c;
    const bool ok = vah::cell_root(t, M[0], M[1], M[2], M[3], q[4], s, &c);
    v[0] = c.e, v[1] = c.ut, v[2] = c.ux, v[3] = c.uy, v[4] = c.un;
    return ok;
}
'''


@pytest.fixture(scope="module")
def cell(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    d = tmp_path_factory.mktemp("cell")
    (d / "c.cpp").write_text(SRC.replace("FACE_H", '"' + os.path.join(CSRC, "vah_face.h") + '"'))
    subprocess.run(["g++", "-O2", "-shared", "-fPIC", "-o", str(d / "c.so"), str(d / "c.cpp")], check=True)
    f = ctypes.CDLL(str(d / "c.so")).cell
    dp = ctypes.POINTER(ctypes.c_double)
    f.argtypes = [ctypes.c_double, dp, ctypes.c_double, dp]
    return f


@pytest.mark.parametrize("kind", [0, 1, 2, 3])
def test_closed_form_recovery_is_where_the_newton_path_ends(oracle_mod, cell, kind):
    """Near starts, far starts, unphysical states and light-like flow.  Rounding
    of M / E reaches u as (u^tau)^2 eps and e as M0 (u^tau)^2 eps (64 eps for the
    operations of both sides); the iteration's stopping rule (|du| <= 1e-7 u,
    then quadratic) adds 1e-11 of u and 1e-12 of M0."""
    L = oracle_mod.lib()
    rng = np.random.default_rng(23 + kind)
    out, v = np.zeros(6), np.zeros(5)
    fired = 0
    for k in range(5000):
        t = rng.uniform(0.3, 5.0)
        q, u0, phys = _state(rng, t, kind)
        if not cell(t, p(q), u0, p(v)):
            continue
        fired += 1
        assert L.orc_recover(t, p(q), 1.0, u0, p(out)) == 0, (k, t, u0)
        eps = 64 * 2.2e-16 * out[2] ** 2
        assert abs(v[0] - out[0]) <= (1e-12 + eps) * abs(q[0] - q[5]), (k, v, out)
        uT = max(np.hypot(out[3], out[4]), 1e-12)
        assert abs(v[1] - out[2]) <= (1e-11 + eps) * out[2], (k, v, out)
        assert max(abs(v[2:4] - out[3:5])) <= (1e-11 + eps) * uT, (k, v, out)
        assert abs(v[4] - out[5]) <= (1e-11 + eps) * max(abs(out[5]), 1e-12), (k, v, out)
    assert fired > (0 if kind in (1, 2) else 4900), fired


def test_state_at_rest(cell):
    q = conserved_from_primitives(0.5, 10.0, 3.0, 1.0, 0.0, 0.0, 0.0, np.zeros(10))
    v = np.zeros(5)
    assert cell(0.5, p(q), 0.0, p(v)) == 1
    assert abs(v[0] - 10.0) < 1e-14 * 10 and abs(v[1] - 1.0) < 1e-15 and np.all(v[2:] == 0.0)


@pytest.mark.parametrize("break_", ["nan", "inf", "zero", "luminal"])
def test_broken_states_go_to_the_iteration(cell, break_):
    q = conserved_from_primitives(0.5, 10.0, 3.0, 1.0, 0.0, 0.0, 0.0, np.zeros(10))
    if break_ == "nan":
        q[1] = np.nan
    elif break_ == "inf":
        q[0] = np.inf
    elif break_ == "zero":
        q[:] = 0.0
    else:
        q[3] = 1.0001 * (q[0] + q[4]) / 0.5
    assert cell(0.5, p(q), 0.1, p(np.zeros(5))) == 0
