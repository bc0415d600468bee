"""Device code on the CPU (tests/host): osbl_line.h compiled for the host with
a stand-in for the HIP header, the lanes of a wave as fibers."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HOST = os.path.join(HERE, "host")
CSRC = os.path.join(HERE, "..", "opensbli_amd", "csrc")
WENO_Z, TENO6 = 3, 5


def _compile(tmp, name):
    out = os.path.join(str(tmp), name + ".so")
    cmd = ["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-Wno-unknown-pragmas", "-I" + HOST,
           "-I" + CSRC, os.path.join(HOST, name + ".cpp"), "-o", out]
    subprocess.run(cmd, check=True)
    return ctypes.CDLL(out)


@pytest.fixture(scope="module")
def lanes(tmp_path_factory):
    return _compile(tmp_path_factory.mktemp("host"), "line_lanes")


def _segment(lib, q, qo, s0, s1, conv, mode, first, down, dt=1e-3):
    n = q.shape[1]
    dp = ctypes.POINTER(ctypes.c_double)
    q = np.ascontiguousarray(q)
    o, qn = np.array(qo), np.full_like(q, np.nan)
    d = ctypes.c_double
    lib.run_segment(conv, mode, n, s0, s1, d(dt), d(n - 1.0), d(0.4), d(0.25), int(first), d(1.4), d(1e-16), d(1e-6),
                    q.ctypes.data_as(dp), o.ctypes.data_as(dp), qn.ctypes.data_as(dp), int(down))
    return qn, o


@pytest.mark.parametrize("conv,mode", [(WENO_Z, 0), (WENO_Z, 1), (TENO6, 0)])
@pytest.mark.parametrize("n", [9, 64, 65, 127, 200])
def test_a_line_does_not_depend_on_the_order_of_the_lanes(lanes, n, conv, mode):
    """One wave over a whole line (a chunk of 63 cells, then 64 at a time), lanes
    upwards and downwards between two barriers, and the same line in parts of 63
    cells: the same bits."""
    rs = np.random.RandomState(n)
    rho, u, p = rs.uniform(0.5, 1.5, n), rs.uniform(-0.5, 0.5, n), rs.uniform(0.5, 1.5, n)
    q = np.stack([rho, rho * u, p / 0.4 + 0.5 * rho * u * u])
    qo = q * rs.uniform(0.9, 1.1, q.shape)
    up = _segment(lanes, q, qo, 0, n, conv, mode, False, False)
    down = _segment(lanes, q, qo, 0, n, conv, mode, False, True)
    assert np.isfinite(up[0]).all()
    for a, b in zip(up, down):
        assert np.array_equal(a, b)
    parts = np.full_like(q, np.nan), np.array(qo)
    for s0 in range(0, n, 63):
        s1 = min(s0 + 63, n)
        for a, b in zip(parts, _segment(lanes, q, qo, s0, s1, conv, mode, False, True)):
            a[:, s0:s1] = b[:, s0:s1]
    for a, b in zip(up, parts):
        assert np.array_equal(a, b)
