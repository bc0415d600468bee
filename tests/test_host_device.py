"""Device code on the CPU (tests/host): osbl_device.h and osbl_line.h compiled
for the host with a stand-in for the HIP header, the lanes of a wave as fibers."""
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


@pytest.fixture(scope="module")
def recon(tmp_path_factory):
    return _compile(tmp_path_factory.mktemp("host"), "recon")


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


def _dp(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def _teno_reference(d, six, quirk, eps, ct):
    """The weights from one quotient each (teno.py:57-234, 407-465): value and
    how near to the cut-off the nearest weight is (relative)."""
    A, B, C, D, E = (np.ascontiguousarray(d[:, k]) for k in range(5))
    b = [13 / 12 * (C - B) ** 2 + 0.25 * (B + C) ** 2,
         13 / 12 * (D - C) ** 2 + 0.25 * (D - 3 * C) ** 2,
         13 / 12 * (B - A) ** 2 + 0.25 * (3 * B - A) ** 2]
    c = [B + 2 * C, 4 * C - D, 5 * B - 2 * A]
    w = [0.55, 0.4, 0.05]
    tau = np.abs(b[0] - b[2])
    if six:
        q3 = C - 2 * D + E
        b.append((11 * C - 7 * D + 2 * E) ** 2 / 36 + 13 / 12 * (3 * D - 2 * C - E) ** 2 +
                 781 / 720 * (2 * q3 if quirk else q3 * q3))
        c.append(4.5 * C - 2 * D + 0.5 * E)
        w = [0.462, 0.3, 0.054, 0.184]
        tau = np.abs(b[3] - (b[0] + b[2] - 4 * b[1]) / 6)
    with np.errstate(all="ignore"):
        a = [(1 + tau / (eps + x)) ** 6 for x in b]
        cut = ct * sum(a)
        near = np.min([np.abs(x / cut - 1) for x in a], axis=0)
        keep = [np.where(x < cut, 0.0, wr) for x, wr in zip(a, w)]
        return sum(k * x for k, x in zip(keep, c)) / sum(keep), near


@pytest.mark.parametrize("six,quirk", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("eps", [1e-140, 1e-100, 4e-16])
@pytest.mark.parametrize("scale", [1e-60, 1e-30, 1.0, 1e30, 1e39, 1e52, 1e70])
def test_teno_weights_over_the_range_of_the_quotients(recon, scale, eps, six, quirk):
    """Differences and eps for which the product of all indicators leaves the
    range of a double: the weights are those of the quotients taken one by one
    (the indicators' rounding, 1e-12, apart; a weight that near to the cut-off
    may fall on either side)."""
    rs = np.random.RandomState(5)
    n = 4000
    d = scale * rs.standard_normal((n, 5)) * 10.0 ** rs.uniform(-3, 0, (n, 5))
    d[::7] = 0.0           # a uniform stretch
    d[1::7] = scale * 0.1  # a linear one
    num, den = np.empty(n), np.empty(n)
    f = ctypes.c_double
    recon.teno(int(six), int(quirk), ctypes.c_long(n), _dp(d), f(eps), f(1e-6), _dp(num), _dp(den))
    want, near = _teno_reference(d, six, quirk, eps, 1e-6)
    ok = np.isfinite(want) & ~(near < 1e-9)
    assert ok.mean() > 0.8
    err = np.abs(num / den - want)[ok] / scale
    assert np.all(err <= 1e-12), (err.max(), int((~(err <= 1e-12)).sum()))


@pytest.mark.parametrize("z,eps", [(1, 4e-14), (0, 4e-6)])
def test_weno_weights_at_the_largest_differences(recon, z, eps):
    """Differences of 1e22, the bound that the header states (a reconstruction
    gets the sum or difference of two such): the same weights as in units 2^40
    times larger."""
    rs = np.random.RandomState(3)
    n = 4000
    d = rs.uniform(-2e22, 2e22, (n, 5))
    f = ctypes.c_double
    out = []
    for unit in (1.0, 2.0 ** -40):
        num, den = np.empty(n), np.empty(n)
        recon.weno(z, ctypes.c_long(n), _dp(d * unit), f(eps * unit * unit), _dp(num), _dp(den))
        assert np.isfinite(num).all() and np.isfinite(den).all()
        out.append(num / den / unit)
    assert np.abs(out[0] - out[1]).max() <= 1e-12 * 2e22


def test_quotients_and_roots_are_rounded_correctly_or_nearly(recon):
    """a/b, 1/b and sqrt(b) from estimates as coarse as the hardware's: within
    0.501 units in the last place (an IEEE result is within 0.5)."""
    rs = np.random.RandomState(1)
    n = 400000
    a, b = (rs.uniform(1, 2, n) * 2.0 ** rs.randint(-40, 40, n) for _ in range(2))
    worst = np.empty(3)
    recon.ulps(ctypes.c_long(n), _dp(a), _dp(b), _dp(worst))
    assert np.all(worst <= 0.501), worst
