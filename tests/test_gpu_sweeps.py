"""Block shapes at which the 2-D and 3-D kernels split their work differently
(rows of one wave or several, chunks of 64 interfaces, tiles and their
remainders), against the oracle: residual and five steps, relative L2 <= 1e-10
per variable."""
import numpy as np
import pytest

from conftest import check_parity

pytestmark = pytest.mark.gpu


def _block(n, conv, bc, averaging="roe", rk="rk3", viscous="none", seed=0):
    """A block of order-one variables, smooth and periodic, on [0, 1)^d."""
    nd = len(n)
    x = np.meshgrid(*[np.arange(k) / k for k in reversed(n)], indexing="ij")
    rs = np.random.RandomState(seed)

    def wave(amp):
        return amp * sum(np.sin(2 * np.pi * (rs.randint(1, 3) * c + rs.rand())) for c in x)
    rho = 1.0 + wave(0.1)
    u = [0.3 + wave(0.1) for _ in range(nd)]
    p = 1.0 + wave(0.1)
    q0 = np.stack([rho] + [rho * v for v in u] + [p / 0.4 + 0.5 * rho * sum(v * v for v in u)])
    delta = [1.0 / k for k in n]
    problem = dict(ndim=nd, n=list(n), delta=delta, conv=conv, averaging=averaging, viscous=viscous, rk=rk,
                   bc=[[bc, bc]] * nd, gama=1.4, Minf=1.0, Re=100.0, Pr=0.71, dt=0.1 * min(delta), eps=1e-16,
                   teno_ct=1e-6)
    return problem, q0


def _check(problem, q0, oracle, what):
    from opensbli_amd.native import Block
    print("case", what, flush=True)
    g, r = Block(problem), oracle.RefSolver(problem)
    g.set_state(q0)
    r.set_state(q0)
    check_parity(g.rhs(), r.rhs(), what + " residual")
    g.set_state(q0)
    r.set_state(q0)
    g.run(5)
    r.run(5)
    check_parity(g.get_state(), r.get_state(), what)


@pytest.mark.parametrize("bc", ["periodic", "extrap0"])
@pytest.mark.parametrize("conv,averaging,rk", [("weno_z", "roe", "rk3"), ("weno_js", "simple", "ls3"),
                                               ("teno5", "roe", "rk3"), ("teno6", "roe", "ls3")])
@pytest.mark.parametrize("n", [(8, 8), (62, 9), (63, 17), (64, 16), (65, 33), (127, 8), (190, 40), (64, 3100)])
def test_2d_shapes(n, conv, averaging, rk, bc, oracle):
    problem, q0 = _block(n, conv, bc, averaging, rk)
    _check(problem, q0, oracle, f"2-D {n} {conv} {averaging} {rk} {bc}")


@pytest.mark.parametrize("conv", ["weno_z", "teno6"])
@pytest.mark.parametrize("n", [(8, 8, 8), (63, 9, 10), (66, 17, 9), (130, 12, 33)])
def test_3d_shapes(n, conv, oracle):
    problem, q0 = _block(n, conv, "periodic", viscous="const")
    _check(problem, q0, oracle, f"3-D {n} {conv}")


@pytest.mark.parametrize("bc", ["periodic", "extrap0"])
@pytest.mark.parametrize("n", [(63, 33, 32), (64, 33, 32), (65, 33, 32), (127, 34, 31), (130, 10, 9), (66, 56, 55)])
def test_3d_rows(n, bc, oracle):
    """Rows of one wave (periodic: the flux left of cell 0 is the last one's)
    and rows split among waves, below and above 1024 and 3072 rows."""
    problem, q0 = _block(n, "weno_z", bc)
    _check(problem, q0, oracle, f"3-D rows {n} {bc}")


@pytest.mark.parametrize("bc", ["periodic", "symmetry"])
@pytest.mark.parametrize("conv,rk,viscous", [("central_skew", "ls3", "const"), ("central_skew", "rk3", "none"),
                                             ("central_cons", "rk3", "const"), ("central_cons", "ls3", "none")])
@pytest.mark.parametrize("n", [(8, 8, 8), (31, 9, 10), (33, 16, 11), (64, 8, 40), (65, 17, 9), (130, 12, 70)])
def test_3d_central_shapes(n, conv, rk, viscous, bc, oracle):
    problem, q0 = _block(n, conv, bc, rk=rk, viscous=viscous)
    _check(problem, q0, oracle, f"3-D {n} {conv} {rk} {viscous} {bc}")


@pytest.mark.parametrize("wall", ["adiabatic_wall", "isothermal_wall"])
@pytest.mark.parametrize("bscheme", ["reduced_access", "carpenter"])
@pytest.mark.parametrize("conv,sensor", [("teno5", True), ("weno_z", False)])
@pytest.mark.parametrize("n", [(20, 40), (31, 46), (45, 61), (47, 44)])
def test_2d_plate_shapes(n, conv, sensor, bscheme, wall, oracle):
    """Closures, metric, Sutherland viscosity and the sensor where a tile's
    last column or row starts in, before or behind a closure row.  (Not TENO6:
    its unsquared indicator lets the cut-off of single interfaces switch by
    rounding on this noisy state, between the oracle's two builds as well --
    8e-11 at 45 x 61 with the isothermal wall -- so no bar of 1e-10 holds.)"""
    from opensbli_amd.problems import flat_plate
    twall = 1.6 if wall == "isothermal_wall" else None
    problem, q0 = flat_plate(n=n, conv=conv, sensor=sensor, noise=1e-3, ndim=2, bscheme=bscheme, wall=wall,
                             Twall=twall)
    _check(problem, q0, oracle, f"plate {n} {conv} {bscheme} {wall}")


@pytest.mark.parametrize("n", [(9, 16), (30, 15), (46, 70)])
def test_2d_periodic_viscous_shapes(n, oracle):
    problem, q0 = _block(n, "weno_z", "periodic", viscous="const", rk="ls3")
    _check(problem, q0, oracle, f"2-D viscous {n}")


@pytest.mark.parametrize("bc", [["periodic", "zero_gradient"], ["extrap0", "periodic"], ["symmetry", "extrap1"]])
@pytest.mark.parametrize("n", [(8, 9), (10, 11), (74, 75), (75, 139)])
def test_2d_faces(n, bc, oracle):
    """Faces that meet: all of a face's lines, none or some of them away from
    the corners, which a kernel treats in the directions' order."""
    problem, q0 = _block(n, "weno_js", "periodic")
    problem["bc"] = [[b, b] for b in bc]
    _check(problem, q0, oracle, f"2-D faces {n} {bc}")


@pytest.mark.parametrize("bc", ["periodic", "symmetry"])
@pytest.mark.parametrize("conv,rk,viscous", [("central_skew", "ls3", "const"), ("central_skew", "rk3", "none"),
                                             ("central_cons", "rk3", "const"), ("central_cons", "ls3", "none")])
@pytest.mark.parametrize("n", [(8, 8), (31, 9), (33, 16), (64, 15), (65, 17)])
def test_2d_central_shapes(n, conv, rk, viscous, bc, oracle):
    problem, q0 = _block(n, conv, bc, rk=rk, viscous=viscous)
    _check(problem, q0, oracle, f"2-D {n} {conv} {rk} {viscous} {bc}")


@pytest.mark.parametrize("conv,averaging", [("teno5", "roe"), ("teno6", "simple")])
@pytest.mark.parametrize("s,eps", [(1.0, 1e-16), (1.0, 1e-100), (1e25, 1e-16), (1e30, 1e-16)])
def test_2d_rough_state_in_other_units(s, eps, conv, averaging, oracle):
    """Velocities times s, pressures times s^2 on a rough state, where TENO's
    cut-off decides: the weights' quotients stay in range with the oracle's."""
    n = (24, 20)
    problem, _ = _block(n, conv, "periodic", averaging)
    problem.update(dt=0.1 * problem["dt"] / s, eps=eps)
    rs = np.random.RandomState(2)
    rho, p = (rs.uniform(0.8, 1.2, n[::-1]) for _ in range(2))
    u = [s * rs.uniform(-0.3, 0.3, n[::-1]) for _ in range(2)]
    q0 = np.stack([rho] + [rho * v for v in u] + [s * s * p / 0.4 + 0.5 * rho * (u[0] ** 2 + u[1] ** 2)])
    _check(problem, q0, oracle, f"2-D in units of {s:g}, eps={eps:g} {conv} {averaging}")


@pytest.mark.parametrize("conv", ["central_skew", "central_cons"])
@pytest.mark.parametrize("viscous", ["const", "none"])
def test_3d_central_residual_of_a_uniform_state_is_zero(viscous, conv):
    """Every first derivative is a sum of differences between points, so it
    vanishes exactly on a uniform state whose products are exact (u a power of
    two, whose second derivatives vanish as well).  T's second derivative is
    rounded: Pr = 1e300 leaves nothing of it."""
    from opensbli_amd.native import Block
    n = (70, 9, 11)
    problem, q0 = _block(n, conv, "periodic", viscous=viscous)
    u = [0.5, -0.25, 0.125]
    for k, v in enumerate([1.0] + u + [1.0 / 3.0 + 2.0]):
        q0[k] = v
    problem["Pr"] = 1e300
    print("case uniform 3-D state", conv, viscous, flush=True)
    g = Block(problem)
    g.set_state(q0)
    assert np.abs(g.rhs()).max() < 1e-280
