"""1-D blocks with zeroth-order extrapolation ends, whose runs take the
line kernels: sizes at the edges of a wave's 63 cells, of the one-workgroup
run (1008 points) and beyond it, every scheme and RK, odd step counts, against
the oracle (relative L2 <= 1e-10 per variable); the residual afterwards (other
kernels, from the same state and halos) as well."""
import pytest

from conftest import check_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("conv,rk,averaging", [("weno_z", "rk3", "roe"), ("weno_js", "ls3", "simple"),
                                               ("teno5", "ls4", "roe"), ("teno6", "ls3_ssp", "simple")])
@pytest.mark.parametrize("n", [8, 62, 63, 64, 65, 126, 127, 1008, 1009, 1135])
def test_line_run_against_oracle(n, conv, rk, averaging, oracle):
    from opensbli_amd.native import Block
    from opensbli_amd.problems import shock_tube
    print(f"case line n={n} {conv} {rk} {averaging}", flush=True)
    problem, q0 = shock_tube(n, conv=conv, rk=rk, averaging=averaging, cfl=0.3)
    g, r = Block(problem), oracle.RefSolver(problem)
    g.set_state(q0)
    r.set_state(q0)
    for steps in (1, 6):
        g.run(steps)
        r.run(steps)
        check_parity(g.get_state(), r.get_state(), f"line n={n} {conv} {rk}")
    check_parity(g.rhs(), r.rhs(), f"line n={n} {conv} {rk} residual")
