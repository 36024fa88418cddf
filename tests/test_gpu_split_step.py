"""Calls between swe_step_begin and swe_step_finish: the first stage takes nothing from the dt pass that they may
have replaced or that the dt pass was not asked for."""
import numpy as np
import pytest

from conftest import same_bits
from test_gpu_membership import PRM, sloshing
from test_gpu_tiles import oracle_run

pytestmark = pytest.mark.gpu


# 1,681 nodes: four lanes per row; 52,900: two-slice tiles
@pytest.mark.parametrize("scheme", ["fct", "viscous"])
@pytest.mark.parametrize("n_side", [41, 230])
def test_euler_of_another_state_in_between(oracle, n_side, scheme):
    from swe_amd import problems
    p = problems.bumps(n_side=n_side, viscosity=scheme)
    ref, rdts, _, err = oracle_run(oracle, p, 2, scheme)
    assert err == 0
    other = p.u0.copy()
    other[:, 0] *= 0.9 + 0.1 * np.random.default_rng(4).random(p.np)
    with p.solver() as s:
        s.set_state(p.u0)
        s.time = 0.0
        for k in range(2):
            dt = s.step_begin()
            assert dt == rdts[k]
            s.euler(other, dt)
            s.step_finish()
        assert same_bits(s.get_state(), ref)


@pytest.mark.parametrize("scheme", ["fct", "viscous"])
@pytest.mark.parametrize("n_side", [41, 230])
def test_limiter_switched_on_in_between(oracle, n_side, scheme):
    from swe_amd import problems
    p = problems.bumps(n_side=n_side, viscosity=scheme)
    ref, rdts, _, err = oracle_run(oracle, p, 1, scheme)
    assert err == 0
    with p.solver(alpha_limit=False) as s:
        s.set_state(p.u0)
        s.time = 0.0
        assert s.step_begin() == rdts[0]
        s.set_params(**p.params)
        s.step_finish()
        assert same_bits(s.get_state(), ref)


@pytest.mark.parametrize("between", ["parameters", "state", "positivity", "run"])
@pytest.mark.parametrize("n_side", [41, 230])
def test_nothing_of_the_dt_pass_where_its_inputs_changed(oracle, n_side, between):
    """The stages are compute_dij's and euler's at the state and parameters of swe_step_finish, as in the reference, whose
    euler evaluates d_ij itself: after parameters or a state were set, and after calls that use the d_ij's memory."""
    from swe_amd.solver import Solver
    p, z, u = sloshing(n_side, 6)
    scheme = "galerkin" if between == "parameters" else "viscous"
    orc = oracle.Oracle(p.ia, p.ja, p.cij, p.lumped, z, viscosity_type=oracle.VISCOUS, alpha_limit=True, **PRM)
    with Solver(p.ia, p.ja, p.cij, p.lumped, z, viscosity=scheme, alpha_limit=True, **PRM) as s:
        s.set_state(u)
        s.time = 0.0
        dt = s.step_begin()
        if between == "parameters":
            s.set_params(viscosity="viscous")
        elif between == "state":
            u = u.copy()
            u[:, 1:] *= -0.5
            s.set_state(u)
        elif between == "run":
            _, dts = s.run(1)
            u = s.get_state()
            dt = dts[0]
        else:
            s.fct_positivity(np.ones(p.np), np.linspace(-1.0, 1.0, p.nnz))
        s.step_finish()
        u1 = orc.euler(u, dt)[0]
        u2 = (3.0 * u + orc.euler(u1, dt)[0]) / 4.0
        assert same_bits(s.get_state(), (u + 2.0 * orc.euler(u2, dt)[0]) / 3.0)
