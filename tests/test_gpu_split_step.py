"""Calls between swe_step_begin and swe_step_finish: the first stage takes nothing from the dt pass that they may
have replaced or that the dt pass was not asked for."""
import numpy as np
import pytest

from conftest import same_bits
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
