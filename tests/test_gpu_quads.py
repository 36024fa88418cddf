"""The four-lanes-per-row kernels (csrc/swe_quads.hip, pools of up to 49,152 rows) against the oracle, bit for
bit: a mesh of one partial slice, a partial last slice, the largest mesh they take, and several meshes that
share each launch, one of which stops first."""
import pytest

from conftest import same_bits
from test_gpu_tiles import oracle_run

pytestmark = pytest.mark.gpu

SCHEMES = [("fct", True), ("fct", False), ("viscous", True), ("viscous", False), ("entropy_visc", True)]


@pytest.mark.parametrize("scheme,alpha", SCHEMES)
@pytest.mark.parametrize("n_side", [5, 17, 181, 221])
def test_sizes_against_oracle(oracle, n_side, scheme, alpha):
    from swe_amd import problems
    from swe_amd.solver import SweError
    p = problems.bumps(n_side=n_side, viscosity=scheme, alpha=alpha)
    ref, rdts, rt, err = oracle_run(oracle, p, 3, scheme, alpha)
    with p.solver() as s:
        s.set_state(p.u0)
        if err:
            with pytest.raises(SweError) as e:
                s.run(3, time=0.0)
            assert e.value.status == err
            return
        t, dts = s.run(3, time=0.0)
        assert same_bits(dts, rdts) and t == rt and same_bits(s.get_state(), ref)


def test_meshes_sharing_a_launch(oracle):
    from swe_amd import problems
    from swe_amd.batch import Batch
    ps = [problems.bumps(n_side=n) for n in (23, 41, 29)]
    steps = (4, 2, 4)
    with Batch(8192, 80000, 8192, 4) as b:
        ids = [b.add_problem(p, max_steps=n) for p, n in zip(ps, steps)]
        b.step(4)
        for k, p, n in zip(ids, ps, steps):
            ref, _, rt, err = oracle_run(oracle, p, n)
            assert err == 0 and b.status(k)[1] == rt and same_bits(b.get_state(k), ref)


@pytest.mark.parametrize("n_side", [41, 200])
@pytest.mark.parametrize("before,after", [(0, 2), (2, 0)])
def test_schedule_set_between_the_parts_of_a_step(oracle, n_side, before, after):
    """What the dt pass leaves for the first stage differs between the tile and the gather kernels."""
    from swe_amd import problems
    p = problems.bumps(n_side=n_side)
    ref, rdts, _, err = oracle_run(oracle, p, 2)
    assert err == 0
    with p.solver() as s:
        s.set_state(p.u0)
        s.time = 0.0
        for k in range(2):
            s.schedule = {n: (b, r, before if n == "k_fct_lo" else kd) for n, (b, r, kd) in s.schedule.items()}
            assert s.step_begin() == rdts[k]
            s.schedule = {n: (b, r, after if n == "k_fct_lo" else kd) for n, (b, r, kd) in s.schedule.items()}
            s.step_finish()
        assert same_bits(s.get_state(), ref)
