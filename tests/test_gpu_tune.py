"""What swe_tune keeps: the family of kernels that runs the whole step faster, and nothing that was not timed."""
import pytest

from conftest import same_bits
from test_gpu_membership import PRM, sloshing

pytestmark = pytest.mark.gpu


def solver_of(n_side, scheme, alpha):
    from swe_amd.solver import Solver
    p, z, u = sloshing(n_side, 5)
    s = Solver(p.ia, p.ja, p.cij, p.lumped, z, viscosity=scheme, alpha_limit=alpha, **PRM)
    s.set_state(u)
    return s, p, z, u


# 4,225 nodes: four lanes per row; 63,001: two-slice tiles
@pytest.mark.parametrize("scheme,alpha", [("fct", True), ("viscous", True), ("entropy_visc", True), ("entropy_visc", False)])
@pytest.mark.parametrize("n_side", [65, 251])
def test_tuning_keeps_the_tile_kernels(oracle, n_side, scheme, alpha):
    """The gather kernels take 1.5 to 2 times as long a step at these sizes."""
    s, p, z, u = solver_of(n_side, scheme, alpha)
    vt = {"fct": oracle.FCT, "viscous": oracle.VISCOUS, "entropy_visc": oracle.ENTROPY_VISC}[scheme]
    ref, _, rt, err = oracle.Oracle(p.ia, p.ja, p.cij, p.lumped, z, viscosity_type=vt, alpha_limit=alpha, **PRM).run(u, 3)
    assert err == 0
    with s:
        sched = s.tune(steps=5)
        print(n_side, scheme, alpha, sched, flush=True)
        assert sched["k_fct_lo"][2] == 2
        # on tiles the workgroup size follows from the tile: none is chosen, and so none by noise
        assert all(b == 256 for b, _, _ in sched.values())
        assert s.run(3, time=0.0)[0] == rt and same_bits(s.get_state(), ref)


def test_entropy_viscosity_pass_is_timed():
    with solver_of(65, "entropy_visc", True)[0] as s:
        for kind in (0, 1, 2):
            s.schedule = {n: (b, r, kind if n == "k_fct_lo" else kd) for n, (b, r, kd) in s.schedule.items()}
            s.enable_kernel_timing("k_fct_lo")
            s.run(2, time=0.0)
            n, ms = s.kernel_timing("k_fct_lo")
            s.enable_kernel_timing(None)
            assert n == 6 and ms > 0.0, kind
