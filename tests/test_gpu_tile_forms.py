"""Every scheme and boundary program on each form of the tile kernels: four lanes per row in one-slice tiles, a lane
per row in two- and in four-slice tiles.  The form follows from the pool's capacity, so the meshes stay small: each
runs in a batch of that capacity, with the default schedule, against the reference's fixtures and the oracle."""
import numpy as np
import pytest

from conftest import golden, rel_diff, same_bits
from test_gpu_membership import sloshing
from test_gpu_parity import RUNS, TOL
from test_gpu_tiles import fan

pytestmark = pytest.mark.gpu

ROWS = {"four lanes": 49152, "two slices": 60000, "four slices": 200000}     # tile_slices_for
FORMS = sorted(ROWS)


def batch_of(form):
    from swe_amd.batch import Batch
    return Batch(ROWS[form], 12 * ROWS[form], 8192, 8)


def params_of(z, **kw):
    from swe_amd.solver import make_params
    g, htiny, hmax, cfl = z["scalars"]
    return make_params(gravity=g, htiny=htiny, cfl=cfl, max_water_h=hmax, **kw)


def arrays_of(z):
    from swe_amd.solver import MeshArrays
    return MeshArrays(z["ia"], z["ja"], z["cij"], z["lumped"], z["bath"], z["h_dir"], z["ux_dir"], z["uy_dir"])


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("name", sorted(RUNS))
def test_reference_runs(name, form):
    z = golden(name)
    visc, alpha, tt, mannings, bc = RUNS[name]
    amp, period, level = z["bc"] if bc == 2 else (0.0, 1.0, 0.0)
    prm = params_of(z, viscosity=visc, alpha_limit=alpha, type_test=tt, mannings=mannings)
    with batch_of(form) as b:
        k = b.add(arrays_of(z), prm, z["u0"], t0=float(z["time0"]), max_steps=z["dts"].size, bc=(bc, amp, period, level))
        done = 0
        ends = [(int(s), u) for s, u in zip(z["snap_steps"], z["snaps"])] + [(z["dts"].size, z["final"])]
        for step, ref in ends:
            print(name, form, "to step", step, flush=True)
            b.step(step - done)
            done = step
            u = b.get_state(k)
            if mannings > 0:
                assert max(rel_diff(u, ref)) <= TOL, step
            else:
                assert same_bits(u, ref), step
        st, t, steps, err = b.status(k)
        assert err == 0 and steps == z["dts"].size
        if mannings == 0:
            assert t == float(z["time"])


@pytest.mark.parametrize("form", FORMS)
def test_reference_runs_without_roundoff_fix(form):
    z, n = golden("par41_modes.npz"), golden("noround.npz")
    for tag, visc, alpha, steps in (("viscous", "viscous", False, 150), ("fct_alpha", "fct", True, 100)):
        print(form, tag, flush=True)
        prm = params_of(z, viscosity=visc, alpha_limit=alpha, type_test=5, roundoff_fix=False)
        with batch_of(form) as b:
            k = b.add(arrays_of(z), prm, z["u0"], t0=float(z["time0"]), max_steps=steps)
            b.step(steps)
            assert b.status(k)[1] == float(n["run_%s_time" % tag])
            assert same_bits(b.get_state(k), n["run_%s_final" % tag]), tag


MODES = [("galerkin", False, 2)] + [(v, a, 2) for v in ("viscous", "entropy_visc", "fct") for a in (False, True)] + \
        [("viscous", False, 1), ("viscous", True, 1)]


# meshes of 3 and 25 slices (fewer than a tile of four; a last tile of one) and one with dry islands and the inflow
@pytest.mark.parametrize("roundoff", [True, False])
@pytest.mark.parametrize("scheme,alpha,vtype", MODES)
@pytest.mark.parametrize("form", FORMS)
def test_every_scheme(oracle, form, scheme, alpha, vtype, roundoff):
    from swe_amd import problems
    from swe_amd.solver import MeshArrays, make_params
    vt = {"galerkin": oracle.GALERKIN, "fct": oracle.FCT, "viscous": oracle.VISCOUS,
          "entropy_visc": oracle.ENTROPY_VISC}[scheme]
    kw = dict(gravity=9.81, htiny=1e-4, cfl=0.25, max_water_h=1.0, type_test=4, viscous_type=vtype, alpha_limit=alpha,
              roundoff_fix=roundoff)
    cases = []
    for n, seed in ((13, 3), (40, 4)):
        p, z, u = sloshing(n, seed)
        cases.append((p, z, u, ((), (), ()), (0, 0.0, 1.0, 0.0)))
    p = problems.bumps(n_side=33)
    cases.append((p, p.bath, p.u0, p.dirichlet(), p.bc))
    prm = make_params(viscosity=scheme, **kw)
    with batch_of(form) as b:
        ids = [b.add(MeshArrays(p.ia, p.ja, p.cij, p.lumped, z, *lists), prm, u, max_steps=3, bc=bc)
               for p, z, u, lists, bc in cases]
        b.step(3)
        for k, (p, z, u, lists, bc) in zip(ids, cases):
            ref, _, rt, err = oracle.Oracle(p.ia, p.ja, p.cij, p.lumped, z, viscosity_type=vt, **kw).run(
                u, 3, bc_kind=bc[0], amp=bc[1], period=bc[2], level=bc[3], nodes_h=lists[0], nodes_ux=lists[1],
                nodes_uy=lists[2])
            assert b.status(k)[3] == err, p.np
            if err == 0:
                assert b.status(k)[1] == rt and same_bits(b.get_state(k), ref), p.np


# rows of 8, 9 and 29 entries: as many as a lane holds in registers, one more, and nearly the most a layout takes (30)
@pytest.mark.parametrize("scheme", ["fct", "viscous", "entropy_visc"])
@pytest.mark.parametrize("n", [7, 8, 28])
@pytest.mark.parametrize("form", FORMS)
def test_long_rows(oracle, form, n, scheme):
    from swe_amd.solver import MeshArrays, assemble, make_params
    rr, jj = fan(n, 12)
    ia, ja, _d, _m, lumped, cij = assemble(jj, rr)
    rng = np.random.default_rng(3)
    z = 0.1 * rng.random(rr.shape[0])
    u0 = np.zeros((rr.shape[0], 3))
    u0[:, 0] = 0.5 + 0.5 * rng.random(rr.shape[0])
    u0[:, 1:] = 0.1 * rng.normal(size=(rr.shape[0], 2))
    vt = {"fct": oracle.FCT, "viscous": oracle.VISCOUS, "entropy_visc": oracle.ENTROPY_VISC}[scheme]
    kw = dict(gravity=9.81, htiny=1e-4, cfl=0.1, max_water_h=1.0, type_test=4, alpha_limit=True)
    ref, _, rt, err = oracle.Oracle(ia, ja, cij, lumped, z, viscosity_type=vt, **kw).run(u0, 4)
    assert err == 0
    with batch_of(form) as b:
        k = b.add(MeshArrays(ia, ja, cij, lumped, z, (), (), ()), make_params(viscosity=scheme, **kw), u0, max_steps=4)
        b.step(4)
        assert b.status(k)[1] == rt and same_bits(b.get_state(k), ref)


@pytest.mark.parametrize("scheme,alpha,vtype", [("viscous", True, 2), ("viscous", False, 2), ("viscous", True, 1)])
@pytest.mark.parametrize("form", FORMS)
def test_sgn_schemes(oracle, form, scheme, alpha, vtype):
    from swe_amd.solver import MeshArrays
    z = golden("sgn_run.npz")
    lam = float(z["lambda_sgn"])
    g, htiny, hmax, cfl = z["scalars"]
    ref, _, rt, err = oracle.Oracle(z["ia"], z["ja"], z["cij"], z["lumped"], z["bath"], gravity=g, htiny=htiny, cfl=cfl,
                                    max_water_h=hmax, viscosity_type=oracle.VISCOUS, viscous_type=vtype,
                                    alpha_limit=alpha, type_test=13, lambda_sgn=lam).run(z["states"][1], 5)
    assert err == 0
    prm = params_of(z, viscosity=scheme, viscous_type=vtype, alpha_limit=alpha, type_test=13, lambda_sgn=lam)
    with batch_of(form) as b:
        k = b.add(MeshArrays(z["ia"], z["ja"], z["cij"], z["lumped"], z["bath"]), prm, z["states"][1], max_steps=5)
        b.step(5)
        assert b.status(k)[1] == rt and same_bits(b.get_state(k), ref)
