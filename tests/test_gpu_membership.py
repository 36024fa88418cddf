"""Batches whose meshes change while the captured step is replayed, in pools of two- and four-slice tiles: other
meshes of as many slices can have more or fewer tiles, so the launches are other ones."""
import numpy as np
import pytest

from conftest import same_bits

pytestmark = pytest.mark.gpu

PRM = dict(gravity=9.81, htiny=1e-4, cfl=0.25, max_water_h=1.0, type_test=4)


def sloshing(n_side, seed):
    """A wet basin without Dirichlet nodes: (mesh arrays, bathymetry, state)."""
    from swe_amd import problems
    p = problems.bumps(n_side=n_side, seed=seed)
    rng = np.random.default_rng(seed)
    z = 0.3 * p.bath / p.bath.max()
    u = np.zeros((p.np, 3))
    u[:, 0] = 1.0 - z + 0.05 * rng.random(p.np)
    u[:, 1:] = 0.05 * rng.normal(size=(p.np, 2))
    return p, z, u


# (pool rows, sides of the meshes that leave, of those that come): tiles of two slices, 5 + 3 slices are 5 tiles and
# 4 + 4 are 4; tiles of four, 3 and 2
@pytest.mark.parametrize("rows", [60000, 200000])
@pytest.mark.parametrize("first,then", [((17, 13), (15, 16)), ((15, 16), (17, 13))])
def test_other_meshes_of_as_many_slices(oracle, rows, first, then):
    from swe_amd.batch import Batch
    from swe_amd.solver import MeshArrays, make_params
    prm = make_params(viscosity="fct", alpha_limit=True, **PRM)
    big = sloshing(40, 1)
    sets = [[sloshing(n, 10 * n + k) for k, n in enumerate(s)] for s in (first, then)]
    assert [sum((p.np + 63) // 64 for p, _, _ in s) for s in sets] == [8, 8]
    steps = {}

    def state_of(case, n):
        p, z, u = case
        ref, _, rt, err = oracle.Oracle(p.ia, p.ja, p.cij, p.lumped, z, viscosity_type=oracle.FCT, alpha_limit=True,
                                        **PRM).run(u, n)
        assert err == 0
        return ref, rt

    with Batch(rows, 9 * rows, 64, 4) as b:
        def add(case):
            p, z, u = case
            return b.add(MeshArrays(p.ia, p.ja, p.cij, p.lumped, z, [], [], []), prm, u)
        kb = add(big)
        total = 0
        for s in sets + sets:                     # there, and back onto the first step captured for the others
            ids = [add(c) for c in s]
            for part in (1, 2):
                b.step(part)
                b.sync()
                total += part
            print("pool of", rows, "rows, meshes of", [c[0].np for c in s], "after", total, "steps", flush=True)
            for k, c in zip(ids, s):
                ref, rt = state_of(c, 3)
                assert b.status(k)[1] == rt and same_bits(b.get_state(k), ref)
                b.remove(k)
        ref, rt = state_of(big, total)
        assert b.status(kb)[1] == rt and same_bits(b.get_state(kb), ref)


def test_another_model_on_the_same_rows(oracle):
    """An emptied batch takes another model: the five components of test 13 after the three of test 11, whose step has
    the same launch extents and scheme."""
    from conftest import golden
    from swe_amd.batch import Batch
    from swe_amd.solver import MeshArrays, make_params
    z = golden("sgn_run.npz")
    g, htiny, hmax, cfl = z["scalars"]
    kw = dict(gravity=g, htiny=htiny, cfl=cfl, max_water_h=hmax, alpha_limit=True)
    with Batch(8192, 80000, 64, 2) as b:
        for tt, lam, u in ((11, 0.0, np.ascontiguousarray(z["states"][1][:, :3])), (13, float(z["lambda_sgn"]), z["states"][1])):
            ref, _, rt, err = oracle.Oracle(z["ia"], z["ja"], z["cij"], z["lumped"], z["bath"], type_test=tt, lambda_sgn=lam,
                                            viscosity_type=oracle.VISCOUS, **kw).run(u, 4)
            assert err == 0
            k = b.add(MeshArrays(z["ia"], z["ja"], z["cij"], z["lumped"], z["bath"]),
                      make_params(viscosity="viscous", type_test=tt, lambda_sgn=lam, **kw), u)
            b.step(4)
            assert b.status(k)[1] == rt and same_bits(b.get_state(k), ref), tt
            b.remove(k)
