"""The tile kernels (csrc/swe_tiles.hip, the default schedule) against the reference's fixtures and the
oracle, bit for bit: every scheme at one stage, whole runs with every boundary program, mesh sizes at the
edges of slices and tiles and in each range of the tile size, rows longer than the kernels hold in
registers, and a mesh whose halos are too long for tiles."""
import numpy as np
import pytest

from conftest import golden, same_bits

pytestmark = pytest.mark.gpu

TILES = 2     # schedule kind of k_fct_lo


def oracle_of(O, p, scheme="fct", alpha=True):
    q = p.params
    vt = {"fct": O.FCT, "viscous": O.VISCOUS, "entropy_visc": O.ENTROPY_VISC}[scheme]
    return O.Oracle(p.ia, p.ja, p.cij, p.lumped, p.bath, gravity=q["gravity"], htiny=q["htiny"], cfl=q["cfl"],
                    max_water_h=q["max_water_h"], viscosity_type=vt, alpha_limit=alpha, type_test=q["type_test"],
                    mannings=q["mannings"])


def oracle_run(O, p, steps, scheme="fct", alpha=True):
    hd, uxd, uyd = p.dirichlet()
    kind, amp, period, level = p.bc
    return oracle_of(O, p, scheme, alpha).run(p.u0, steps, bc_kind=kind, amp=amp, period=period, level=level,
                                              nodes_h=hd, nodes_ux=uxd, nodes_uy=uyd)


def test_euler_every_mode():
    from swe_amd.solver import SWE_ENEG_H, Solver, SweError
    z = golden("par41_modes.npz")
    g, htiny, hmax, cfl = z["scalars"]
    for k in range(2):
        for m, mode in enumerate(z["modes"]):
            visc, alpha, vt = str(mode).split("|")
            print("euler state", k, "mode", mode, flush=True)
            with Solver(z["ia"], z["ja"], z["cij"], z["lumped"], z["bath"], gravity=g, htiny=htiny, cfl=cfl,
                        max_water_h=hmax, viscosity=visc, viscous_type=1 if vt == "type1" else 2,
                        alpha_limit=bool(int(alpha)), type_test=5, h_dir=z["h_dir"], ux_dir=z["ux_dir"],
                        uy_dir=z["uy_dir"]) as s:
                assert s.schedule["k_fct_lo"][2] == TILES
                if z["status"][k, m] == 1:
                    with pytest.raises(SweError) as e:
                        s.euler(z["states"][k], float(z["dts"][k]))
                    assert e.value.status == SWE_ENEG_H
                else:
                    assert same_bits(s.euler(z["states"][k], float(z["dts"][k])), z["unext"][k, m]), mode


@pytest.mark.parametrize("name", ["bumps_run.npz", "cav025_run.npz"])
def test_runs_against_reference(name):
    from swe_amd.solver import Solver
    z = golden(name)
    g, htiny, hmax, cfl = z["scalars"]
    with Solver(z["ia"], z["ja"], z["cij"], z["lumped"], z["bath"], gravity=g, htiny=htiny, cfl=cfl, max_water_h=hmax,
                viscosity="fct", alpha_limit=True, type_test=4, h_dir=z["h_dir"], ux_dir=z["ux_dir"],
                uy_dir=z["uy_dir"]) as s:
        if name == "bumps_run.npz":
            s.set_bc(2, *z["bc"])
        s.set_state(z["u0"])
        t, d = s.run(z["dts"].size, time=float(z["time0"]))
        assert same_bits(d, z["dts"]) and same_bits(s.get_state(), z["final"]) and t == float(z["time"])


# 64, 529 and 33,124 nodes: one slice, a partial last slice, the two-slice tiles; 131,769: the four-slice tiles
@pytest.mark.parametrize("scheme,alpha", [("fct", True), ("fct", False), ("viscous", True), ("entropy_visc", False)])
@pytest.mark.parametrize("n_side", [8, 23, 182, 363])
def test_sizes_against_oracle(oracle, n_side, scheme, alpha):
    from swe_amd import problems
    if n_side == 363 and scheme != "fct":
        pytest.skip("the largest size once per limiter")
    from swe_amd.solver import SweError
    p = problems.bumps(n_side=n_side, viscosity=scheme, alpha=alpha)
    ref, rdts, rt, err = oracle_run(oracle, p, 3, scheme, alpha)
    for dev in (False, True):
        print(n_side, scheme, alpha, "device layout" if dev else "host layout", flush=True)
        with p.solver(device_setup=dev) as s:
            s.set_state(p.u0)
            if err:      # the scheme itself stops there (Min h<0 on a coarse mesh with islands)
                with pytest.raises(SweError) as e:
                    s.run(3, time=0.0)
                assert e.value.status == err
                continue
            t, dts = s.run(3, time=0.0)
            assert same_bits(dts, rdts) and t == rt
            assert same_bits(s.get_state(), ref)


def fan(n, rings):
    """A disk of `rings` rings of n nodes around a hub whose row has n + 1 entries."""
    a = 2.0 * np.pi * np.arange(n) / n
    rr = np.concatenate([[[0.0, 0.0]]] + [np.stack([k * np.cos(a), k * np.sin(a)], 1) for k in range(1, rings + 1)])
    jj = [[0, 1 + q, 1 + (q + 1) % n] for q in range(n)]
    for k in range(1, rings):
        o, i = 1 + k * n, 1 + (k - 1) * n
        for q in range(n):
            r = (q + 1) % n
            jj += [[i + q, o + q, o + r], [i + q, o + r, i + r]]
    return rr, np.array(jj, np.int32)


@pytest.mark.parametrize("scheme", ["fct", "viscous", "entropy_visc"])
@pytest.mark.parametrize("n", [7, 8, 28])
def test_long_rows_against_oracle(oracle, n, scheme):
    from swe_amd.solver import Solver, assemble
    rr, jj = fan(n, 6)
    ia, ja, _d, _m, lumped, cij = assemble(jj, rr)
    rng = np.random.default_rng(3)
    z = 0.1 * rng.random(rr.shape[0])
    u0 = np.zeros((rr.shape[0], 3))
    u0[:, 0] = 0.5 + 0.5 * rng.random(rr.shape[0])
    u0[:, 1:] = 0.1 * rng.normal(size=(rr.shape[0], 2))
    vt = {"fct": oracle.FCT, "viscous": oracle.VISCOUS, "entropy_visc": oracle.ENTROPY_VISC}[scheme]
    kw = dict(gravity=9.81, htiny=1e-4, cfl=0.1, max_water_h=1.0)
    ref, rdts, _t, err = oracle.Oracle(ia, ja, cij, lumped, z, viscosity_type=vt, alpha_limit=True, type_test=4,
                                       **kw).run(u0, 4)
    assert err == 0
    with Solver(ia, ja, cij, lumped, z, viscosity=scheme, alpha_limit=True, type_test=4, **kw) as s:
        s.set_state(u0)
        _, dts = s.run(4, time=0.0)
        assert same_bits(dts, rdts) and same_bits(s.get_state(), ref)


def test_scattered_numbering_runs_without_tiles(oracle, monkeypatch):
    """A random numbering kept as it is (SWE_REORDER=0): 64-row runs border on more rows than a tile holds, so
    the gather kernels run the mesh; alone and in a batch beside a mesh that could be tiled."""
    from swe_amd import mesh as M, problems
    from swe_amd.batch import Batch
    monkeypatch.setenv("SWE_REORDER", "0")
    p = problems.bumps(n_side=41)
    perm = np.random.default_rng(2).permutation(p.np)      # node k becomes perm[k]
    inv = np.argsort(perm)
    m = p.mesh
    q = problems.Problem(**{**p.__dict__, "mesh": M.Mesh(rr=m.rr[inv], jj=perm[m.jj].astype(np.int32), neigh=m.neigh,
                                                        i_d=m.i_d, jjs=perm[m.jjs].astype(np.int32), neighs=m.neighs,
                                                        sides=m.sides), "bath": p.bath[inv],
                            "u0": np.ascontiguousarray(p.u0[inv])})
    q.ia, q.ja, q.diag, _mass, q.lumped, q.cij = __import__("swe_amd.solver").solver.assemble(q.mesh.jj, q.mesh.rr)
    ref, rdts, _, err = oracle_run(oracle, q, 4)
    assert err == 0
    for dev in (False, True):
        with q.solver(device_setup=dev) as s:
            s.set_state(q.u0)
            _, dts = s.run(4, time=0.0)
            assert same_bits(dts, rdts) and same_bits(s.get_state(), ref)
    small = problems.bumps(n_side=23)
    small_ref, _, _, err = oracle_run(oracle, small, 4)
    assert err == 0
    with Batch(8192, 80000, 8192, 4) as b:
        ids = [b.add_problem(x, max_steps=4) for x in (small, q)]
        b.step(4)
        assert same_bits(b.get_state(ids[0]), small_ref) and same_bits(b.get_state(ids[1]), ref)
        b.remove(ids[1])
        again = b.add_problem(small, max_steps=4, device_setup=True)    # tiles again, on the freed rows
        b.step(4)
        assert same_bits(b.get_state(again), small_ref)
