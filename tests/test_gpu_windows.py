"""Meshes whose halos are too long for tiles keep rows sorted inside single slices: seen by the entry slots that a batch
gives them (64 x the longest row of each 64 rows of the caller's order), with the results of the oracle."""
import numpy as np
import pytest

from conftest import same_bits

pytestmark = pytest.mark.gpu

PRM = dict(gravity=9.81, htiny=1e-4, cfl=0.25, max_water_h=1.0, type_test=4)


def slots(ia, rows_per_window):
    """Slots of rows sorted by length inside windows of so many, padded to 64-row slices."""
    n = np.diff(ia)
    n = np.concatenate([np.sort(n[k:k + rows_per_window]) for k in range(0, n.size, rows_per_window)])
    n = np.concatenate([n, np.zeros(-n.size % 64, n.dtype)])
    return int(64 * n.reshape(-1, 64).max(1).sum())


@pytest.mark.parametrize("device", [False, True])
@pytest.mark.parametrize("scattered", [True, False])
@pytest.mark.parametrize("rows,window", [(49152, 64), (60000, 128), (200000, 256)])
def test_slots_and_results(oracle, monkeypatch, rows, window, scattered, device):
    from swe_amd import problems
    from swe_amd.batch import Batch
    from swe_amd.solver import MeshArrays, assemble, make_params
    monkeypatch.setenv("SWE_REORDER", "0")
    p = problems.bumps(n_side=41)
    order = np.random.default_rng(2).permutation(p.np) if scattered else np.arange(p.np)
    inv = np.argsort(order)
    jj, rr, z = order[p.mesh.jj].astype(np.int32), np.ascontiguousarray(p.mesh.rr[inv]), 0.3 * p.bath[inv] / p.bath.max()
    ia, ja, _d, _m, lumped, cij = assemble(jj, rr)
    u = np.zeros((p.np, 3))
    u[:, 0] = 1.0 - z + 0.05 * np.random.default_rng(3).random(p.np)
    want = slots(ia, 64 if scattered else window)
    ref, _, rt, err = oracle.Oracle(ia, ja, cij, lumped, z, viscosity_type=oracle.FCT, alpha_limit=True, **PRM).run(u, 3)
    assert err == 0
    prm = make_params(viscosity="fct", alpha_limit=True, **PRM)
    entries = 12 * rows
    with Batch(rows, entries, 64, 2) as b:
        if device:
            k = b.add_elements(jj, rr, z, prm, u, max_steps=3)
        else:
            k = b.add(MeshArrays(ia, ja, cij, lumped, z), prm, u, max_steps=3)
        assert entries - b.free()[1] == want
        b.step(3)
        assert b.status(k)[1] == rt and same_bits(b.get_state(k), ref)
