"""con2prim of states whose conserved energy or density is infinite, zero,
NaN, denormal or far outside the range of a run, against the oracle, whose
quotients are divisions: the same status, the same components finite, and the
finite ones within the 1e-10 of the other batch tests.  A state that cannot be
inverted must be reported (a run repairs it from its neighbours)."""
import numpy as np
import pytest

from scenarios import fireball3d, rmhd_fireball

pytestmark = pytest.mark.gpu

SPECIAL = [np.inf, -np.inf, np.nan, 0.0, -0.0, 5e-324, 1e-310, 1e-200, 1e-160, 1e-30, 1e30, 1e160, 1e200,
           1e308, -1.0, -1e-3]


@pytest.mark.parametrize("eqstate", [1, 2, 3])
@pytest.mark.parametrize("system", ["hydro", "viscous", "rmhd", "vrmhd"])
def test_special_energies_and_densities(oracle, system, eqstate):
    from echoamd import EchoGrid
    visc = system in ("viscous", "vrmhd")
    make = rmhd_fireball if "rmhd" in system else fireball3d
    ic, rc, v0 = make(6, 5, 4, viscosity=int(visc), eqstate=eqstate)
    oracle.setup(ic, rc)
    assert oracle.init_from_prim(v0) == 0
    v, u = (a.reshape(a.shape[0], -1)[:, ::30] for a in oracle.state())
    U, G = [u], [v]
    for s in SPECIAL:
        for k, rest in ((4, False), (4, True), (0, False)):
            a = u.copy()
            if rest:
                a[1:4] = 0.0
            a[k] = s
            U.append(a)
            G.append(v)
    U, G = np.ascontiguousarray(np.concatenate(U, 1)), np.ascontiguousarray(np.concatenate(G, 1))
    g = EchoGrid(ic, rc)
    vg, st = g.cons2prim_batch(U, G)
    g.close()
    for i in range(U.shape[1]):
        e, vo, _ = oracle.cons2prim(U[:, i], G[:, i])
        assert st[i] == e, (U[:, i], st[i], e)
        fin = np.isfinite(vo)
        assert np.array_equal(np.isfinite(vg[:, i]), fin), (U[:, i], vg[:, i], vo)
        if e == 0 and fin.any():
            assert np.abs(vg[fin, i] - vo[fin]).max() <= 1e-10 * np.abs(vo[fin]).max(), (U[:, i], vg[:, i], vo)
    inf_energy = np.isinf(U[4])
    assert eqstate != 3 or (st[inf_energy] != 0).all()
