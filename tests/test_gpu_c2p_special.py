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


def test_cubic_without_quadratic_term():
    """Algorithm 5 where the cubic c3 W^3 + c2 W^2 - (S.B)^2/2 = 0 has c2 = 0:
    its Newton iteration starts at the cube root and stops there (its next
    correction is below 1e-12 W, which is not applied), so the root must hold to
    rounding.  Bar: with u = 2^-53, the rounding of the eight inputs and of some
    ten operations on v = (S + (v.B) B) / (W + B^2) is a few u; the median
    relative error of v stays below 8 u."""
    from echoamd import EchoGrid
    from scenarios import mhd3d
    rng = np.random.default_rng(3)
    n = 20000
    speed = rng.uniform(0.05, 0.9, n)
    d = rng.standard_normal((3, n))
    d /= np.linalg.norm(d, axis=0)
    p = rng.uniform(0.9, 1.1, n) * 10 ** rng.uniform(-3, 2, n)
    L = np.longdouble
    v, W = L(1) * speed * d, 4 * L(1) * p / (1 - L(1) * speed ** 2)
    # c2 = 0 is (v.B)^2 = 2 (W - p); any field across v may be added
    along = np.sqrt(2 * (W - p)) / speed
    e = rng.standard_normal((3, n))
    e -= d * (e * d).sum(0)
    e /= np.linalg.norm(e, axis=0)
    B = np.asarray(along * d + along * rng.uniform(0, 1, n) * e, dtype=float)
    v2, B2, vb = (v * v).sum(0), (L(1) * B * B).sum(0), (v * B).sum(0)
    W = 4 * p / (1 - v2)
    u = np.concatenate([(1 / np.sqrt(1 - v2))[None], (W + B2) * v - vb * B,
                        (W - p + (B2 + B2 * v2 - vb * vb) / 2)[None], B])
    guess = np.concatenate([np.ones((1, n)), np.asarray(v * (1 + 1e-3 * rng.standard_normal(n)), dtype=float),
                            p[None], B])
    ic, rc, _ = mhd3d(6, 5, 4, eqstate=1, algo=5, coordinates=1, divclean=0)
    g = EchoGrid(ic, rc)
    vg, st = g.cons2prim_batch(np.ascontiguousarray(u, dtype=float), np.ascontiguousarray(guess))
    g.close()
    assert not st.any()
    err = np.abs(vg[1:4] - v).max(0) / speed
    assert np.median(err) <= 8 * 2.0 ** -53, np.median(err)
