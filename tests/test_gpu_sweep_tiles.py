"""GPU parity of the sweeps at the edges of their tiles, and of steps that
meet a failed inversion in the middle of a call.

The sweeps work on tiles of 256 cells (x: 256 slots of the rows one after the
other, ghost cells included; y and z: 16 x 16, 32 x 8 or 8 x 32 cells, one
row of cells less in interfaces), so what can go wrong lies at tile ends, at
row ends inside a tile, in partial tiles, in dimensions shorter than a stencil
and in the periodic wrap.  Bar: relative L-infinity <= 1e-10 against the
oracle after three steps, the trajectory bar of the other tests.

Steps run without the repair's launches until a stage leaves failed cells; the
step that meets one is finished with the repair.  The same steps one at a time
and stage by stage (which always launch the repair) must give the same state
bit for bit and the same number of repairs."""
import numpy as np
import pytest

from scenarios import (fireball3d, force_superluminal, forced_background, mhd2d, mhd3d, rel_linf,
                       rmhd_fireball)

pytestmark = pytest.mark.gpu
TOL = 1e-10

# cells chosen around 256-slot tiles (x), 15-, 7- and 31-interface tiles (y, z)
SIZES = [(3, 3, 3), (5, 16, 3), (253, 3, 4), (254, 4, 3), (17, 15, 31), (31, 32, 14), (33, 7, 30), (64, 14, 6)]


def _check(oracle, ic, rc, v0, tiles=()):
    from echoamd import EchoGrid
    oracle.setup(ic, rc)
    assert oracle.init_from_prim(v0) == 0
    assert oracle.steps(3) == 0
    vo, uo = oracle.state()
    g = EchoGrid(ic, rc)
    for d, r in tiles:
        g.set_tile(d, r)
    assert g.init_from_prim(v0) == 0
    g.steps(3)
    vg, ug = g.state()
    g.close()
    ev, eu = rel_linf(vg, vo), rel_linf(ug, uo)
    assert ev <= TOL and eu <= TOL, (ev, eu)


@pytest.mark.parametrize("bc", [0, 2])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_tile_edges_vs_oracle(oracle, size, bc):
    print(f"\n{size} bc={bc}", flush=True)
    _check(oracle, *fireball3d(*size, bc=bc))


@pytest.mark.parametrize("rows", [2, 4])
@pytest.mark.parametrize("bc", [0, 2])
def test_tile_shapes_vs_oracle(oracle, rows, bc):
    _check(oracle, *fireball3d(13, 33, 9, viscosity=1, eqstate=3, bc=bc), tiles=((1, rows), (2, rows)))


@pytest.mark.parametrize("make", [
    lambda: fireball3d(255, 3, 5, viscosity=1, eqstate=3),
    lambda: mhd3d(18, 17, 16, eqstate=1, algo=5),
    lambda: mhd2d(47),
    lambda: rmhd_fireball(19, 16, 7, viscosity=0, nrk=3, bc=0),
    lambda: rmhd_fireball(6, 17, 32, viscosity=1, nrk=4),
], ids=["visc", "mhd-glm", "mhd-2d", "rmhd", "vrmhd-imex"])
def test_systems_at_tile_edges(oracle, make):
    _check(oracle, *make())


@pytest.mark.parametrize("rec", ["TVD2", "CENO3", "WENO3", "PPM4", "MPE3", "MPE5"])
def test_reconstructions_at_tile_edges(oracle, rec):
    _check(oracle, *fireball3d(17, 16, 15, rec=rec, bc=0))


@pytest.mark.parametrize("nrk", [2, 3])
def test_failed_cells_in_the_middle_of_a_call(nrk):
    from echoamd import EchoGrid

    def run(how):
        ic, rc, v0 = forced_background()
        ic = ic.copy()
        ic[10] = nrk
        g = EchoGrid(ic, rc)
        assert g.init_from_prim(v0) == 0
        g.steps(2)
        v, u = g.state()
        g.upload(v, force_superluminal(u))
        if how == "call":
            g.steps(5)
        else:
            for _ in range(5):
                if how == "steps":
                    g.steps(1)
                else:
                    for irk in range(1, nrk + 1):
                        g.rk_stage(irk)
                    g.end_step()
        out = g.state() + (g.repairs(), g.scalars())
        g.close()
        return out

    ref = run("stages")
    assert ref[2] >= 3 and ref[3]["iter"] == 7
    for how in ("call", "steps"):
        v, u, n, s = run(how)
        # (with RK2 the oracle's own run of this state holds NaNs from its
        # second step on)
        assert np.array_equal(v, ref[0], equal_nan=True) and np.array_equal(u, ref[1], equal_nan=True), how
        assert n == ref[2] and s == ref[3], (how, n, ref[2], s, ref[3])
