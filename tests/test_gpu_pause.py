"""Steps that meet a failed inversion, on grids and in places where what
follows the failed stage must be held back until the repair.

echo_steps launches steps without the repair until one needs it.  The same
steps stage by stage (echo_rk_stage, which always launches the repair) must
give the same state bit for bit, the same number of repairs and the same
scalars."""
import numpy as np
import pytest

from echoamd.initial import make_config
from scenarios import force_superluminal, mhd_fireball3d

pytestmark = pytest.mark.gpu


def _advance(g, n, how):
    if how == "call":
        g.steps(n)
        return
    for _ in range(n):
        for irk in range(1, g.cfg.nrk + 1):
            g.rk_stage(irk)
        g.end_step()


def _same(a, b):
    assert np.all(np.isfinite(a[0])) and np.all(np.isfinite(a[1]))
    assert a[2] == b[2] and a[3] == b[3], (a[2:], b[2:])
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("nrk", [2, 3])
@pytest.mark.parametrize("viscosity", [0, 1])
@pytest.mark.parametrize("coordinates", [1, 2])
def test_single_cell(coordinates, viscosity, nrk):
    """One cell has no sweep between its stages.  Its conserved state is
    superluminal, so the inversion fails in every stage of the first step."""
    from echoamd import EchoGrid
    ic, rc = make_config(nx=1, ny=1, nz=1, coordinates=coordinates, viscosity=viscosity, bulk=1, eqstate=1,
                         nrk=nrk, init_type=0, maxdt=0.05)
    v0 = np.zeros((12 if viscosity else 5, 1, 1, 1))
    v0[0], v0[1], v0[4] = 1.0, 0.3, 0.5

    def run(how):
        g = EchoGrid(ic, rc)
        assert g.init_from_prim(v0) == 0
        g.steps(2)
        v, u = g.state()
        g.upload(v, force_superluminal(u, ((0, 0, 0),)))
        _advance(g, 3, how)
        out = g.state() + (g.repairs(), g.scalars())
        g.close()
        return out

    ref = run("stages")
    assert ref[2] == nrk and ref[3]["iter"] == 5
    _same(run("call"), ref)


def test_ensemble_tune_between_stages():
    """The ensemble's tuner may run while an event is inside a step; its sweeps
    change nothing of that step, the cleaning speed of the next stage (the
    speeds of this one's sweeps) included."""
    from echoamd import Ensemble
    ic, rc, v0 = mhd_fireball3d(20, 18, 12)
    v0[1] *= 0.1      # the y sweep, which the tuner runs, has the largest speed

    def run(tune):
        ens = Ensemble([(ic, rc)])
        g = ens.grids[0]
        assert g.init_from_prim(v0) == 0
        ens.steps(2)
        for irk in (1, 2, 3):
            g.rk_stage(irk)
            if tune and irk < 3:
                ens.tune(reps=1)
        g.end_step()
        out = g.state() + (g.repairs(), g.scalars())
        ens.close()
        return out

    _same(run(True), run(False))
