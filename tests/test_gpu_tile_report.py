"""echo_get_tile returns the shapes that the sweeps take: the ones a grid starts
with (chosen by the number of blocks), and after setting one sweep's shape the
others unchanged.  Whatever it returns can be set."""
import pytest

from scenarios import fireball3d, gubser2d, rmhd_fireball

pytestmark = pytest.mark.gpu


def _blocks(nx, m, other, rows):
    """Blocks of a y or z sweep of m cells: tx columns, 256 / tx rows of cells and
    one row of interfaces less, in multiples of the 8 XCDs."""
    tx = {1: 16, 2: 32}[rows]
    n = -(-nx // tx) * -(-(m + 1) // (256 // tx - 1)) * other
    return -(-n // 8) * 8


def _start(nx, ny, nz, nv):
    """The one with fewer blocks; a z sweep's 16 columns off the cache lines count
    1.05 (12 variables) or 1.1 (19)."""
    out = [1]
    for m, other in ((ny, nz), (nz, ny)):
        b1, b2 = _blocks(nx, m, other, 1), _blocks(nx, m, other, 2)
        if len(out) == 2 and nx % 16:
            b1 *= 1.1 if nv == 19 else 1.05 if nv == 12 else 1.0
        out.append(1 if m == 1 or b1 <= b2 else 2)
    return out


@pytest.mark.parametrize("nv", [5, 12, 19])
def test_weighted_choice(nv):
    """Sizes whose z sweep has as many blocks of either shape, or 8.7 % more of 32
    columns, on and off the cache lines."""
    from echoamd import EchoGrid
    expect = {(17, 16, 21): {5: 1, 12: 2, 19: 2}, (33, 20, 30): {5: 1, 12: 1, 19: 2}, (32, 16, 21): {5: 1, 12: 1, 19: 1}}
    for size, z in expect.items():
        ic, rc, _ = (rmhd_fireball if nv == 19 else fireball3d)(*size, viscosity=int(nv > 5))
        g = EchoGrid(ic, rc)
        assert g.nv == nv
        assert list(g.tile()) == _start(*size, nv) and g.tile()[2] == z[nv], size
        g.close()


@pytest.mark.parametrize("rec", ["WENO5", "MPE5"])
@pytest.mark.parametrize("size", [(24, 20, 16), (64, 14, 6), (47, 41, 29), (12, 10, 8), (33, 30, 15), (32, 32, 1)],
                         ids=lambda s: "x".join(map(str, s)))
def test_reported_shape(size, rec):
    from echoamd import EchoError, EchoGrid
    ic, rc, _ = fireball3d(*size, rec=rec) if size[2] > 1 else gubser2d(size[0], rec=rec)
    g = EchoGrid(ic, rc)
    start = _start(*size, g.nv)
    assert list(g.tile()) == start
    for d in (0, 1, 2):
        g.set_tile(d, start[d])
    assert list(g.tile()) == start
    if rec == "WENO5":
        g.set_tile(2, 4)
        assert list(g.tile()) == start[:2] + [4]
    else:
        with pytest.raises(EchoError):
            g.set_tile(2, 4)
    g.set_tile(1, 1)
    assert list(g.tile()) == [1, 1, 4 if rec == "WENO5" else start[2]]
    g.close()
