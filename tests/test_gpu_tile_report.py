"""echo_get_tile returns the shapes that the sweeps take: the ones a grid starts
with (chosen by the number of blocks), and after setting one sweep's shape the
others unchanged.  Whatever it returns can be set."""
import pytest

from scenarios import fireball3d, gubser2d

pytestmark = pytest.mark.gpu


def _blocks(nx, m, other, rows):
    """Blocks of a y or z sweep of m cells: tx columns, 256 / tx rows of cells and
    one row of interfaces less, in multiples of the 8 XCDs."""
    tx = {1: 16, 2: 32}[rows]
    n = -(-nx // tx) * -(-(m + 1) // (256 // tx - 1)) * other
    return -(-n // 8) * 8


def _start(nx, ny, nz):
    out = [1]
    for m, other in ((ny, nz), (nz, ny)):
        b1, b2 = _blocks(nx, m, other, 1), _blocks(nx, m, other, 2)
        out.append(1 if m == 1 or b1 * (1.1 if nx % 16 else 1.0) <= b2 else 2)
    return out


@pytest.mark.parametrize("rec", ["WENO5", "MPE5"])
@pytest.mark.parametrize("size", [(24, 20, 16), (64, 14, 6), (47, 41, 29), (12, 10, 8), (33, 30, 15), (32, 32, 1)],
                         ids=lambda s: "x".join(map(str, s)))
def test_reported_shape(size, rec):
    from echoamd import EchoError, EchoGrid
    ic, rc, _ = fireball3d(*size, rec=rec) if size[2] > 1 else gubser2d(size[0], rec=rec)
    g = EchoGrid(ic, rc)
    start = _start(*size)
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
