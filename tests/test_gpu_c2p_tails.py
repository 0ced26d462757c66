"""The learned inversion at the edges of its tiles of 64 states, of its blocks
of four tiles and of a launch's blocks (a wave takes its next tile while it
works on this one).

A state's result comes from the same instructions wherever it stands in a
batch, so a batch of n states gives bit for bit what the same states give
within a longer one; the longer one is held to the exact primitives within
1e-10, the accuracy the network's three Newton iterations are made for.
"""
import numpy as np
import pytest

from test_gpu_c2p_mlp import _dev, _scales, _snap, _weights_or_skip

pytestmark = pytest.mark.gpu

LONG = 3 * 256 * 4 * 64 * 2 + 65      # two tiles a wave and a ragged rest on 256 CUs


def _invert(net, g, u, guess):
    n = u.shape[1]
    du, dv, ds = _dev(u), _dev(guess), _dev(np.full(n, -7, dtype=np.int32))
    net.invert(g, du.ptr, dv.ptr, ds.ptr, n, iters=3)
    return dv.numpy(), ds.numpy()


@pytest.mark.parametrize("divclean", [0, 1])
def test_tails(divclean):
    from echoamd import C2pNet
    from echoamd.surrogate import e3p_grid, mhd_e3p_states
    P = _weights_or_skip()
    g = e3p_grid(0, divclean=divclean)
    u, vt, vw = mhd_e3p_states(LONG, _snap(), seed=7)
    if divclean:
        psi = np.linspace(-0.01, 0.01, LONG)[None]
        u, vw = np.concatenate([u, psi]), np.concatenate([vw, 0 * psi])
    net = C2pNet(0, P)
    v, st = _invert(net, g, u, vw)
    assert np.all(st == 0)
    assert (np.abs(v[:8] - vt) / _scales(vt)).max() <= 1e-10
    if divclean:
        assert np.array_equal(v[8], u[8])
    for n in (1, 63, 64, 65, 255, 256, 257, 4097):
        a = LONG - n                  # the last n states
        vn, sn = _invert(net, g, np.ascontiguousarray(u[:, a:]), np.ascontiguousarray(vw[:, a:]))
        assert np.array_equal(sn, st[a:]), n
        assert np.array_equal(vn, v[:, a:]), n
    net.close()
    g.close()
