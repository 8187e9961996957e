"""The horizontal pressure differences inside an element take a short series or a
longer form by their size.  The choice belongs to each node: an element with
large differences must leave the tendency of every element that shares no node
with it bitwise what it is beside smooth ones (four elements share a wavefront)."""
import numpy as np
import pytest

from cadycore import geometry as G
from cadycore import initial as I
from test_gpu_parity import PAR, _torch
from cadycore import params as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("factor", [1.2, 1.6, 20.0, float("nan")])
@pytest.mark.parametrize("hyperdiff", [False, True])
def test_large_differences_stay_in_their_element(hyperdiff, factor):
    torch = _torch()
    from cadycore.lib import DryDycore

    g = G.cubed_sphere(4, G.tanh_stretched_faces(10, 30000.0, 300.0), PAR.planet_radius, PAR.Omega)
    d = DryDycore(g, PAR, P.Numerics(dt=100.0, hyperdiff=hyperdiff))
    Y = d.state(I.sphere_state(g, PAR, seed=3))
    node = np.asarray(g.node_id).reshape(-1, 16)

    def tendency(e):
        Yb, T = Y.clone(), d.zeros()
        if e is not None:  # rho and rho e_tot of every other node: T stays, p jumps
            v = Yb.view(-1, g.ncol)
            v[:g.nlev, 16 * e + 1:16 * e + 16:2] *= factor
            v[3 * g.nlev:4 * g.nlev, 16 * e + 1:16 * e + 16:2] *= factor
        d.remaining_tendency(T, Yb)
        return T.view(-1, node.shape[0], 16)

    clean = tendency(None)
    assert torch.isfinite(clean).all()
    for e in (0, 1, 6, node.shape[0] - 1):
        apart = [k for k in range(node.shape[0]) if not np.intersect1d(node[k], node[e]).size]
        assert any(k // 4 == e // 4 for k in apart)  # one of them in the same wavefront
        got = tendency(e)
        assert torch.equal(got[:, apart], clean[:, apart]), e
        assert not torch.equal(got[:, e], clean[:, e])
    d.close()
