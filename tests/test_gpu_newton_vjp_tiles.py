"""The reverse implicit stage on tiles of 8 columns (up to 32 levels) and 4
columns (33 to 64): the pullback of two steps at the edges of both ranges,
against float64 central differences of the oracle, with the gate of the same
check at other depths (test_step_adjoint: 1e-3 for the float32 linearisation
point)."""
import numpy as np
import pytest

from cadycore import geometry as G
from cadycore import initial as I
from cadycore import params as P
from test_step_adjoint import PAR, _cotangent, _direction, _oracle_steps, _torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nlev", [3, 31, 32, 33, 63, 64])
def test_step_pullback_at_tile_edges(nlev):
    torch = _torch()
    from cadycore.lib import DryDycore

    dz = min(100.0, 15000.0 / nlev)
    g = G.cubed_sphere(2, G.tanh_stretched_faces(nlev, 30000.0, dz), PAR.planet_radius, PAR.Omega)
    num = P.Numerics(dt=100.0, vert_diff=True)
    D0 = np.full(g.n_nodes, 1.0)[g.node_id]
    Y0 = I.sphere_state(g, PAR, seed=2).astype(np.float32).astype(np.float64)
    w = _cotangent(g, _oracle_steps(g, num, D0, Y0, 2), 17)
    d = DryDycore(g, PAR, num, D0_col=D0)
    yb = d.step_adjoint(d.state(Y0), d.state(w), num.dt, 2, every=2)
    again = d.step_adjoint(d.state(Y0), d.state(w), num.dt, 2, every=2)
    assert torch.equal(yb, again)
    yb = yb.cpu().numpy().astype(np.float64)
    d.close()
    assert np.all(np.isfinite(yb))
    for field in (3, 4):
        v = _direction(g, Y0, field, 40 + field)
        eps = 1e-7
        fd = (w @ _oracle_steps(g, num, D0, Y0 + eps * v, 2)
              - w @ _oracle_steps(g, num, D0, Y0 - eps * v, 2)) / (2 * eps)
        rel = abs(float(yb @ v) - fd) / abs(fd)
        print(f"nlev {nlev} field {field}: rel {rel:.2e}")
        assert rel <= 1e-3
