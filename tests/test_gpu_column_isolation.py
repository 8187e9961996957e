"""Columns of a sphere are solved side by side, two to a wavefront up to 64 levels:
a column that is not finite must leave every other column of the solve bitwise
what it is beside finite ones, whichever of the two it is, at the edges of the
lane shapes (32 and 64 levels fill every lane)."""
import numpy as np
import pytest

from cadycore import geometry as G
from cadycore import initial as I
from cadycore import params as P
from test_gpu_parity import PAR, _torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nlev", [3, 31, 32, 33, 63, 64, 65, 128])
@pytest.mark.parametrize("where", ["residual", "state"])
def test_solve_of_one_column_does_not_reach_another(nlev, where):
    torch = _torch()
    from cadycore.lib import DryDycore

    g = G.cubed_sphere(2, G.tanh_stretched_faces(nlev, 30000.0, 200.0), PAR.planet_radius, PAR.Omega)
    d = DryDycore(g, PAR, P.Numerics(hyperdiff=False, rayleigh=True, dt=20.0))
    Y = d.state(I.sphere_state(g, PAR, seed=4))
    rng = np.random.default_rng(7)
    R = Y * torch.from_numpy(1e-3 * rng.standard_normal(Y.numel()).astype(np.float32)).to(Y)
    dtg = 0.4358665215 * 20.0

    def solve(bad, value):
        Yb, Rb = Y.clone(), R.clone()
        if bad is not None:
            (Rb if where == "residual" else Yb).view(-1, g.ncol)[:4 * nlev, bad] = value
        d.update_jacobian(Yb, dtg)
        dY = d.zeros()
        d.ldiv(dY, Rb)
        return dY.view(-1, g.ncol)

    clean = solve(None, 0.0)
    assert torch.isfinite(clean).all()
    for bad, value in ((0, float("nan")), (5, float("nan")), (16, float("inf")), (g.ncol - 1, -float("inf"))):
        got = solve(bad, value)
        keep = [c for c in range(g.ncol) if c != bad]
        assert torch.equal(got[:, keep], clean[:, keep]), (bad, value)
        assert not torch.isfinite(got[:4 * nlev, bad]).all()
    d.close()
