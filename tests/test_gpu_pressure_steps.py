"""The horizontal pressure differences of the explicit tendency and the
Laplacians, formed with log1p and expm1 of the relative difference to the
element's first node: a short series when every difference of a wavefront is at
most 1/4 and a longer form otherwise.  The tendency of states whose pressure
jumps by a given factor inside elements must match the float64 oracle on both
sides of that line."""
import numpy as np
import pytest

from cadycore import geometry as G
from cadycore import initial as I
from cadycore import params as P

pytestmark = pytest.mark.gpu

PAR = P.Params.from_toml()


@pytest.mark.parametrize("amp", [0.0, 0.05, 0.2, 0.6, 2.5])
def test_tendency_with_pressure_jumps_matches_oracle(amp):
    """rho and rho e_tot scaled together by a seeded factor per node in
    [1 / (1 + amp), 1 + amp]: T is unchanged and p jumps by up to (1 + amp)^2
    between the nodes of an element."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cadycore.lib import DryDycore
    from oracle import Oracle

    g = G.cubed_sphere(2, G.tanh_stretched_faces(10, 30000.0, 300.0), PAR.planet_radius, PAR.Omega)
    num = P.Numerics(dt=100.0)
    f = I.unpack(I.sphere_state(g, PAR, seed=3), g.ncol, g.nlev)
    rng = np.random.default_rng(5)
    scale = (1.0 + amp) ** rng.uniform(-1.0, 1.0, size=(g.nlev, g.n_nodes))[:, g.node_id]
    Y = I.pack(f[0] * scale, f[1], f[2], f[3] * scale, f[4]).astype(np.float32).astype(np.float64)
    d, o = DryDycore(g, PAR, num), Oracle(g, PAR, num)
    T = d.zeros()
    d.remaining_tendency(T, d.state(Y))
    got = I.unpack(T.cpu().numpy().astype(np.float64), g.ncol, g.nlev)
    d.close()
    Yo = Y.copy()
    o.set_precomputed(Yo)
    ref = I.unpack(o.remaining_tendency(Yo), g.ncol, g.nlev)
    for name, a, b in zip(I.FIELD_NAMES, got, ref):
        if name == "u3":
            a, b = a[1:-1], b[1:-1]
        err = np.linalg.norm(a - b) / np.linalg.norm(b)
        print(f"amp {amp} {name} {err:.2e}")
        assert err <= 1e-5, (amp, name, err)  # the hooks' stated gate
