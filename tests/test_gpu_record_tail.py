"""The stage records of a recorded run's last checkpoint segment are kept for its
pullback: a second pullback of the same record, and records of one and of
several segments, give bitwise the same cotangents as records of every step."""
import numpy as np
import pytest

from cadycore import geometry as G
from cadycore import initial as I
from cadycore import params as P

pytestmark = pytest.mark.gpu

PAR = P.Params.from_toml()


@pytest.mark.parametrize("nsteps,every", [(1, 1), (3, 8), (4, 4), (5, 2), (5, 3)])
@pytest.mark.parametrize("poison", [False, True])
def test_pullback_with_kept_segment_is_bitwise_and_repeatable(nsteps, every, poison):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cadycore.lib import DryDycore

    g = G.cubed_sphere(2, G.tanh_stretched_faces(10, 30000.0, 300.0), PAR.planet_radius, PAR.Omega)
    num = P.Numerics(dt=100.0, vert_diff=True)
    rng = np.random.default_rng(3)
    D0 = rng.uniform(1.0, 50.0, size=g.n_nodes)[g.node_id]
    d = DryDycore(g, PAR, num, D0_col=D0)
    d.set_debug_poison(poison)
    Y0 = d.state(I.sphere_state(g, PAR, seed=3))
    Yb = d.state(rng.standard_normal(d.S))

    def gradient(ev, pulls):
        out = []
        d.step_record(Y0.clone(), 100.0, nsteps, ev)
        for _ in range(pulls):
            b = torch.zeros(g.ncol, device=Y0.device)
            out.append((d.step_pullback(Yb, b).clone(), b))
        return out

    (ref,) = gradient(0, 1)
    for y, b in gradient(every, 2):
        assert torch.isfinite(y).all() and torch.isfinite(b).all()
        assert torch.equal(y, ref[0]) and torch.equal(b, ref[1])
    d.close()
