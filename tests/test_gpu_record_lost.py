"""A reverse-mode call whose records do not fit in memory gives up the buffers of the
trajectory recorded before: the pullback of that one is refused, not run on
freed memory, and the handle records and pulls back as before."""
import numpy as np
import pytest

from cadycore import geometry as G
from cadycore import initial as I
from cadycore import params as P
from test_gpu_parity import PAR, _torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("every", [0, 1, 2])
def test_pullback_after_a_failed_request_is_refused(every):
    torch = _torch()
    from cadycore.lib import DryDycore

    g = G.cubed_sphere(2, G.tanh_stretched_faces(10, 30000.0, 300.0), PAR.planet_radius, PAR.Omega)
    d = DryDycore(g, PAR, P.Numerics(dt=50.0))
    Y0 = d.state(I.sphere_state(g, PAR, seed=4))
    rng = np.random.default_rng(1)
    w = torch.from_numpy(rng.standard_normal(Y0.numel()).astype(np.float32)).to(Y0) / (Y0.abs() + 1.0)

    def record():
        Y = Y0.clone()
        d.step_record(Y, 50.0, 2, every)
        return Y

    Y = record()
    ref = d.step_pullback(w)
    with pytest.raises(RuntimeError, match="memory"):
        d.step_adjoint(Y0, w, 50.0, 1, every=1 << 30)  # a thousand times the card's memory
    with pytest.raises(RuntimeError, match="no trajectory"):
        d.step_pullback(w)
    assert torch.equal(record(), Y)
    assert torch.equal(d.step_pullback(w), ref)
    assert torch.isfinite(ref).all()
    d.close()
