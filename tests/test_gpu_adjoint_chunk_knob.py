"""The reverse-mode chunk may be set to 8 levels or more after the workspace
exists, also where the default is larger (9 at this size)."""
import numpy as np
import pytest

from cadycore import geometry as G
from cadycore import initial as I
from cadycore import params as P
from test_gpu_parity import PAR, _torch

pytestmark = pytest.mark.gpu


def test_chunk_of_eight_after_the_first_reverse_call():
    torch = _torch()
    from cadycore.lib import CA_TUNE_ADJ_CHUNK, DryDycore

    g = G.cubed_sphere(15, G.tanh_stretched_faces(100, 30000.0, 30.0), PAR.planet_radius, PAR.Omega)
    rng = np.random.default_rng(3)
    d = DryDycore(g, PAR, P.Numerics(dt=50.0, vert_diff=True), D0_col=rng.uniform(0.1, 50.0, g.ncol))
    Y = d.state(I.sphere_state(g, PAR, seed=1))
    w = torch.from_numpy(rng.standard_normal(Y.numel()).astype(np.float32)).to(Y) / (Y.abs() + 1.0)

    def vjp():
        D0b = torch.zeros(g.ncol, dtype=torch.float32, device=Y.device)
        Yb = d.zeros()
        d.remaining_tendency_vjp(Yb, w, Y, D0b=D0b)
        return Yb, D0b

    ref, refD = vjp()
    assert d.get_tuning(CA_TUNE_ADJ_CHUNK) == 9
    for chunk in (8, 12):
        d.set_tuning(CA_TUNE_ADJ_CHUNK, chunk)
        got, D = vjp()
        assert torch.isfinite(got).all()
        # chunks only move float32 rounding between levels (a handful of sums)
        assert torch.linalg.norm(got - ref) <= 16 * 2.0 ** -24 * torch.linalg.norm(ref)
        assert torch.linalg.norm(D - refD) <= 16 * 2.0 ** -24 * torch.linalg.norm(refD)
    with pytest.raises(RuntimeError, match="cannot shrink"):
        d.set_tuning(CA_TUNE_ADJ_CHUNK, 7)
    d.close()
