"""EnsembleSolve's value and its gradient belong to one trajectory: the value and the
pullback of n steps are, bit for bit, those of k steps followed by n - k steps from
the value after k.  With van Leer's limiter, whose branches turn a last bit of
the state into a visible change of the gradient.  And two solves may be pulled back
in any order, more than once."""
import pytest

from test_gpu_ensemble_adjoint_scratch import _make
from test_gpu_parity import _torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nlevs,nsteps,k,every", [([3], 2, 1, 1), ([32, 5, 17], 6, 3, 2), ([33, 64, 8], 9, 4, 8),
                                                  ([128, 65, 30, 3], 10, 7, 3), ([30, 63, 128] * 20, 16, 8, 5), ([40, 30], 44, 4, 2)],
                         ids=lambda v: str(v)[:16])
def test_solve_composes(nlevs, nsteps, k, every):
    torch = _torch()
    from cadycore.adjoint import EnsembleSolve

    e, Y0, w = _make(nlevs)
    D0 = torch.tensor([m.D0 for m in e.members], dtype=torch.float64)
    aw = torch.tensor([m.alpha_w for m in e.members], dtype=torch.float64)

    def solve(Y, n):
        return EnsembleSolve.apply(Y, D0, aw, e, 10.0, n, every)

    Y0.requires_grad_(True)
    whole = solve(Y0, nsteps)
    mid = solve(Y0, k)
    parts = solve(mid, nsteps - k)
    gp = torch.autograd.grad(parts, Y0, w, retain_graph=True)[0]
    gw = torch.autograd.grad(whole, Y0, w)[0]
    again = torch.autograd.grad(parts, Y0, w)[0]
    assert torch.isfinite(whole).all() and torch.isfinite(gw).all()
    assert torch.equal(whole, parts)
    assert torch.equal(gw, gp) and torch.equal(gp, again)
    assert torch.equal(gw, e.adjoint(Y0.detach(), w, 10.0, nsteps, every)[0])
    e.close()
