"""ca_ensemble_adjoint has two schedules: every step's stage states kept (three
launches) and checkpoints with recomputed segments (the no-allocation entry
always).  They run the same step and reverse functions, so they agree up to the
order in which a compiler may contract a product and a sum."""
import numpy as np
import pytest

from cadycore import geometry as G
from cadycore import initial as I
from cadycore import params as P
from test_gpu_parity import PAR, _torch

pytestmark = pytest.mark.gpu

# One member-lane of the widest LDS shape, its neighbours, and every shape's
# lane count (33, 65 and 129 faces).
CASES = [
    ([3], 1, 1),
    ([32, 5, 17], 5, 2),
    ([33, 64, 8], 4, 3),
    ([128, 65, 30, 3], 3, 8),
    ([30] * 300, 2, 1),
]


@pytest.mark.parametrize("nlevs,nsteps,every", CASES, ids=lambda v: str(v)[:16])
def test_kept_states_match_recomputed_segments(nlevs, nsteps, every):
    torch = _torch()
    from cadycore.ensemble import ColumnEnsemble, Member

    mem = [Member(z_face=G.tanh_stretched_faces(nl, 30000.0, 200.0), alpha_w=1.0e-3, D0=2.0, f3=1.0e-4)
           for nl in nlevs]
    rng = np.random.default_rng(len(nlevs))
    Y = []
    for i, nl in enumerate(nlevs):
        g = G.columns(1, G.tanh_stretched_faces(nl, 30000.0, 200.0), 1.0e-4)
        Y.append(I.column_state(g, PAR, seed=i, T_s=np.array([290.0 + i % 15])).ravel())
    Y0 = np.concatenate(Y).astype(np.float32)
    # first-order upwinding: its derivative depends on the state through the sign
    # of u_3 only, so a rounding difference is not amplified by a limiter branch
    num = P.Numerics(hyperdiff=False, rayleigh=True, vert_diff=True, upwinding=1, dt=10.0)
    e = ColumnEnsemble(mem, PAR, num)
    w = torch.from_numpy((rng.standard_normal(Y0.size) / np.maximum(np.abs(Y0), 1.0)).astype(np.float32)).cuda()
    y = torch.from_numpy(Y0).cuda()
    a = [t.cpu().numpy().astype(np.float64) for t in e.adjoint(y, w, 10.0, nsteps, every)]
    a2 = [t.cpu().numpy().astype(np.float64) for t in e.adjoint(y, w, 10.0, nsteps, every)]
    b = [t.cpu().numpy().astype(np.float64) for t in e.adjoint(y, w, 10.0, nsteps, every, noalloc=True)]
    e.close()
    # float32 storage of the states and cotangents: 2^-24 per operation, some
    # hundreds of them in a row per step, and the stage's stiffness about 10
    tol = nsteps * 1000 * 2.0 ** -24
    for name, u, u2, v in zip(("Y0", "D0", "alpha_w"), a, a2, b):
        assert np.all(np.isfinite(u)) and np.array_equal(u, u2), name
        assert np.linalg.norm(u - v) <= tol * np.linalg.norm(v), (name, np.linalg.norm(u - v), np.linalg.norm(v))
