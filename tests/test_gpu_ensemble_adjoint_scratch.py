"""The ensemble's reverse mode gives the same bits however its scratch is cut:
any checkpoint spacing, the handle's scratch or the library's fixed array, all
members at once or some at a time, stage records of a segment or of one step.
With van Leer's limiter, whose branches turn a last bit into a visible change of
the gradient.  And `every` bounds what it allocates."""
import numpy as np
import pytest

from cadycore import geometry as G
from cadycore import initial as I
from cadycore import params as P
from test_gpu_parity import PAR, _torch

pytestmark = pytest.mark.gpu


def _make(nlevs):
    from cadycore.ensemble import ColumnEnsemble, Member

    faces = {nl: G.tanh_stretched_faces(nl, 30000.0, 200.0) for nl in set(nlevs)}
    cols = {nl: [I.column_state(G.columns(1, zf, 1.0e-4), PAR, seed=i, T_s=np.array([290.0 + 3 * i])).ravel()
                 for i in range(4)] for nl, zf in faces.items()}
    mem = [Member(z_face=faces[nl], alpha_w=1.0e-3 * (1 + i % 3), D0=2.0, f3=1.0e-4) for i, nl in enumerate(nlevs)]
    e = ColumnEnsemble(mem, PAR, P.Numerics(hyperdiff=False, rayleigh=True, vert_diff=True, upwinding=3, dt=10.0))
    Y0 = e.state([cols[nl][i % 4] for i, nl in enumerate(nlevs)])
    rng = np.random.default_rng(len(nlevs))
    w = e.torch.from_numpy(rng.standard_normal(e.S).astype(np.float32)).to(Y0) / (Y0.abs() + 1.0)
    return e, Y0, w


@pytest.mark.parametrize("nlevs,nsteps", [([3], 1), ([32, 5, 17], 5), ([33, 64, 8], 7), ([128, 65, 30, 3], 9),
                                          ([30] * 300, 2), ([33, 64, 8], 40)], ids=lambda v: str(v)[:16])
def test_gradient_does_not_depend_on_the_scratch(nlevs, nsteps):
    torch = _torch()
    e, Y0, w = _make(nlevs)
    ref = e.adjoint(Y0, w, 10.0, nsteps, nsteps)
    assert all(torch.isfinite(x).all() for x in ref)
    for every in (1, 2, 4, nsteps + 5):  # 40 steps with 2 or 4 run their segments again
        for noalloc in (False, True):
            got = e.adjoint(Y0, w, 10.0, nsteps, every, noalloc=noalloc)
            for name, a, b in zip(("Y0", "D0", "alpha_w"), ref, got):
                assert torch.equal(a, b), (name, every, noalloc)
    e.close()


@pytest.mark.parametrize("nsteps,every", [(1, 1), (2, 2), (2, 1)])
def test_fixed_array_takes_the_members_in_parts(nsteps, every):
    """4000 members of 128 levels: 3 or 4 states fit the array of 2^24 floats, the 7
    to 8 that also hold one step's stage records do not."""
    torch = _torch()
    e, Y0, w = _make([128] * 4000)
    assert 4 * e.S <= 1 << 24 < 7 * e.S
    ref = e.adjoint(Y0, w, 10.0, nsteps, every)
    got = e.adjoint(Y0, w, 10.0, nsteps, every, noalloc=True)
    for name, a, b in zip(("Y0", "D0", "alpha_w"), ref, got):
        assert torch.isfinite(a).all() and torch.equal(a, b), name
    e.close()


def test_every_bounds_the_memory():
    """512 steps with a checkpoint every 16: 31 checkpoints and the 7 states of 16
    steps are 143 states, 7 states of every step would be 3584."""
    torch = _torch()
    e, Y0, w = _make([128] * 64)
    e.adjoint(Y0, w, 10.0, 1, 1)  # the kernels are loaded
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    e.adjoint(Y0, w, 10.0, 512, 16)
    torch.cuda.synchronize()
    taken = free - torch.cuda.mem_get_info()[0]
    assert taken <= 2 * 143 * 4 * e.S, taken  # twice: the allocators' granularity
    e.close()
