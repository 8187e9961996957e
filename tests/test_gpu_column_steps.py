"""Whole steps of a column grid in one launch (a wavefront per column, one or two
levels per lane): against the float64 oracle at the edges of the level ranges,
bitwise independent of how the steps are split over calls, and with every
column independent of the others."""
import numpy as np
import pytest

from cadycore import geometry as G
from cadycore import initial as I
from cadycore import params as P
from test_gpu_parity import PAR, _storage_floor, _torch, field_errors

pytestmark = pytest.mark.gpu


def _case(ncol, nlev):
    g = G.columns(ncol, G.tanh_stretched_faces(nlev, 30000.0, 200.0), 1.0e-4)
    num = P.Numerics(hyperdiff=False, rayleigh=True, dt=10.0)
    Ts = 290.0 + np.arange(ncol) % 15
    return g, num, I.column_state(g, PAR, seed=2, T_s=Ts).astype(np.float32).astype(np.float64)


@pytest.mark.parametrize("ncol,nlev", [(1, 3), (2, 31), (5, 63), (3, 64), (2, 65), (7, 127), (1, 128)])
def test_one_step_matches_oracle(ncol, nlev):
    torch = _torch()
    from cadycore.lib import DryDycore
    from oracle import Oracle

    g, num, Y32 = _case(ncol, nlev)
    d = DryDycore(g, PAR, num)
    Y = d.state(Y32)
    d.step(Y, num.dt, 1)
    torch.cuda.synchronize()
    got = Y.cpu().numpy().astype(np.float64)
    d.close()
    ref = Y32.copy()
    o = Oracle(g, PAR, num)
    o.set_precomputed(ref)
    o.step(ref, num.dt, 1)
    e = field_errors(got, ref, g)
    fl = _storage_floor(g, num, Y32, num.dt, 1, ref)["u3"]
    print(ncol, nlev, e, "u3 storage floor", fl)
    for name in ("rho", "u1", "u2", "rhoe"):
        assert e[name] <= 1e-5, (name, e[name])
    assert e["u3"] <= 3.0 * fl
    u3 = I.unpack(got, ncol, nlev)[4]
    assert np.all(u3[0] == 0) and np.all(u3[-1] == 0)


@pytest.mark.parametrize("ncol,nlev", [(6, 30), (3, 64), (5, 100)])
def test_steps_do_not_depend_on_the_calls_or_the_other_columns(ncol, nlev):
    torch = _torch()
    from cadycore.lib import DryDycore

    g, num, Y32 = _case(ncol, nlev)
    d = DryDycore(g, PAR, num)
    a, b, c = d.state(Y32), d.state(Y32), d.state(Y32)
    d.step(a, num.dt, 4)
    for _ in range(4):
        d.step(b, num.dt, 1)
    c.reshape(-1, ncol)[:, 1] = float("nan")  # one column not a number at every level
    d.step(c, num.dt, 4)
    torch.cuda.synchronize()
    d.close()
    assert torch.equal(a, b)
    keep = [i for i in range(ncol) if i != 1]
    assert torch.equal(a.reshape(-1, ncol)[:, keep], c.reshape(-1, ncol)[:, keep])
    assert not torch.isfinite(c.reshape(-1, ncol)[:4 * nlev, 1]).any()  # the centre fields
