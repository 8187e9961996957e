"""The step's rounding errors against those of the recorded step, whose implicit
stage forms every face flux once and hands it to both centres.  The step's own
stage forms a flux in each of the two centres; rounded differently there, the
fluxes no longer cancel between neighbours and the winds' error grows by 1.5%.

The error of a field is the rms of N = 387,072 rounding errors, correlated over
some tens of neighbours: it is known to 1 / sqrt(2 N / 40) = 0.7%, and the two
steps share most of their rounding; over two states and two wind components the
mean ratio may be off by 0.5%."""
import numpy as np
import pytest

from cadycore import geometry as G
from cadycore import initial as I
from cadycore import params as P
from test_gpu_parity import PAR, _torch

pytestmark = pytest.mark.gpu


def test_step_is_as_accurate_as_the_recorded_step():
    torch = _torch()
    from cadycore.lib import DryDycore
    from oracle import Oracle

    nlev, dt, nsteps = 63, 100.0, 4
    g = G.cubed_sphere(8, G.tanh_stretched_faces(nlev, 30000.0, 30.0), PAR.planet_radius, PAR.Omega)
    num = P.Numerics(dt=dt)
    d, o = DryDycore(g, PAR, num), Oracle(g, PAR, num)
    ratios = []
    for seed in (1, 2):
        Y32 = I.sphere_state(g, PAR, seed=seed).astype(np.float32).astype(np.float64)
        a, b, ref = d.state(Y32), d.state(Y32), Y32.copy()
        d.step(a, dt, nsteps)
        d.step_record(b, dt, nsteps, 8)
        o.dss(ref)
        o.step(ref, dt, nsteps)
        err = []
        for y in (a, b):
            f = I.unpack(y.cpu().numpy().astype(np.float64), g.ncol, nlev)
            err.append([np.linalg.norm(x - r) / np.linalg.norm(r) for x, r in zip(f, I.unpack(ref, g.ncol, nlev))])
        print(seed, err)
        ratios += [err[0][i] / err[1][i] for i in (1, 2)]
    d.close()
    assert np.mean(ratios) <= 1.005, ratios
