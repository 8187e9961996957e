"""The column hooks (implicit tendency, Jacobian and solve, upwind correction)
at the edges of their level chunks and lane shapes, on a sphere and on aligned
and ragged column counts, against the float64 oracle with the hooks' gate (1e-5
per field); and the solve in place (dY and R the same buffer).

The upwind correction is built from the layer differences of a float32 enthalpy
(half a unit in the last place of |h|, 2^-25 |h|, at each of the two centres of
a difference, and the limiter takes up to four differences per cell): its gate
is 1e-5 plus 8 x 2^-25 max|h| / rms(dh)."""
import numpy as np
import pytest

from cadycore import geometry as G
from cadycore import initial as I
from cadycore import params as P
from test_gpu_parity import PAR, _torch, field_errors

pytestmark = pytest.mark.gpu


def _grid(kind, size, nlev):
    zf = G.tanh_stretched_faces(nlev, 30000.0, 200.0)
    if kind == "sphere":
        return G.cubed_sphere(size, zf, PAR.planet_radius, PAR.Omega)
    return G.columns(size, zf, 1.0e-4)


@pytest.mark.parametrize("kind,size,nlev", [("sphere", 2, 3), ("sphere", 2, 32), ("sphere", 2, 33), ("sphere", 2, 64),
                                            ("sphere", 2, 65), ("sphere", 2, 128), ("sphere", 2, 129),
                                            ("columns", 1, 5), ("columns", 17, 64), ("columns", 8, 100),
                                            ("columns", 3, 128)])
def test_column_hooks_match_oracle(kind, size, nlev):
    torch = _torch()
    from cadycore.lib import DryDycore
    from oracle import Oracle

    g = _grid(kind, size, nlev)
    num = P.Numerics(hyperdiff=False, rayleigh=True, dt=20.0)
    make = I.sphere_state if kind == "sphere" else I.column_state
    f = I.unpack(make(g, PAR, seed=4), g.ncol, nlev)
    rng = np.random.default_rng(7)
    jvf = g.vertical()[2][:, None]
    u3 = 0.3 * jvf * rng.standard_normal((nlev + 1, g.n_nodes))[:, g.node_id]  # w of 0.3 m/s
    u3[0] = u3[-1] = 0.0
    Y = I.pack(*f[:4], u3).astype(np.float32).astype(np.float64)
    d, o = DryDycore(g, PAR, num), Oracle(g, PAR, num)
    Yo = Y.copy()
    o.set_precomputed(Yo)
    Yg = d.state(Y)
    dtg = 0.4358665215 * num.dt
    T, C = d.zeros(), d.zeros()
    d.implicit_tendency(T, Yg)
    d.correct_implicit_advection_tendency(C, Yg)
    d.update_jacobian(Yg, dtg)
    o.update_jacobian(Yo, dtg)
    # a residual with every component and the boundary faces in it
    scale = [np.abs(x).max() * 1e-3 for x in I.unpack(Y, g.ncol, nlev)]
    R = I.pack(*(s * rng.standard_normal(x.shape) for s, x in zip(scale, I.unpack(Y, g.ncol, nlev))))
    R = R.astype(np.float32).astype(np.float64)
    dY, inplace = d.zeros(), d.state(R)
    d.ldiv(dY, d.state(R))
    d.ldiv(inplace, inplace)
    torch.cuda.synchronize()
    res = {
        "T_imp": (T, o.implicit_tendency(Yo)),
        "T_post_imp": (C, o.correct_implicit(Yo)),
        "ldiv": (dY, o.ldiv(R)),
    }
    fY = I.unpack(Y, g.ncol, nlev)
    e, zc = fY[3] / fY[0], g.zc[:, None]
    T_c = PAR.T_0 + (e - PAR.grav * zc + PAR.R_d * PAR.T_0) / PAR.cv_d  # up to the kinetic energy
    h = e + PAR.R_d * T_c
    gate = dict.fromkeys(("T_imp", "ldiv"), 1e-5)
    gate["T_post_imp"] = 1e-5 + 8.0 * 2.0 ** -25 * np.abs(h).max() / np.sqrt(np.mean(np.diff(h, axis=0) ** 2))
    res = {k: field_errors(a.cpu().numpy().astype(np.float64), b, g) for k, (a, b) in res.items()}
    same = torch.equal(dY, inplace)
    d.close()
    print(kind, size, nlev, res, gate)
    for hook, errs in res.items():
        for name, err in errs.items():
            assert err <= gate[hook], (hook, name, err)
    assert same
