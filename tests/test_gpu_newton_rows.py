"""The implicit stage with a column in a wavefront's registers: one or two
levels per lane, one or two columns per wavefront, 16- and 32-column tiles.
Each shape is stepped once at the edges of its range of levels against the
float64 oracle, with the gates of test_gpu_parity: rho, u_h and rho e_tot within
1e-5, u_3 within three times the float32 storage floor, or, where a column is
deep, within the error of the oracle built in float32 throughout."""
import numpy as np
import pytest

from cadycore import geometry as G
from cadycore import initial as I
from cadycore import params as P
from test_gpu_parity import PAR, _float32_throughout, _storage_floor, _torch, field_errors

pytestmark = pytest.mark.gpu


def _step_vs_oracle(g, num, Y32, tuning=None, T_sfc_col=None):
    torch = _torch()
    from cadycore.lib import DryDycore
    from oracle import Oracle

    d = DryDycore(g, PAR, num, T_sfc_col=T_sfc_col)
    for knob, value in (tuning or {}).items():
        d.set_tuning(knob, value)
    Yg = d.state(Y32)
    d.step(Yg, num.dt, 1)
    torch.cuda.synchronize()
    got = Yg.cpu().numpy().astype(np.float64)
    d.close()
    o = Oracle(g, PAR, num, T_sfc_col=T_sfc_col)
    ref = Y32.copy()
    o.dss(ref)
    o.set_precomputed(ref)
    o.step(ref, num.dt, 1)
    return field_errors(got, ref, g), ref


@pytest.mark.parametrize("nlev", [3, 31, 32, 33, 63, 64, 65, 94, 95, 96, 97, 127, 128, 129])
def test_sphere_step_at_the_edges_of_the_level_ranges(nlev):
    g = G.cubed_sphere(2, G.tanh_stretched_faces(nlev, 30000.0, 200.0), PAR.planet_radius, PAR.Omega)
    num = P.Numerics(dt=100.0)
    Y32 = I.sphere_state(g, PAR, seed=3).astype(np.float32).astype(np.float64)
    e, ref = _step_vs_oracle(g, num, Y32)
    guard = max(3.0 * _storage_floor(g, num, Y32, num.dt, 1, ref)["u3"],
                _float32_throughout(g, num, Y32, num.dt, 1, ref))
    print("nlev", nlev, e, "u3 guard", guard)
    for name in ("rho", "u1", "u2", "rhoe"):
        assert e[name] <= 1e-5, (name, e[name])
    assert e["u3"] <= guard


@pytest.mark.parametrize("ncol,nlev", [(1, 30), (5, 45), (16, 64), (17, 63), (8, 100), (19, 128), (3, 129)])
def test_columns_step_with_surface_fluxes(ncol, nlev):
    """Independent columns, aligned and ragged column counts (surface fluxes
    keep the step on the kernels that the sphere uses)."""
    g = G.columns(ncol, G.tanh_stretched_faces(nlev, 30000.0, 200.0), 1.0e-4)
    num = P.Numerics(hyperdiff=False, rayleigh=True, sfc_flux=True, dt=10.0)
    Y32 = I.column_state(g, PAR, seed=1).astype(np.float32).astype(np.float64)
    Ts = I.surface_temperature(g)
    e, ref = _step_vs_oracle(g, num, Y32, T_sfc_col=Ts)
    print("ncol", ncol, "nlev", nlev, e)
    for name in ("rho", "u1", "u2", "rhoe"):
        assert e[name] <= 1e-5, (name, e[name])
    assert e["u3"] <= 1e-3


def test_large_grid_shape_matches_the_32_column_tiles():
    """nlev > 56 on at least 65,536 columns takes one level per lane in
    16-column tiles; the 32-column tiles run the same column algebra."""
    torch = _torch()
    from cadycore.lib import CA_TUNE_NEWTON, DryDycore

    g = G.cubed_sphere(27, G.tanh_stretched_faces(57, 30000.0, 30.0), PAR.planet_radius, PAR.Omega)
    Y32 = I.sphere_state(g, PAR, seed=3)
    d = DryDycore(g, PAR, P.Numerics(dt=60.0))
    out = []
    for v in (1, 2):
        d.set_tuning(CA_TUNE_NEWTON, v)
        Y = d.state(Y32)
        d.step(Y, 60.0, 1)
        torch.cuda.synchronize()
        out.append(Y.cpu().numpy().astype(np.float64))
    d.close()
    for name, err in field_errors(out[0], out[1], g).items():
        assert err <= (1e-6 if name != "u3" else 1e-4), (name, err)  # rounding order at most
