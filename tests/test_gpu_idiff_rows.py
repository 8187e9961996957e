"""The fused implicit-diffusion stage at the edges of its level ranges (one or two
levels per lane, one or two columns per wavefront), both closures, 1 and 3
iterations of its solve: one step against the float64 oracle with the gates of
test_gpu_implicit_diffusion (1e-5 per field; u_3, whose float32 storage floor is
1e-4, within 1e-3), and an unaligned state bitwise like an aligned one."""
import numpy as np
import pytest

from cadycore import geometry as G
from cadycore import initial as I
from cadycore import params as P
from test_gpu_parity import PAR, _torch, field_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,size,nlev,iters,model", [
    ("sphere", 2, 3, 1, "DecayWithHeightDiffusion"), ("sphere", 2, 32, 1, "DecayWithHeightDiffusion"),
    ("sphere", 2, 33, 3, "VerticalDiffusion"), ("sphere", 2, 64, 1, "DecayWithHeightDiffusion"),
    ("sphere", 2, 65, 3, "DecayWithHeightDiffusion"), ("sphere", 2, 128, 1, "VerticalDiffusion"),
    ("columns", 5, 30, 3, "DecayWithHeightDiffusion"), ("columns", 4, 64, 1, "VerticalDiffusion"),
    ("columns", 3, 100, 1, "DecayWithHeightDiffusion")])
def test_step_matches_oracle(kind, size, nlev, iters, model):
    torch = _torch()
    from cadycore.lib import DryDycore
    from oracle import Oracle

    zf = G.tanh_stretched_faces(nlev, 30000.0, 200.0)
    sphere = kind == "sphere"
    g = G.cubed_sphere(size, zf, PAR.planet_radius, PAR.Omega) if sphere else G.columns(size, zf, 1.0e-4)
    num = P.Numerics(hyperdiff=sphere, dt=100.0 if sphere else 10.0, vert_diff=True, implicit_diffusion=True,
                     solve_iters=iters, vert_diff_model=model, vert_diff_H=800.0)
    Y = I.sphere_state(g, PAR, seed=1) if sphere else I.column_state(g, PAR, seed=1, u=(10.0, 4.0))
    f = I.unpack(Y, g.ncol, nlev)
    shear = (1.0 + 0.5 * np.sin(np.pi * g.zc / zf[-1]))[:, None]  # of u_h, so that its diffusion is not a residual
    Y = I.pack(f[0], f[1] * shear, f[2] * shear, f[3], f[4]).astype(np.float32).astype(np.float64)
    rng = np.random.default_rng(7)
    D0 = np.exp(rng.uniform(np.log(1.0), np.log(50.0), g.n_nodes))[g.node_id]
    kw = dict(D0_col=D0) if model == "DecayWithHeightDiffusion" else {}
    d, o = DryDycore(g, PAR, num, **kw), Oracle(g, PAR, num, **kw)
    Yg = d.state(Y)
    buf = torch.empty(d.S + 1, device=Yg.device)
    off = buf[1:]
    off.copy_(Yg)
    d.step(Yg, num.dt, 1)
    d.step(off, num.dt, 1)
    torch.cuda.synchronize()
    same = torch.equal(Yg, off)
    got = Yg.cpu().numpy().astype(np.float64)
    d.close()
    ref = Y.copy()
    o.dss(ref)
    o.set_precomputed(ref)
    o.step(ref, num.dt, 1)
    e = field_errors(got, ref, g)
    print(kind, size, nlev, iters, model, e)
    for name in ("rho", "u1", "u2", "rhoe"):
        assert e[name] <= 1e-5, (name, e)
    assert e["u3"] <= 1e-3, e
    assert same
