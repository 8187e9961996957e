"""The FieldVector hooks at the edges of the transposing move's tiles (32 levels by 64
columns): one and two level tiles, a tile that holds the top face alone, ragged
column tiles; level-fastest and column-fastest arrays with padding in every
stride.  Bitwise the native hooks, and nothing between the values is touched."""
import numpy as np
import pytest

from cadycore import geometry as G
from cadycore import initial as I
from cadycore import params as P
from test_gpu_parity import PAR, _torch

pytestmark = pytest.mark.gpu

FILL = -12345.0


class _Strided:
    """A padded FieldVector over two flat arrays, and where its values lie."""

    def __init__(self, d, kind):
        from cadycore.lib import CaFieldVector

        g, t = d.grid, d.torch
        self.t = t
        nh, col = -(-g.ncol // 16), np.arange(g.ncol)
        h, j, i = col >> 4, (col >> 2) & 3, col & 3
        self.fv, idx, parts = CaFieldVector(), [], []
        for arr, ncomp, nv in (("c", 4, g.nlev), ("f", 1, g.nlev + 1)):
            if kind == "levels":
                sv, si = 1, nv + 3
                sj = 4 * si + 1
                sc = 4 * sj + 2
                sh = ncomp * sc + 5
                size = 7 + nh * sh
            else:
                si, sj, sh = 1, 5, 23
                sv = nh * sh + 11
                sc = nv * sv + 13
                size = 7 + ncomp * sc
            a = t.full((size,), FILL, device=d.device, dtype=t.float32)
            setattr(self, arr, a)
            setattr(self.fv, arr, a.data_ptr())
            at = []
            for p in range(ncomp):
                lay = self.fv.lay[p if arr == "c" else 4]
                lay.offset, lay.s_v, lay.s_i, lay.s_j, lay.s_h = 7 + p * sc, sv, si, sj, sh
                at.append((lay.offset + np.arange(nv)[:, None] * sv + (i * si + j * sj + h * sh)[None]).reshape(-1))
            idx.append(t.from_numpy(np.concatenate(at)).to(d.device))
        self.idx = idx

    def put(self, Y):
        n = self.idx[0].numel()
        self.c[self.idx[0]] = Y[:n]
        self.f[self.idx[1]] = Y[n:]
        return self

    def get(self):
        return self.t.cat([self.c[self.idx[0]], self.f[self.idx[1]]])

    def padding_kept(self):
        c, f = self.c.clone(), self.f.clone()
        c[self.idx[0]] = FILL
        f[self.idx[1]] = FILL
        return bool((c == FILL).all() and (f == FILL).all())


@pytest.mark.parametrize("kind", ["levels", "columns"])
@pytest.mark.parametrize("size,nlev", [(2, 31), (2, 32), (3, 33), (3, 63), (2, 64), (3, 65), (3, 3)])
def test_sphere_hooks_on_padded_arrays(size, nlev, kind):
    torch = _torch()
    from cadycore.lib import DryDycore

    g = G.cubed_sphere(size, G.tanh_stretched_faces(nlev, 30000.0, 200.0), PAR.planet_radius, PAR.Omega)
    d = DryDycore(g, PAR, P.Numerics(dt=20.0))
    f = I.unpack(I.sphere_state(g, PAR, seed=4), g.ncol, nlev)
    u3 = np.random.default_rng(1).normal(0.0, 5.0, (nlev + 1, g.ncol))  # off the boundary filter too
    Y = d.state(I.pack(*f[:4], u3).astype(np.float32).astype(np.float64))
    _hooks(d, torch, Y, kind, sphere=True)
    d.close()


@pytest.mark.parametrize("kind", ["levels", "columns"])
@pytest.mark.parametrize("ncol,nlev", [(1, 31), (70, 32), (129, 64)])
def test_column_hooks_on_padded_arrays(ncol, nlev, kind):
    torch = _torch()
    from cadycore.lib import DryDycore

    g = G.columns(ncol, G.tanh_stretched_faces(nlev, 30000.0, 200.0), 1.0e-4)
    d = DryDycore(g, PAR, P.Numerics(hyperdiff=False, rayleigh=True, dt=20.0))
    Y = d.state(I.column_state(g, PAR, seed=2, T_s=290.0 + np.arange(ncol) % 15).astype(np.float32).astype(np.float64))
    _hooks(d, torch, Y, kind, sphere=False)
    d.close()


def _hooks(d, torch, Y, kind, sphere):
    def same(x, ref, what):
        torch.cuda.synchronize()
        assert torch.isfinite(ref).all(), what
        assert torch.equal(x.get(), ref), what
        assert x.padding_kept(), what

    # in, and the filtered face component alone out
    ref, y = Y.clone(), _Strided(d, kind).put(Y)
    d.set_implicit_precomputed_quantities(ref)
    d.set_implicit_precomputed_quantities_fv(y.fv)
    same(y, ref, "cache_imp!")
    Y = ref
    # in, and all components out
    ref, y, T = d.zeros(), _Strided(d, kind).put(Y), _Strided(d, kind)
    d.implicit_tendency(ref, Y)
    d.implicit_tendency_fv(T.fv, y.fv)
    same(T, ref, "implicit_tendency!")
    same(y, Y, "its input")
    # and the limited tendency cleared
    ref, T, lim = d.zeros(), _Strided(d, kind), _Strided(d, kind)
    d.remaining_tendency(ref, Y)
    d.remaining_tendency_fv(T.fv, lim.fv, y.fv)
    same(T, ref, "remaining_tendency!")
    same(lim, torch.zeros_like(Y), "Yt_lim")
    if sphere:  # in place
        ref = Y.clone()
        d.dss(ref)
        d.dss_fv(y.fv)
        same(y, ref, "dss!")
