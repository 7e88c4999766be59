"""The mapping of the 2D elastic and FSG free-surface gradients from the refined
rows to the windows on the GPU: ragged column counts, and windows so large that
the shots are mapped in more than one group."""
import numpy as np
import pytest

from helpers import rel_l2
from owl_amd import Elastic2DBatch, FSG2DBatch, Geometry, Receiver, Source
from owl_amd.fsg2d import GRADS
from test_gpu_elastic2d import _model, _oracle_args, _window_grid
from test_gpu_fsg2d import _oracle_args as _fsg_oracle_args, _sub
from test_oracle_pinning_fsg2d import _tti_model

pytestmark = pytest.mark.gpu

SURF = dict(refine=3.0, dz_max=14.0)


@pytest.mark.parametrize("nx,nz,tmax,wins", [
    (130, 33, 0.05, [None, dict(nxbeg=2, nxend=66, nzbeg=1, nzend=30), dict(nxbeg=60, nxend=123, nzbeg=2, nzend=31)]),
    (1400, 300, 0.07, [None, dict(nxbeg=2, nxend=1399, nzbeg=1, nzend=300), None]),
])
def test_surface_gradient_windows(oracle32, gpu, nx, nz, tmax, wins):
    """Per-shot windows within 1e-4 of the oracle (FP32 imaging there, FP64
    here), their sum the merged gradient to rounding of the windows' FP32."""
    pml, R, dx, dt = 12, 4, 10.0, 2.5e-4
    vp, vs, rho = _model(nz, nx, seed=4)
    geoms = []
    for k, w in enumerate(wins):
        x0 = dx * ((w or dict(nxbeg=1))["nxbeg"] - 1)
        z0 = dx * ((w or dict(nzbeg=1))["nzbeg"] - 1)
        geoms.append((Geometry(id=k + 1, srcr=[Source(x=x0 + 203.0, y=0.0, z=z0 + 25.0, f0=20.0, mechanism="force",
                                                      polar=0.3, amp=1e4)],
                               recr=[Receiver(x=x0 + 80.0 + 10.0 * m, y=0.0, z=z0 + 5.0) for m in range(30)]), w))
    print(f"case: surface columns {nx} x {nz}", flush=True)
    b = Elastic2DBatch(nx, nz, dx, dx, vp, vs, rho, geoms, dt, tmax, pml=pml, fdhalf=R, surface=SURF)
    syn = b.forward(save_boundary=True)
    obs = [tuple(np.float32(0.5) * c for c in s) for s in syn]
    adj = [tuple((s - o).astype(np.float32) for s, o in zip(sy, ob)) for sy, ob in zip(syn, obs)]
    grads = b.adjoint(adj)
    full = [np.zeros((nz, nx)) for _ in range(3)]
    for n, ((geom, win), gw, a) in enumerate(zip(geoms, grads, adj)):
        g, sl = _window_grid(vp, win, dx, dt, b.nt, pml, R)
        if nx < 1000 or n == len(geoms) - 1:
            srcs, recs = _oracle_args(geom, g, dx)
            *og, _ = oracle32.elastic2d_gradient_owl_fs(g, SURF, vp[sl], vs[sl], rho[sl], srcs, recs, np.stack(a))
            for k in range(3):
                assert gw[k].shape == og[k].shape and np.abs(og[k]).max() > 0
                assert rel_l2(gw[k], og[k]) < 1e-4, (geom.id, k, rel_l2(gw[k], og[k]))
        for k in range(3):
            full[k][sl] += gw[k]
    _, *merged, _ = b.gradient(obs)
    for m, f in zip(merged, full):
        assert np.allclose(m, f, rtol=0, atol=2.0 ** -22 * np.abs(f).max())
    b.close()


@pytest.mark.parametrize("nx,nz,wins", [
    (130, 33, [None, dict(nxbeg=2, nxend=66, nzbeg=1, nzend=30), dict(nxbeg=60, nxend=123, nzbeg=1, nzend=33)]),
    (1000, 300, [None, None]),
])
def test_fsg_surface_gradient_windows(oracle32, gpu, nx, nz, wins):
    """The same of the FSG solver under a tilted, curved surface, where every
    column has its own depths."""
    pml, R, dx, dt, tmax = 12, 4, 10.0, 2.5e-4, 0.06
    cij, rho = _tti_model(nz, nx, seed=3)
    xt = np.linspace(-400.0, dx * nx + 400.0, 41)
    surf = dict(topo=(xt, 12.0 * np.sin(xt / 170.0)), interp="cubic", refine=4.0, dz_max=15.0,
                src_from_surface=True, rec_from_surface=True)
    geoms = []
    for k, w in enumerate(wins):
        x0 = dx * ((w or dict(nxbeg=1))["nxbeg"] - 1)
        geoms.append((Geometry(id=k + 1, srcr=[Source(x=x0 + 203.0, y=0.0, z=25.0, f0=25.0, mechanism="force",
                                                      polar=0.3, amp=1e4)],
                               recr=[Receiver(x=x0 + 80.0 + 10.0 * m, y=0.0, z=5.0) for m in range(30)]), w))
    print(f"case: FSG surface columns {nx} x {nz}", flush=True)
    b = FSG2DBatch(nx, nz, dx, dx, cij, rho, geoms, dt, tmax, pml=pml, fdhalf=R, surface=surf)
    syn = b.forward(save_boundary=True)
    obs = [tuple(np.float32(0.5) * c for c in s) for s in syn]
    adj = [tuple((s - o).astype(np.float32) for s, o in zip(sy, ob)) for sy, ob in zip(syn, obs)]
    grads = b.adjoint(adj)
    full = {k: np.zeros((nz, nx)) for k in GRADS}
    for n, ((geom, win), gw, a) in enumerate(zip(geoms, grads, adj)):
        g, sl = _window_grid(rho, win, dx, dt, b.nt, pml, R)
        g["aniso"] = 1
        if nx < 1000 or n == len(geoms) - 1:
            srcs, recs = _fsg_oracle_args(geom, g, dx)
            og, _ = oracle32.fsg2d_gradient_owl_fs(g, surf, _sub(cij, sl), np.ascontiguousarray(rho[sl]), srcs, recs,
                                                   np.stack(a))
            for name in GRADS:
                assert gw[name].shape == og[name].shape and np.abs(og[name]).max() > 0
                assert rel_l2(gw[name], og[name]) < 1e-4, (geom.id, name, rel_l2(gw[name], og[name]))
        for name in GRADS:
            full[name][sl] += gw[name]
    _, merged, _ = b.gradient(obs)
    for name in GRADS:
        assert np.allclose(merged[name], full[name], rtol=0, atol=2.0 ** -22 * np.abs(full[name]).max())
    b.close()
