"""The launch-dependent forms of the 2D acoustic steps on the GPU: one fused
launch per step against the two sweeps in OWL's forward and gradient, and the
sweeps' rows per thread."""
import numpy as np
import pytest

from helpers import rel_l2, simple_geometry
from owl_amd import OWL_CKPT_BINOMIAL, OWL_GRAD_EXACT, OWL_STORE_F32, Acoustic2DBatch, Window
from owl_amd.synthetic import gardner, random_field

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,tmax", [(2, 0.1), (4, 0.1), (4, 0.101), (8, 0.1)])
def test_owl_gradient_fused_steps_match_the_sweeps(gpu, R, tmax):
    """OWL's forward and reverse passes by the fused step (five ragged
    windows, steps of both parities): bit-identical to the sweeps."""
    print(f"case: OWL gradient fused, R={R} tmax={tmax}", flush=True)
    nz, nx, dx = 61, 150, 10.0
    vp = (2000.0 * (1 + 0.05 * random_field((nz, nx), 4.0, 3))).astype(np.float32)
    rho = gardner(vp)
    wins = [None, Window(1, 75, 1, 58, 0.0, 0.0), Window(50, 131, 5, 60, 490.0, 40.0),
            Window(30, 62, 1, 33, 290.0, 0.0), Window(3, 96, 2, 58, 20.0, 10.0)]
    geoms = []
    for k, w in enumerate(wins):
        x0, z0, n = (0.0, 0.0, nx) if w is None else ((w.nxbeg - 1) * dx, (w.nzbeg - 1) * dx, w.nx)
        rx = x0 + 5.0 + 10.0 * np.arange(n - 1)
        geoms.append(simple_geometry(k + 1, x0 + 5.0 * (n - 1) + 3.3, z0 + 80.0, rx, np.full(n - 1, z0 + 30.0),
                                     f0=20.0))
    b = Acoustic2DBatch(nx, nz, dx, dx, vp, rho, list(zip(geoms, wins)), 0.001, tmax, pml=max(10, R), fdhalf=R)
    out = []
    for mode in ("sweeps", "fused", "sweeps"):
        b.set_step_kernel(mode)
        b.set_profiling(True)
        plain = b.forward()
        tr = b.forward(save_boundary=True)
        grads = b.adjoint([(0.5 * t).astype(np.float32) for t in tr])
        assert (b.kernel_stats()["step_fused"]["launches"] > 0) == (mode == "fused")
        b.set_profiling(False)
        out.append(list(plain) + list(tr) + [g for pair in grads for g in pair])
    assert all(np.abs(a).max() > 0 for a in out[0])
    for other in out[1:]:
        for x, y in zip(out[0], other):
            assert np.array_equal(x, y)
    b.close()


@pytest.mark.parametrize("nx,nz,shots", [(61, 47, 1), (391, 403, 5), (391, 403, 11)])
def test_rows_per_thread_match_the_oracle(oracle32, gpu, nx, nz, shots):
    """The sweeps' one, two and four rows per thread (by the number of
    wavefronts that one row per thread would take), ragged against the tiles,
    the receivers sampled after the source's steps and beside the v-sweep
    once they are over: traces bit-identical to the oracle."""
    print(f"case: sweeps on {nx} x {nz}, {shots} shots", flush=True)
    dx = 10.0
    vp = (2000.0 + 0.1 * np.arange(nz)[:, None] + 0.1 * np.arange(nx)[None, :]).astype(np.float32)
    rho = gardner(vp)
    rx = 5.0 + 10.0 * np.arange(55)
    geoms = [simple_geometry(k + 1, 200.0 + 95.0 * k, 60.0, rx, np.full(55, 22.5), f0=70.0) for k in range(shots)]
    b = Acoustic2DBatch(nx, nz, dx, dx, vp, rho, [(g, None) for g in geoms], 0.001, 0.06, pml=10)
    b.set_step_kernel("sweeps")
    got = b.forward()
    g = dict(nx=nx, nz=nz, dx=dx, dz=dx, dt=0.001, nt=b.nt, pml=10, R=4)
    for geom, tr in list(zip(geoms, got))[::5]:
        src = [dict(x=s.x, z=s.z, f0=s.f0) for s in geom.srcr]
        rec = [dict(x=r.x, z=r.z, weight=r.weight) for r in geom.recr]
        assert np.array_equal(tr, oracle32.acoustic2d_forward(g, vp, rho, src, rec))
    b.close()


@pytest.mark.parametrize("nx,nz,shots,R,fused", [(120, 100, 4, 4, False), (380, 364, 4, 4, True),
                                                 (380, 364, 3, 4, False), (380, 364, 4, 6, False)])
def test_default_step_kernel_follows_the_batch(gpu, nx, nz, shots, R, fused):
    """The default takes the fused step from 4 shots and, by the stencil, 0.6
    or 1.2 million nodes on; the exact gradient as by the other kernel."""
    print(f"case: default step kernel, {shots} x {nx} x {nz}, R={R}", flush=True)
    vp = (2000.0 * (1 + 0.05 * random_field((nz, nx), 4.0, 5))).astype(np.float32)
    rho = gardner(vp)
    rx = 15.0 + 10.0 * np.arange(60)
    geoms = [simple_geometry(k + 1, 100.0 + 90.0 * k, 60.0, rx, np.full(60, 30.0), f0=25.0) for k in range(shots)]
    b = Acoustic2DBatch(nx, nz, 10.0, 10.0, vp, rho, [(g, None) for g in geoms], 0.001, 0.06, pml=12, fdhalf=R)
    obs = [np.float32(0.5) * t for t in b.forward()]
    kw = dict(mode=OWL_GRAD_EXACT, ckpt=OWL_CKPT_BINOMIAL, ckpt_param=6, store=OWL_STORE_F32)
    b.set_profiling(True)
    m0, gv0, gr0, s0 = b.gradient(obs, **kw)
    st = b.kernel_stats()
    assert (st["step_fused"]["launches"] > 0) == fused == (st["adjoint_fused"]["launches"] > 0)
    b.set_step_kernel("sweeps" if fused else "fused")
    m1, gv1, gr1, s1 = b.gradient(obs, **kw)
    assert np.array_equal(m0, m1) and np.array_equal(gv0, gv1) and np.abs(gv0).max() > 0
    assert all(np.array_equal(x, y) for x, y in zip(s0, s1))
    assert rel_l2(gr1, gr0) <= 1e-12
    b.close()
