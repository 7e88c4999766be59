"""Receiver sampling and adjoint-source tables of the 2D acoustic solver on
the GPU against the oracle: sums of one to many taps, spread over blocks."""
import numpy as np
import pytest

from helpers import rel_l2
from owl_amd import Acoustic2DBatch, Geometry, Receiver, Source
from owl_amd.synthetic import gardner, random_field

pytestmark = pytest.mark.gpu


def _model(nz, nx):
    vp = (2000.0 + 10.0 * np.arange(nz)[:, None]) * (1.0 + 0.05 * random_field((nz, nx), 4.0, 1))
    vp = vp.astype(np.float32)
    return vp, gardner(vp)


def _line(first, n, z, step=10.0):
    return [Receiver(x=first + step * k, z=z) for k in range(n)]


@pytest.mark.parametrize("case", ["one off the nodes", "17 off the nodes", "300 on the nodes", "2100 at one place",
                                  "unequal counts", "zero weights"])
def test_sampling_and_adjoint_source_tables(oracle32, gpu, case):
    """Receiver sums split over blocks (1, 9 or 81 taps a receiver, counts at
    and past a block's sums), and tables shared between shots of one spread:
    traces bit-identical to the oracle, OWL's gradient as the oracle's."""
    print(f"case: receiver tables, {case}", flush=True)
    nx, nz, dx, dt, tmax, pml = 61, 47, 10.0, 0.001, 0.12, 10
    vp, rho = _model(nz, nx)
    per_shot = {"one off the nodes": [[Receiver(x=203.0, z=27.0)]] * 2,
                "17 off the nodes": [_line(102.5, 17, 22.5)] * 2,
                "300 on the nodes": [_line(100.0, 300, 20.0, step=0.0)] * 2,
                "2100 at one place": [_line(101.25, 2100, 21.0, step=0.0)] * 2,
                "unequal counts": [_line(52.5, 40, 22.5), _line(102.5, 3, 20.0), _line(52.5, 40, 22.5)],
                "zero weights": [[Receiver(x=r.x, z=r.z, weight=float(k % 3 > 0)) for k, r in
                                  enumerate(_line(92.5, 20, 22.5))]] * 2}[case]
    geoms = [Geometry(id=k + 1, srcr=[Source(x=200.0 + 95.0 * k, z=60.0, f0=25.0)], recr=recs)
             for k, recs in enumerate(per_shot)]
    b = Acoustic2DBatch(nx, nz, dx, dx, vp, rho, [(g, None) for g in geoms], dt, tmax, pml=pml)
    got = b.forward(save_boundary=True)
    adj = [(0.5 * t).astype(np.float32) for t in got]
    grads = b.adjoint(adj)
    g = dict(nx=nx, nz=nz, dx=dx, dz=dx, dt=dt, nt=b.nt, pml=pml, R=4)
    for geom, tr, (gv, gr), a in zip(geoms, got, grads, adj):
        src = [dict(x=s.x, z=s.z, f0=s.f0) for s in geom.srcr]
        rec = [dict(x=r.x, z=r.z, weight=r.weight) for r in geom.recr]
        assert np.array_equal(tr, oracle32.acoustic2d_forward(g, vp, rho, src, rec))
        rv, rr, _ = oracle32.acoustic2d_gradient_owl(g, vp, rho, src, rec, a)
        assert rel_l2(gv, rv) < 1e-4 and rel_l2(gr, rr) < 1e-4
    b.close()
