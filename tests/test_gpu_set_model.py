"""A new model for an acoustic 2D batch (owl_acoustic2d_set_model): refilled
on the device for explosion sources, planned again for forces."""
import numpy as np
import pytest

from owl_amd import OWL_GRAD_OWL, Acoustic2DBatch, Geometry, Receiver, Source, Window
from owl_amd._lib import OwlError
from owl_amd.synthetic import gardner, random_field

pytestmark = pytest.mark.gpu

NX, NZ, DX, DT, TMAX = 67, 45, 10.0, 0.001, 0.12


def _model(seed, v0):
    vp = (v0 + 8.0 * np.arange(NZ)[:, None]) * (1.0 + 0.05 * random_field((NZ, NX), 4.0, seed))
    vp = vp.astype(np.float32)
    return vp, gardner(vp)


def _batch(vp, rho, mechanism, ragged):
    shots = []
    for k in range(3):
        w = Window(1 + 9 * k, 40 + 13 * k, 1, NZ, 90.0 * k, 0.0) if ragged else None
        shots.append((Geometry(id=k + 1, srcr=[Source(x=230.0 + 60.0 * k, z=60.0, f0=25.0, mechanism=mechanism,
                                                      polar=0.3)],
                               recr=[Receiver(x=212.5 + 10.0 * i, z=32.5) for i in range(15)]), w))
    return Acoustic2DBatch(NX, NZ, DX, DX, vp, rho, shots, DT, TMAX, pml=11, fdhalf=5)


@pytest.mark.parametrize("mechanism", ["explosion", "force"])
@pytest.mark.parametrize("ragged", [False, True])
def test_new_model_equals_a_new_batch(gpu, mechanism, ragged):
    print(f"case: set_model, {mechanism}, ragged={ragged}", flush=True)
    b = _batch(*_model(1, 2000.0), mechanism, ragged)
    b.observe()
    b.set_model(*_model(2, 2300.0))   # other edge velocities: other PML profiles
    fresh = _batch(*_model(2, 2300.0), mechanism, ragged)
    for a, c in zip(b.forward(), fresh.forward()):
        assert np.array_equal(a, c)
    obs = [0.8 * t for t in fresh.forward()]
    for a, c in zip(b.gradient(obs, mode=OWL_GRAD_OWL)[:3], fresh.gradient(obs, mode=OWL_GRAD_OWL)[:3]):
        assert np.array_equal(a, c)
    b.close()
    fresh.close()


@pytest.mark.parametrize("bad", ["too fast", "negative", "nan"])
def test_refused_model_leaves_the_one_before(gpu, bad):
    print(f"case: refused model, {bad}", flush=True)
    vp, rho = _model(1, 2000.0)
    b = _batch(vp, rho, "explosion", True)
    ref = b.forward()
    v = vp.copy()
    v[20, 30] = {"too fast": 9000.0, "negative": -1.0, "nan": np.nan}[bad]
    with pytest.raises(OwlError):
        b.set_model(v, rho)
    for a, c in zip(b.forward(), ref):
        assert np.array_equal(a, c)
    b.close()
