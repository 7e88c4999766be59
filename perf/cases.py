"""Workloads whose speed and results this framework is held to.

Each case is one call that a modelling or inversion program makes: a batch of
shots through one solver, forward or with its gradient.  `listed()` names the
reference set, `draw()` takes further cases of the same ranges, `prepare()`
builds what the program holds before the call (model, geometry, batch,
observed data), `run()` is the call, `work()` its compulsory traffic and
arithmetic, `tolerance()` the error another correct FP32 implementation may
show, and `exact()` the same outputs from FP64 tensors.

Lengths: a production run has thousands of time steps of the same two or
three kernels.  The cases keep the grids, shot counts and options of such
runs and shorten the time axis so that a pass stays below a second.
"""
import math

import numpy as np
import torch

from owl_amd import (OWL_CKPT_BINOMIAL, OWL_CKPT_FULL, OWL_CKPT_UNIFORM, OWL_GRAD_EXACT, OWL_GRAD_OWL, OWL_STORE_BF16,
                     OWL_STORE_F16, OWL_STORE_F32, Acoustic2DBatch, Acoustic3DBatch, Elastic2DBatch, Elastic3DBatch,
                     FSG2DBatch, Geometry, Receiver, Source, Window)
from owl_amd.autograd import propagate
from owl_amd.fsg2d import tti_cij

CKPT = {"full": OWL_CKPT_FULL, "uniform": OWL_CKPT_UNIFORM, "binomial": OWL_CKPT_BINOMIAL}
STORE = {"f32": OWL_STORE_F32, "f16": OWL_STORE_F16, "bf16": OWL_STORE_BF16}
VMAX = 4500.0


def _case(kind, n, nt, shots=1, pml=20, fdhalf=4, d=10.0, f0=20.0, ragged=False, surface=False, ckpt="full",
          snapshots=0, store="f32", autotune=False, **kw):
    """n: (nx, nz) or (nx, ny, nz).  dt is 0.1 ms (2D acoustic) or 0.08 ms
    per metre of grid spacing: inside every solver's stability bound at VMAX."""
    c = dict(kind=kind, nx=n[0], ny=n[1] if len(n) == 3 else 1, nz=n[-1], nt=nt, shots=shots, pml=pml, fdhalf=fdhalf,
             d=d, dt=round((1.0e-4 if kind.startswith("acoustic2d") else 0.8e-4) * d, 9), f0=f0, ragged=ragged,
             surface=surface, ckpt=ckpt, snapshots=snapshots, store=store, autotune=autotune)
    c.update(kw)
    return c


def listed():
    cases = [
        # the solver type's own call on a toy model: launch latency and host set-up are all there is
        _case("acoustic2d_forward", (64, 48), 240, pml=12, surface=True, name="acoustic2d_forward_small"),
        # one shot at the size of the published examples, as a one-shot-at-a-time driver runs it
        _case("acoustic2d_forward", (401, 401), 500, pml=40, name="acoustic2d_forward_one_shot"),
        # one iteration of OWL's inversion (new model, OWL's gradient) over a batch of 32 shots
        _case("acoustic2d_gradient_owl", (401, 401), 300, shots=32, pml=40, name="acoustic2d_owl_gradient_32_shots"),
        # one iteration with the exact adjoint under a snapshot budget
        _case("acoustic2d_gradient_exact", (401, 401), 320, shots=32, pml=40, ckpt="binomial", snapshots=40,
              name="acoustic2d_exact_gradient_32_shots"),
        # a torch program that differentiates through the solver: few shots, uneven windows, 16-bit snapshots
        _case("acoustic2d_autograd", (301, 157), 250, shots=6, pml=21, fdhalf=6, ragged=True, ckpt="uniform",
              snapshots=16, store="f16", name="acoustic2d_autograd_ragged"),
        # 3D modelling of a survey: 16 shots, uneven apertures of one layered model
        _case("acoustic3d_forward", (256, 256, 256), 60, shots=16, ragged=True, autotune=True, f0=25.0,
              name="acoustic3d_forward_16_shots"),
        # 3D acoustic gradient of a few shots under a free surface
        _case("acoustic3d_gradient", (121, 110, 93), 120, shots=2, surface=True, f0=25.0, pml=18,
              name="acoustic3d_gradient_surface"),
        # 2D elastic inversion iteration with OWL's depth-refined free surface
        _case("elastic2d_gradient", (301, 201), 250, shots=8, surface=True, name="elastic2d_gradient_surface"),
        # 3D elastic modelling of a survey, flat free surface
        _case("elastic3d_forward", (200, 200, 150), 40, shots=8, surface=True, autotune=True, f0=30.0,
              name="elastic3d_forward_8_shots"),
        # 3D elastic gradient with BF16 boundary records, small uneven model
        _case("elastic3d_gradient", (117, 90, 75), 80, shots=2, store="bf16", pml=15, f0=30.0,
              name="elastic3d_gradient_bf16"),
        # anisotropic modelling of a whole line under a free surface
        _case("fsg2d_forward", (801, 401), 250, shots=32, d=5.0, ragged=True, surface=True, autotune=True, f0=30.0,
              name="fsg2d_forward_32_shots"),
        # anisotropic gradient of a few shots with FP16 boundary records
        _case("fsg2d_gradient", (333, 171), 200, shots=8, d=5.0, ragged=True, store="f16", pml=15, f0=30.0,
              name="fsg2d_gradient_f16"),
    ]
    return cases


# The ranges that the listed cases stand for: per kind the largest edge, time
# steps, shots, and the options its users switch.
RANGES = {
    "acoustic2d_forward": dict(n=(40, 501), nt=(100, 500), shots=(1, 8), surface=(False, True)),
    "acoustic2d_gradient_owl": dict(n=(60, 401), nt=(120, 300), shots=(1, 32), surface=(False, True)),
    "acoustic2d_gradient_exact": dict(n=(60, 401), nt=(120, 320), shots=(1, 32), surface=(False,)),
    "acoustic2d_autograd": dict(n=(60, 320), nt=(100, 250), shots=(1, 8), surface=(False,)),
    "acoustic3d_forward": dict(n=(40, 256), nt=(30, 80), shots=(1, 16), surface=(False, True)),
    "acoustic3d_gradient": dict(n=(40, 130), nt=(80, 120), shots=(1, 3), surface=(False, True)),
    "elastic2d_gradient": dict(n=(60, 301), nt=(120, 250), shots=(1, 8), surface=(False, True)),
    "elastic3d_forward": dict(n=(40, 200), nt=(30, 60), shots=(1, 8), surface=(False, True)),
    "elastic3d_gradient": dict(n=(40, 110), nt=(60, 90), shots=(1, 2), surface=(False, True)),
    "fsg2d_forward": dict(n=(80, 801), nt=(100, 250), shots=(1, 32), surface=(False, True)),
    "fsg2d_gradient": dict(n=(60, 333), nt=(120, 200), shots=(1, 8), surface=(False, True)),
}


def draw(rng):
    top = max(work(c)["bytes"] for c in listed())

    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    while True:
        kind = rng.choice(sorted(RANGES))
        r = RANGES[kind]
        big = log_int(*r["n"])
        dims = 3 if "3d" in kind else 2
        n = tuple(max(r["n"][0], int(big * rng.uniform(0.5, 1.0))) for _ in range(dims - 1))
        n = (big,) + n
        d = 5.0 if kind.startswith("fsg") else 10.0
        surface = rng.choice(r["surface"])
        ckpt = rng.choice(["full", "uniform", "binomial"]) if kind[10:] in ("_gradient_exact", "_autograd") else "full"
        has_records = kind in ("elastic2d_gradient", "elastic3d_gradient", "fsg2d_gradient")
        store = rng.choice(["f32", "f16", "bf16"] if has_records else ["f32", "f32", "f16"]) \
            if has_records or ckpt != "full" else "f32"
        c = _case(kind, n, rng.randint(*r["nt"]), shots=log_int(*r["shots"]), pml=rng.randint(12, 40 if dims == 2 else 20),
                  fdhalf=rng.choice([4, 4, 4, 2, 3, 5, 6, 8]), d=d, f0=30.0 if dims == 3 or d == 5.0 else 20.0,
                  ragged=rng.random() < 0.5, surface=surface, ckpt=ckpt,
                  snapshots=rng.randint(8, 40) if ckpt != "full" else 0, store=store, autotune=rng.random() < 0.5)
        w = work(c)["bytes"]
        if w <= top and w < 4.0e12:
            return c


# ---- inputs -----------------------------------------------------------------
def _dims(c):
    return 3 if "3d" in c["kind"] else 2


def _shape(c):
    return (c["nz"], c["ny"], c["nx"]) if _dims(c) == 3 else (c["nz"], c["nx"])


def _smooth_field(shape, seed, cell=8):
    """A smooth random field with values within [-1, 1]: a coarse normal grid
    interpolated linearly."""
    g = torch.Generator().manual_seed(seed)
    coarse = torch.randn([1, 1] + [max(2, s // cell + 1) for s in shape], generator=g).clamp(-2.5, 2.5) / 2.5
    mode = "trilinear" if len(shape) == 3 else "bilinear"
    return torch.nn.functional.interpolate(coarse, size=shape, mode=mode, align_corners=True)[0, 0].numpy()


def _model(c, seed, shift=0.0):
    """vp grows with depth from 1600 to 4000 m/s with +-8 % of smooth
    heterogeneity; Gardner's rho."""
    shape = _shape(c)
    z = np.arange(shape[0], dtype=np.float32).reshape((-1,) + (1,) * (len(shape) - 1)) / np.float32(max(1, shape[0] - 1))
    vp = (1600.0 + 2400.0 * z) * (1.0 + 0.08 * _smooth_field(shape, seed) + shift)
    vp = np.clip(vp, 1450.0, VMAX).astype(np.float32)
    return vp, (310.0 * np.power(vp, 0.25)).astype(np.float32)


def _elastic(c, seed, shift=0.0):
    vp, rho = _model(c, seed, shift)
    return vp, (vp / np.float32(1.8)).astype(np.float32), rho


def _windows(c):
    """Per shot 1-based (beg, end) along x (and y): the whole model, or an
    aperture of 0.5 to 1 of it.  A survey's apertures are part of the case,
    not of its inputs."""
    rng = np.random.default_rng(c["nx"] + 1000 * c["nz"])
    out = []
    for k in range(c["shots"]):
        w = []
        for n in ((c["nx"], c["ny"]) if _dims(c) == 3 else (c["nx"],)):
            size = int(rng.integers(n // 2, n + 1)) if c["ragged"] else n
            centre = int(rng.integers(1, n + 1))
            beg = min(max(1, centre - size // 2), n - size + 1)
            w.append((beg, beg + size - 1))
        out.append(w)
    return out


def _acquisition(c, seed):
    """Per shot (sources, receivers, window): positions on quarter cells, so
    most taps are off the nodes; a receiver line at every node (2D) or a grid
    of 12 x 12 (3D) near the top of the window."""
    rng = np.random.default_rng(seed + 13)
    d, out = c["d"], []
    force = not c["kind"].startswith("acoustic")
    for w in _windows(c):
        src = dict(f0=c["f0"], amp=1.0e6 if force else 1.0, mechanism="force" if force else "explosion")
        depth = 3.0 + 0.25 * int(rng.integers(0, 8))
        pos = []
        for beg, end in w:
            pos.append((beg - 1 + 0.25 * int(rng.integers(4 * ((end - beg) // 4), 4 * (3 * (end - beg) // 4) + 1))) * d)
        src.update(x=pos[0], z=depth * d)
        if len(w) == 2:
            src["y"] = pos[1]
            xs, ys = [np.linspace(b + 1, e - 3, 12).astype(int) for b, e in w]
            rec = [dict(x=float(x * d), y=float((y + 0.25) * d), z=2.5 * d) for y in ys for x in xs]
        else:
            rec = [dict(x=float((i - 0.75) * d), z=2.25 * d) for i in range(w[0][0] + 1, w[0][1])]
        out.append((src, rec, w))
    return out


def _shots(c, seed):
    out = []
    for k, (s, recs, w) in enumerate(_acquisition(c, seed)):
        g = Geometry(id=k + 1, srcr=[Source(**s)], recr=[Receiver(**r) for r in recs])
        if not c["ragged"]:
            win = None
        elif c["kind"].startswith("acoustic2d"):
            win = Window(w[0][0], w[0][1], 1, c["nz"], (w[0][0] - 1) * c["d"], 0.0)
        else:
            win = dict(nxbeg=w[0][0], nxend=w[0][1], nzbeg=1, nzend=c["nz"])
            if len(w) == 2:
                win.update(nybeg=w[1][0], nyend=w[1][1])
        out.append((g, win))
    return out


LAG = 4


def _late(a):
    out = a * 0
    out[..., LAG:] = a[..., :-LAG]
    return out


def prepare(case, seed):
    c, kind, d = case, case["kind"], case["d"]
    tmax = (c["nt"] - 1) * c["dt"]
    shots = _shots(c, seed)
    opts = dict(pml=c["pml"], fdhalf=c["fdhalf"])
    st = dict(case=c)
    if kind.startswith("acoustic2d"):
        vp, rho = _model(c, seed)
        true = _model(c, seed, 0.03)
        grad = kind != "acoustic2d_forward"
        b = Acoustic2DBatch(c["nx"], c["nz"], d, d, *(true if grad else (vp, rho)), shots, c["dt"], tmax,
                            free_surface=c["surface"], **opts)
        if kind == "acoustic2d_autograd":
            obs = np.concatenate(b.forward(), axis=0)
            st.update(obs=torch.from_numpy(obs).cuda(), vp=torch.from_numpy(vp).cuda().requires_grad_(),
                      rho=torch.from_numpy(rho).cuda().requires_grad_())
        elif grad:
            b.observe()
            st.update(vp=vp, rho=rho)
    elif kind.startswith("acoustic3d"):
        b = Acoustic3DBatch(c["nx"], c["ny"], c["nz"], d, d, d, *_model(c, seed), shots, c["dt"], tmax,
                            free_surface=c["surface"], **opts)
    elif kind.startswith("elastic2d"):
        b = Elastic2DBatch(c["nx"], c["nz"], d, d, *_elastic(c, seed), shots, c["dt"], tmax,
                           surface={} if c["surface"] else None, **opts)
    elif kind.startswith("elastic3d"):
        b = Elastic3DBatch(c["nx"], c["ny"], c["nz"], d, d, d, *_elastic(c, seed), shots, c["dt"], tmax,
                           free_surface=c["surface"], **opts)
    else:
        vp, vs, rho = _elastic(c, seed)
        eps, delta = 0.08 + 0.06 * _smooth_field(_shape(c), seed + 1), 0.04 + 0.03 * _smooth_field(_shape(c), seed + 2)
        theta = 0.4 * _smooth_field(_shape(c), seed + 3)
        b = FSG2DBatch(c["nx"], c["nz"], d, d, tti_cij("thomsen", vp, vs, rho, eps, delta, theta), rho, shots, c["dt"],
                       tmax, surface={} if c["surface"] else None, **opts)
    if kind.endswith("_gradient") and not kind.startswith("acoustic"):
        b.set_record_storage(STORE[c["store"]])
    if kind.endswith("_gradient"):
        # observed data: the modelled traces, weaker and LAG samples late
        st["obs"] = [0.9 * _late(t) if isinstance(t, np.ndarray) else tuple(0.9 * _late(x) for x in t)
                     for t in b.forward()]
    if c["autotune"] and not kind.startswith("acoustic2d"):
        b.autotune()
    st["batch"] = b
    return st


# ---- one pass ---------------------------------------------------------------
def run(state):
    c, b = state["case"], state["batch"]
    kind = c["kind"]
    if kind.endswith("_forward"):
        return b.forward()
    if kind == "acoustic2d_gradient_owl":
        b.set_model(state["vp"], state["rho"])
        return b.gradient(mode=OWL_GRAD_OWL, want_traces=False)[:3]
    if kind == "acoustic2d_gradient_exact":
        b.set_model(state["vp"], state["rho"])
        return b.gradient(mode=OWL_GRAD_EXACT, ckpt=CKPT[c["ckpt"]], ckpt_param=c["snapshots"], store=STORE[c["store"]],
                          want_traces=False)[:3]
    if kind == "acoustic2d_autograd":
        vp, rho = state["vp"], state["rho"]
        tr = propagate(vp, rho, b, CKPT[c["ckpt"]], c["snapshots"], STORE[c["store"]])
        loss = 0.5 * ((tr - state["obs"]) ** 2).sum()
        return (tr.detach(),) + torch.autograd.grad(loss, (vp, rho))
    return b.gradient(state["obs"])


# ---- compulsory work --------------------------------------------------------
# Per updated point and step: bytes of the wavefields read and written once
# (state), of the medium (model), PML memory variables per damped axis, and
# arithmetic beyond the stencils.
SOLVER = {"acoustic2d": dict(state=24, model=8, mem=2, sten=4, flops=16, grads=2),
          "acoustic3d": dict(state=32, model=8, mem=2, sten=6, flops=22, grads=2),
          "elastic2d": dict(state=40, model=20, mem=4, sten=8, flops=30, grads=3),
          "elastic3d": dict(state=72, model=32, mem=6, sten=18, flops=70, grads=3),
          "fsg2d": dict(state=80, model=56, mem=8, sten=16, flops=70, grads=7)}


def _binomial_steps(n, s):
    """Forward steps of an optimal checkpoint schedule over n steps with s
    snapshots: each step at most r times, r the smallest with C(s+r, s) >= n."""
    if s >= n:
        return n
    r = 1
    while math.comb(s + r, s) < n:
        r += 1
    return r * n - math.comb(s + r, r - 1) + 1


def work(case):
    c, p = case, SOLVER[case["kind"].split("_")[0]]
    pml, nt, kind = c["pml"], c["nt"], c["kind"]
    pts = distinct = slab = inside = 0
    seen = set()
    for w in _windows(c):
        sides = [e - b + 1 for b, e in w] + [c["nz"]]
        n = math.prod(s + 2 * pml for s in sides)
        pts += n
        inside += math.prod(sides)
        slab += sum(2 * pml * n // (s + 2 * pml) for s in sides)
        if tuple(w) not in seen:
            seen.add(tuple(w))
            distinct += n
    step = p["state"] * pts + p["model"] * distinct + 8 * p["mem"] * slab
    flop = (p["sten"] * (3 * c["fdhalf"] - 1) + p["flops"]) * pts
    if kind.endswith("_forward"):
        return {"bytes": float(step * (nt - 1)), "flops": float(flop * (nt - 1))}
    if "exact" in kind or "autograd" in kind:
        n = nt - 1
        fwd = n if c["ckpt"] == "full" else 2 * n if c["ckpt"] == "uniform" else max(n, _binomial_steps(n, c["snapshots"]))
        # the adjoint step reads the forward state and updates two FP64 sums
        return {"bytes": float(step * fwd + (step + (12 + 32) * pts) * n), "flops": float(flop * (fwd + n) + 10 * pts * n)}
    back = max(1, nt - int(round(1.0 / c["f0"] / c["dt"])) + 1)
    return {"bytes": float(step * (nt - 1) + (2 * step + 16 * p["grads"] * inside) * back),
            "flops": float(flop * (nt - 1) + (2 * flop + 12 * p["grads"] * inside) * back)}


def tolerance(case):
    """About four times the distance of the FP32 path from FP64 (largest over
    the outputs: 5e-6 for traces, 2e-6 for gradients, which sum in FP64);
    wider where the caller asks for 16-bit snapshots or records."""
    if case["store"] == "bf16":
        return {"rel": 1e-2}
    if case["store"] == "f16":
        return {"rel": 1e-3}
    return {"rel": 2e-5}


# ---- FP64 restatement in torch ----------------------------------------------
COEF = {2: (1.129042, -0.04301412), 3: (1.185991, -0.07249965, 0.006301572),
        4: (1.217990, -0.09382142, 0.01507536, -0.001700324),
        5: (1.236607, -0.1082265, 0.0234344, -0.005033546, 0.0006817483),
        6: (1.247662, -0.1175538, 0.0299797, -0.008719078, 0.002215897, -0.0003462075),
        7: (1.254799, -0.1238928, 0.03494371, -0.01208897, 0.004132531, -0.00119711, 0.0002122227),
        8: (1.259312, -0.1280347, 0.03841945, -0.01473229, 0.005924913, -0.002248618, 0.0007179226, -0.0001400855)}
DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _f64(a):
    return torch.as_tensor(np.asarray(a, np.float64), device=DEV)


def _sinc9(x):
    """Weights of nodes -4 .. 4 for a point at x: sinc under a Kaiser window."""
    if x == 0.0:
        return np.eye(9)[4]
    t = np.arange(-4, 5) - x
    u = t / 4.0
    w = np.where(np.abs(u) <= 1, np.i0(6.31 * np.sqrt(np.maximum(0, 1 - u * u))) / np.i0(6.31), 0.0)
    return np.sinc(t) * w


class _Grid:
    """Padded grids of shots with one window shape, stacked along a leading
    axis; spatial axes (z, x) or (z, y, x) with `pad` = pml + R cells a side.
    Node 1 is element pad."""

    def __init__(self, c, shots, windows, medium, velocity):
        self.c, self.R, self.pml = c, c["fdhalf"], c["pml"]
        self.pad = self.pml + self.R
        self.d, self.dt, self.nt = float(np.float32(c["d"])), float(np.float32(c["dt"])), c["nt"]
        self.dims = _dims(c)
        self.fs = c["surface"]
        self.n = [c["nz"]] + [e - b + 1 for b, e in reversed(windows[0])]
        self.ns = len(shots)
        self.shape = [self.ns] + [n + 2 * self.pad for n in self.n]
        cut = [[slice(0, c["nz"])] + [slice(b - 1, e) for b, e in reversed(w)] for w in windows]
        self.medium = [torch.stack([self._padded(_f64(m[tuple(k)])) for k in cut]) for m in medium]
        edge = []
        for k in cut:
            v = velocity[tuple(k)].astype(np.float64)
            edge.append(max(np.take(v, i, axis).max() for axis in range(self.dims) for i in (0, -1)))
        self.edge = np.array(edge)
        self.org = [[0] + [b - 1 for b, _ in reversed(w)] for w in windows]
        self.shots = shots
        self.amax = math.pi * c["f0"]
        n = int(math.ceil(np.float32(2.0) / np.float32(c["f0"]) / np.float32(c["dt"])))
        tau = np.arange(n) * self.dt - 1.0 / c["f0"]
        a = (math.pi * c["f0"] * tau) ** 2
        w = (1 - 2 * a) * np.exp(-a)
        self.stf = w / np.abs(w).max()
        self.hnt = int(math.floor(n / 2.0 + 0.5))

    def _padded(self, m):
        for axis in range(self.dims):
            idx = (torch.arange(m.shape[axis] + 2 * self.pad, device=DEV) - self.pad).clamp(0, m.shape[axis] - 1)
            m = m.index_select(axis, idx)
        return m

    def zeros(self):
        return torch.zeros(self.shape, dtype=torch.float64, device=DEV)

    def box(self, axis_ranges=None):
        """Slices of the updated nodes 1 - pml .. n + pml."""
        return (slice(None),) + tuple(slice(self.R, -self.R) for _ in range(self.dims))

    def diff(self, f, axis, off):
        """Staggered difference along spatial axis: off 0: f(i+m) - f(i-m+1); off -1: f(i+m-1) - f(i-m), on the box."""
        R, out = self.R, 0.0
        for m, cm in enumerate(COEF[R], 1):
            def part(s):
                k = [slice(None)] + [slice(R, -R)] * self.dims
                k[axis + 1] = slice(R + s, f.shape[axis + 1] - R + s)
                return f[tuple(k)]
            out = out + cm * (part(m + off) - part(1 - m + off))
        return out / self.d

    def profile(self, axis, half, elastic=False):
        """CFS-PML (a, b) along one axis over the box, zero outside the slabs, shaped to broadcast.  Half nodes lie
        half a cell before the node; a free surface has no top slab."""
        n, pml = self.n[axis], self.pml
        i = np.arange(1 - pml, n + pml + 1, dtype=np.float64)
        lo, hi = i <= 1, i >= (n if elastic else n + 1)
        dist = np.where(i <= 1, np.abs(i - 1 - 0.5 * half), np.abs(i - n - 0.5 * half))
        if self.fs and axis == 0:
            lo[:] = False
        on = lo | hi
        if not elastic:
            on &= (i <= 1) | (i >= n + 1) if half else (i <= 0) | (i >= n + 1)
        nd = dist / pml
        alpha = np.maximum(self.amax * (1 - nd), 0.25 * self.amax)
        damp = self.edge[:, None] * 3 * math.log(1e5) / (2 * pml * self.d) * (nd * nd)[None]
        den = 2 + self.dt * (alpha + damp)
        a = np.where(on, -2 * self.dt * damp / den, 0.0)
        b = np.where(on, (2 - self.dt * (alpha + damp)) / den, 0.0)
        shape = [self.ns] + [1] * self.dims
        shape[axis + 1] = len(i)
        return _f64(a).reshape(shape), _f64(b).reshape(shape)

    def taps(self, s, point, half_axis=None):
        """(flat cells, weights) of a point of shot s: 9 sinc weights an axis, on half nodes along half_axis."""
        idx, wts = [], []
        pos = [point["z"]] + [point[k] for k in (("y", "x") if self.dims == 3 else ("x",))]
        for axis, x in enumerate(pos):
            g = x / self.d - self.org[s][axis] + (0.5 if axis == half_axis else 0.0)
            near = math.floor(g + 0.5)
            idx.append(near + self.pad + np.arange(-4, 5))
            wts.append(_sinc9(g - near))
        cells, w = idx[0], wts[0]
        for axis in range(1, self.dims):
            cells = (cells[..., None] * self.shape[axis + 1] + idx[axis])
            w = w[..., None] * wts[axis]
        cells, w = cells.ravel(), w.ravel()
        cells = cells + s * int(np.prod(self.shape[1:]))
        return cells[w != 0], w[w != 0]

    def below(self, cells):
        """Cells at depth node 2 or deeper (all of them without a free surface)."""
        z = cells % int(np.prod(self.shape[1:])) // int(np.prod(self.shape[2:])) - self.pad + 1
        return z >= 2 if self.fs else z >= -10 ** 9

    def point_map(self, half_axis=None):
        """Sparse (receivers of all shots) x (cells) sampling matrix."""
        rows, cells, w, r = [], [], [], 0
        for s, (_, recs, _) in enumerate(self.shots):
            for p in recs:
                cc, ww = self.taps(s, p, half_axis)
                rows.append(np.full(len(cc), r))
                cells.append(cc)
                w.append(ww)
                r += 1
        rows, cells, w = (np.concatenate(a) for a in (rows, cells, w))
        idx = torch.as_tensor(np.stack([rows, cells]).astype(np.int64), device=DEV)
        return idx, _f64(w), r

    def sample(self, m, f):
        (rows, cells), w, n = m
        return torch.zeros(n, dtype=torch.float64, device=DEV).index_add(0, rows, f.reshape(-1)[cells] * w)

    def source(self, half_axis=None):
        cells, w = zip(*(self.taps(s, p, half_axis) for s, (p, _, _) in enumerate(self.shots)))
        cells, w = np.concatenate(cells), np.concatenate(w)
        keep = self.below(cells)
        return torch.as_tensor(cells[keep], device=DEV), _f64(w[keep])


class _Acoustic(_Grid):
    """Pressure-velocity scheme: p on nodes, v[a] half a cell before them along axis a."""

    def __init__(self, c, shots, windows, vp, rho):
        super().__init__(c, shots, windows, (vp, rho), vp)
        self.src = self.source()
        self.map = self.point_map()
        self.pi = [self.profile(a, False) for a in range(self.dims)]
        self.ph = [self.profile(a, True) for a in range(self.dims)]
        box = self.box()
        z = torch.arange(1 - self.pml, self.n[0] + self.pml + 1, device=DEV).reshape([1, -1] + [1] * (self.dims - 1))
        self.keep_p = (z >= 2).double() if self.fs else None
        self.keep_v = [((z >= (2 if a == 0 else 1)).double() if self.fs else None) for a in range(self.dims)]
        self.set_model(*self.medium)
        self.boxs = box

    def set_model(self, vp, rho):
        box = self.box()
        self.K = (rho * vp ** 2)[box]
        self.buoy = []
        for a in range(self.dims):
            self.buoy.append(1.0 / (0.5 * (rho + rho.roll(1, a + 1)))[box])

    def start(self):
        box = self.zeros()[self.box()]
        return [self.zeros() for _ in range(1 + self.dims)] + [torch.zeros_like(box) for _ in range(2 * self.dims)]

    def write(self, f, new):
        out = f.clone()
        out[self.box()] = new
        return out

    def step(self, st, dt):
        """One update with time step dt (negative for the reverse pass); returns new tensors."""
        D = self.dims
        p, v, mp, mv = st[0], st[1:1 + D], st[1 + D:1 + 2 * D], st[1 + 2 * D:]
        div, mp2, mv2, v2 = 0.0, [], [], []
        for a in range(D):
            g = self.diff(v[a], a, 0)
            m = self.pi[a][0] * g + self.pi[a][1] * mp[a]
            if self.fs:
                m = m * self.keep_p
            mp2.append(m)
            div = div + g + m
        inc = dt * self.K * div
        p = self.write(p, p[self.box()] - (inc if self.keep_p is None else inc * self.keep_p))
        if self.fs:
            top = self.pad  # element of node 1; p(2 - j) = -p(j)
            p = p.clone()
            p[:, top - self.pml:top] = -p[:, top + 1:top + 1 + self.pml].flip(1)
        for a in range(D):
            g = self.diff(p, a, -1)
            m = self.ph[a][0] * g + self.ph[a][1] * mv[a]
            if self.keep_v[a] is not None:
                m = m * self.keep_v[a]
            mv2.append(m)
            inc = dt * self.buoy[a] * (g + m)
            v2.append(self.write(v[a], v[a][self.box()] - (inc if self.keep_v[a] is None else inc * self.keep_v[a])))
        return [p] + v2 + mp2 + mv2

    def inject(self, st, t):
        if t <= len(self.stf):
            amp = self.stf[t - 1] * float(np.float32(1.0)) * self.dt
            st = [st[0].reshape(-1).index_add(0, self.src[0], amp * self.src[1]).reshape(self.shape)] + st[1:]
        return st

    def advance(self, st, t):
        return self.inject(self.step(st, self.dt), t)

    def forward(self, keep=None):
        """Traces (receivers, nt); keep(t, state) sees the state at the start of step t."""
        st = self.start()
        tr = [self.sample(self.map, st[0])]
        if keep:
            keep(1, st)
        for t in range(1, self.nt):
            st = self.advance(st, t)
            tr.append(self.sample(self.map, st[0]))
            if keep:
                keep(t + 1, st)
        return torch.stack(tr, 1), st

    def differentiable_forward(self, vp, rho, chunk=16):
        """forward() under autograd, `chunk` steps recomputed at a time."""
        from torch.utils.checkpoint import checkpoint

        def some(t0, t1, vp, rho, *st):
            self.set_model(vp, rho)
            st, tr = list(st), []
            for t in range(t0, t1):
                st = self.advance(st, t)
                tr.append(self.sample(self.map, st[0]))
            return (torch.stack(tr, 1),) + tuple(st)

        st = self.start()
        out = [self.sample(self.map, st[0])[:, None]]
        for t0 in range(1, self.nt, chunk):
            got = checkpoint(some, t0, min(t0 + chunk, self.nt), vp, rho, *st, use_reentrant=False)
            out.append(got[0])
            st = list(got[1:])
        return torch.cat(out, 1)

    def faces(self, axis):
        """The recorded band of v[axis]: R nodes around each face, whole window plus R on the other axes."""
        R, pad, n = self.R, self.pad, self.n
        k = [slice(None)] + [slice(pad - R, pad + m + R) for m in n]
        lo, hi = list(k), list(k)
        lo[axis + 1] = slice(pad + 1 - R, pad + 1)
        hi[axis + 1] = slice(pad + n[axis], pad + n[axis] + R)
        return tuple(lo), tuple(hi)

    def owl_gradient(self, obs):
        """(misfit per shot, per-shot window gradients, traces) of the boundary-record algorithm; obs None: the
        traces themselves, weaker and late."""
        records, D = {}, self.dims

        def keep(t, st):
            records[t] = [[st[1 + a][f].clone() for f in self.faces(a)] for a in range(D)]

        syn, final = self.forward(keep)
        mis, adj = _l2(self, syn, 0.9 * _late(syn) if obs is None else obs)
        (rows, cells), w, _ = self.map
        st = final[:1 + D] + self.start()[1 + D:]
        rev = self.start()
        inner = (slice(None),) + tuple(slice(self.pad, self.pad + m) for m in self.n)

        def pairs(f, a):
            nxt = list(inner)
            nxt[a + 1] = slice(self.pad + 1, self.pad + self.n[a] + 1)
            return f[inner] + f[tuple(nxt)]

        vp, rho = (m[inner] for m in self.medium)
        gv, gr = torch.zeros_like(vp), torch.zeros_like(vp)
        prev = None
        for t in range(self.nt, max(self.hnt, 1) - 1, -1):
            st = [f.clone() for f in st]
            for a in range(D):
                for f, r in zip(self.faces(a), records[t][a]):
                    st[1 + a][f] = r
            st = self.step(st, -self.dt)
            rev = self.step(rev, -self.dt)
            rev[0] = rev[0].reshape(-1).index_add(0, cells, adj[rows, t - 1] * w).reshape(self.shape)
            dp = st[0][inner] - (prev[0][inner] if prev else 0.0)
            gv = gv - dp * rev[0][inner] / (rho * vp ** 3)
            for a in range(D):
                gr = gr + (pairs(st[1 + a], a) - (pairs(prev[1 + a], a) if prev else 0.0)) * pairs(rev[1 + a], a)
            prev = st
        return mis, gv, gr, syn


class _Elastic3(_Grid):
    """3D isotropic velocity-stress scheme with force sources; axes (z, y, x)."""

    def __init__(self, c, shots, windows, vp, vs, rho):
        super().__init__(c, shots, windows, (vp, vs, rho), vp)
        vp, vs, rho = self.medium
        box = self.box()
        mu = rho * vs ** 2
        self.c11, self.c12 = (rho * vp ** 2)[box], (rho * vp ** 2 - 2 * mu)[box]
        inv = 1.0 / mu

        def harmonic(a, b):
            return (4.0 / (inv + inv.roll(1, a + 1) + inv.roll(1, b + 1) + inv.roll(1, a + 1).roll(1, b + 1)))[box]

        self.mu = {(a, b): harmonic(a, b) for a, b in ((0, 1), (0, 2), (1, 2))}
        self.buoy = [1.0 / (0.5 * (rho + rho.roll(1, a + 1)))[box] for a in range(3)]
        self.pi = [self.profile(a, False, True) for a in range(3)]
        self.ph = [self.profile(a, True, True) for a in range(3)]
        self.map = [self.point_map(a) for a in range(3)]
        self.src = self.source(0)  # a vertical force: vz at half nodes along z
        self.rho_src = [float(rho[s].reshape(-1)[int(self._node(s))]) for s in range(self.ns)]
        z = torch.arange(1 - self.pml, self.n[0] + self.pml + 1, device=DEV).reshape(1, -1, 1, 1)
        self.keep1 = (z >= 1).double() if self.fs else 1.0
        self.keep2 = (z >= 2).double() if self.fs else 1.0
        self.row1 = z == 1

    def _node(self, s):
        p = self.shots[s][0]
        k = [math.floor(x / self.d - o + 0.5) + self.pad for x, o in zip((p["z"], p["y"], p["x"]), self.org[s])]
        return (k[0] * self.shape[2] + k[1]) * self.shape[3] + k[2]

    def forward(self):
        box, dt, top = self.box(), self.dt, self.pad
        v = [self.zeros() for _ in range(3)]
        sn = [self.zeros() for _ in range(3)]
        ss = {k: self.zeros() for k in self.mu}
        mem = {}

        def damped(key, g, prof, keep):
            a, b = prof
            m = (a * g + b * mem.get(key, 0.0)) * keep
            mem[key] = m
            return g + m

        def top_zero(planes):
            for m in range(1, planes + 1):
                v[0][:, top + 1 - m] = 0.0
                v[1][:, top - m] = 0.0
                v[2][:, top - m] = 0.0

        out = [[], [], []]
        for t in range(1, self.nt + 1):
            if self.fs:
                for m in range(1, 5):
                    v[1][:, top - m] = v[1][:, top + m]
                    v[2][:, top - m] = v[2][:, top + m]
                    v[0][:, top + 1 - m] = v[0][:, top + m]
            for a in range(3):
                out[a].append(self.sample(self.map[a], v[a]))
            if t == self.nt:
                break
            if self.fs:
                top_zero(self.R)
            e = [damped(("n", a), self.diff(v[a], a, 0), self.pi[a], self.keep1) for a in range(3)]
            if self.fs:
                ratio = self.c12 / self.c11
                e[0] = torch.where(self.row1, -ratio * (e[1] + e[2]), e[0])
                mem[("n", 0)] = torch.where(self.row1, 0.0, mem[("n", 0)])
            for a in range(3):
                inc = self.c11 * e[a] + self.c12 * (e[(a + 1) % 3] + e[(a + 2) % 3])
                sn[a][box] += dt * inc * self.keep1
            for (a, b), f in ss.items():
                keep = self.keep2 if a == 0 else self.keep1
                g = damped(("s", a, b), self.diff(v[b], a, -1), self.ph[a], keep)
                g = g + damped(("s", b, a), self.diff(v[a], b, -1), self.ph[b], keep)
                f[box] += dt * self.mu[a, b] * g * keep
            if self.fs:
                for m in range(1, self.R + 1):
                    for f in (sn[0], sn[1], sn[2], ss[1, 2]):
                        f[:, top - m] = -f[:, top + m]
                    sn[0][:, top] = 0.0
                    ss[0, 1][:, top + 1 - m] = -ss[0, 1][:, top + m]
                    ss[0, 2][:, top + 1 - m] = -ss[0, 2][:, top + m]
            for a in range(3):
                keep = self.keep2 if a == 0 else self.keep1
                g = damped(("v", a, a), self.diff(sn[a], a, -1), self.ph[a], keep)
                for b in range(3):
                    if b != a:
                        g = g + damped(("v", a, b), self.diff(ss[min(a, b), max(a, b)], b, 0), self.pi[b], keep)
                v[a][box] += dt * self.buoy[a] * g * keep
            if t <= len(self.stf):
                cells, w = self.src
                size = int(np.prod(self.shape[1:]))
                amp = _f64([self.stf[t - 1] * 1.0e6 * dt / r for r in self.rho_src])
                v[0] = v[0].reshape(-1).index_add(0, cells, amp[cells // size] * w).reshape(self.shape)
        return [torch.stack(o, 1) for o in out]


def _l2(g, syn, obs):
    """Per-shot misfit and adjoint source of the L2 misfit; traces far below the largest one are left out."""
    mis, adj, r = [], torch.zeros_like(syn), 0
    for _, recs, _ in g.shots:
        k = slice(r, r + len(recs))
        r += len(recs)
        no, ns = obs[k].norm(dim=1), syn[k].norm(dim=1)
        ok = (no >= 1e-6 * no.max()) & (ns >= 1e-6 * ns.max()) & (no * ns != 0)
        adj[k] = (syn[k] - obs[k]) * ok[:, None]
        mis.append(float((adj[k] ** 2).sum()))
    return mis, adj


def _groups(c, seed):
    """(shot numbers, acquisition) of shots whose windows have one shape, few enough at a time for the card."""
    acq = _acquisition(c, seed)
    by = {}
    for k, (_, _, w) in enumerate(acq):
        by.setdefault(tuple(e - b for b, e in w), []).append(k)
    most = 8 if _dims(c) == 2 else 1
    return [(ks[i:i + most], [acq[k] for k in ks[i:i + most]]) for ks in by.values() for i in range(0, len(ks), most)]


def exact(case, seed):
    """FP64 outputs of run() from plain tensors.  None for the gradients of
    the elastic and anisotropic solvers and the anisotropic forward, whose
    plain-tensor form (per-shot refined meshes, reconstruction, scans of the
    Christoffel equation per edge cell) takes minutes."""
    c, kind = case, case["kind"]
    if kind.startswith("fsg") or kind.endswith("_gradient") and kind.startswith("elastic"):
        return None
    with torch.no_grad():
        if kind == "elastic3d_forward":
            out, med = [None] * c["shots"], _elastic(c, seed)
            for ks, shots in _groups(c, seed):
                vz, vy, vx = _Elastic3(c, shots, [s[2] for s in shots], *med).forward()
                n = len(shots[0][1])
                for i, k in enumerate(ks):
                    out[k] = tuple(f[i * n:(i + 1) * n].cpu().numpy() for f in (vx, vy, vz))
            return out
        med = _model(c, seed)
        if kind.endswith("_forward"):
            out = [None] * c["shots"]
            for ks, shots in _groups(c, seed):
                tr, _ = _Acoustic(c, shots, [s[2] for s in shots], *med).forward()
                n = len(shots[0][1])
                for i, k in enumerate(ks):
                    out[k] = tr[i * n:(i + 1) * n].cpu().numpy()
            return out
        true = None if kind == "acoustic3d_gradient" else _model(c, seed, 0.03)
        mis = np.zeros(c["shots"])
        gv, gr = (torch.zeros(_shape(c), dtype=torch.float64, device=DEV) for _ in range(2))
        traces = [None] * c["shots"]
        for ks, shots in _groups(c, seed):
            wins = [s[2] for s in shots]
            obs = _Acoustic(c, shots, wins, *true).forward()[0] if true else None
            g = _Acoustic(c, shots, wins, *med)
            n = len(shots[0][1])
            if kind in ("acoustic2d_gradient_owl", "acoustic3d_gradient"):
                m, a, r, tr = g.owl_gradient(obs)
            else:
                with torch.enable_grad():
                    cut = [(slice(0, c["nz"]),) + tuple(slice(b - 1, e) for b, e in reversed(w)) for w in wins]
                    leaf = [[_f64(x[k]).requires_grad_() for k in cut] for x in med]
                    pads = [torch.stack([g._padded(x) for x in xs]) for xs in leaf]
                    tr = g.differentiable_forward(*pads)
                    if kind == "acoustic2d_autograd":
                        m, adj = [0.0] * len(ks), tr.detach() - obs
                    else:
                        m, adj = _l2(g, tr.detach(), obs)
                    got = torch.autograd.grad((tr * adj).sum(), leaf[0] + leaf[1])
                    a, r, tr = got[:len(ks)], got[len(ks):], tr.detach()
            for i, k in enumerate(ks):
                traces[k] = tr[i * n:(i + 1) * n]
                mis[k] = m[i]
                at = (slice(0, c["nz"]),) + tuple(slice(b - 1, e) for b, e in reversed(wins[i]))
                gv[at] += a[i]
                gr[at] += r[i]
        if kind == "acoustic2d_autograd":
            return torch.cat(traces), gv, gr
        out = (mis, gv.cpu().numpy(), gr.cpu().numpy())
        return out + ([t.cpu().numpy() for t in traces],) if kind == "acoustic3d_gradient" else out
