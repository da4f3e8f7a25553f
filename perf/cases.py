"""The framework's measured workloads: forward modelling, RTM, FWI gradients
and the snapshot codec, through the public Python entry points.

Every case is a dict of plain values; `family` picks the path:

  fwd     Propagator.run + record        (2D / 3D; GPU, CPU and TTI form; split / unsplit)
  rtm     Propagator.rtm_shot(_eb, _learned) + rtm_image   (2D / 3D)
  batch   Batch.rtm + image              (many uneven 2D shots)
  grad    Gradient.run                   (2D / 3D, FP32 / FP64)
  codec   Autoencoder.bq_encode + bq_decode

Models are a depth gradient with smooth random anomalies; observed records
are synthetic reflection hyperbolas with noise, so that inputs depend on the
seed alone.  `exact` restates the equations in plain torch float64.
"""
import math
import random

import numpy as np
import torch

from geophysics_amd import vti

PI = 3.141592653          # the value the method's source terms and tapers are defined with
C4 = (1.196289, -0.0797526, 0.009570313, -0.0006975447)
DEV = "cuda" if torch.cuda.is_available() else "cpu"


# ------------------------------------------------------------------ cases ----
def listed():
    return [
        # the smallest call: a test shot over a 60 x 50 model, 300 steps with the SV taper (launches and latency)
        dict(name="fwd2d_60x50", family="fwd", form="gpu", nx=60, nz=50, npml=20, nt=300, sv=1, unsplit=0),
        # the 2D configuration of the CPU driver's semantics: 400 x 400, 2000 steps
        dict(name="fwd2d_400x400_cpuform", family="fwd", form="cpu", nx=400, nz=400, npml=20, nt=2000, sv=0, unsplit=0),
        # the tilted (TTI) program's own size: 600 x 300, 50-cell layer, 801 steps
        dict(name="fwd2d_tti_600x300", family="fwd", form="tti", nx=600, nz=300, npml=50, nt=801, sv=1, unsplit=0),
        # a long 2D line, odd sizes, with the unsplit interior
        dict(name="fwd2d_2401x803_unsplit", family="fwd", form="gpu", nx=2401, nz=803, npml=20, nt=400, sv=1, unsplit=1),
        # 3D modelling in the drop-in (split) form on a ragged volume
        dict(name="fwd3d_201x187x143_split", family="fwd", form="gpu", nx=201, ny=187, nz=143, npml=20, nt=60, sv=1,
             unsplit=0, rec_step=2),
        # the headline volume: 512^3, 30-cell layer, unsplit interior
        dict(name="fwd3d_512_unsplit", family="fwd", form="gpu", nx=512, ny=512, nz=512, npml=30, nt=12, sv=1,
             unsplit=1, rec_step=2),
        # migration of one 2D shot with a few checkpoints
        dict(name="rtm2d_601x301", family="rtm", how="plain", nx=601, nz=301, npml=20, nt=600, nsnap=32, every=1,
             unsplit=0),
        # migration of one 3D shot from checkpoints, unsplit interior
        dict(name="rtm3d_128_unsplit", family="rtm", how="plain", nx=128, ny=128, nz=128, npml=20, nt=160, nsnap=12,
             every=4, unsplit=1),
        # the same with the source field kept by the quantized snapshot codec
        dict(name="rtm3d_128_learned", family="rtm", how="learned", nx=128, ny=128, nz=128, npml=20, nt=240, nsnap=0,
             every=4, unsplit=1),
        # a line's shots migrated together: uneven grids, checkpoints
        dict(name="batch_rtm_24shots", family="batch", shots=24, lo=300, hi=1200, nt=96, nsnap=10, unsplit=1),
        # one FWI gradient of a 1000 x 300 line
        dict(name="grad2d_1000x300", family="grad", ndim=2, nx=1000, nz=300, npml=20, nt=400, nsnap=40, fp64=0),
        # a stored 384^3 snapshot: encode and decode
        dict(name="codec_384", family="codec", n=384, tol=7e-4),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One case of the ranges that the listed ones stand for."""
    f = rng.choice(["fwd2d", "fwd2d", "fwd3d", "fwd3d", "rtm2d", "rtm3d", "batch", "grad", "codec"])
    if f == "fwd2d":
        form = rng.choice(["gpu", "gpu", "cpu", "tti"])
        nx, nz = _logint(rng, 60, 2400), _logint(rng, 50, 800)
        return dict(family="fwd", form=form, nx=nx, nz=nz, npml=rng.choice([10, 20, 20, 30, 50]),
                    nt=_logint(rng, 100, 800), sv=rng.randint(0, 1), unsplit=rng.randint(0, 1) if form == "gpu" else 0)
    if f == "fwd3d":
        n = [_logint(rng, 40, 400) for _ in range(3)]
        return dict(family="fwd", form="gpu", nx=n[0], ny=n[1], nz=n[2], npml=rng.choice([10, 20, 30]),
                    nt=rng.randint(8, 40), sv=rng.randint(0, 1), unsplit=rng.randint(0, 1), rec_step=rng.randint(1, 3))
    if f == "rtm2d":
        return dict(family="rtm", how=rng.choice(["plain", "plain", "eb"]), nx=_logint(rng, 100, 1200),
                    nz=_logint(rng, 80, 600), npml=20, nt=_logint(rng, 100, 500), nsnap=rng.randint(4, 40),
                    every=rng.randint(1, 4), unsplit=rng.randint(0, 1))
    if f == "rtm3d":
        how = rng.choice(["plain", "learned", "eb"])
        n = [8 * rng.randint(6, 18)] * 3 if how == "learned" else [_logint(rng, 40, 140) for _ in range(3)]
        return dict(family="rtm", how=how, nx=n[0], ny=n[1], nz=n[2], npml=rng.choice([10, 20]),
                    nt=_logint(rng, 40, 160), nsnap=rng.randint(4, 20), every=4, unsplit=rng.randint(0, 1))
    if f == "batch":
        return dict(family="batch", shots=rng.randint(2, 24), lo=100, hi=rng.randint(300, 1000),
                    nt=_logint(rng, 30, 96), nsnap=rng.randint(4, 16), unsplit=rng.randint(0, 1))
    if f == "grad":
        if rng.random() < 0.35:
            return dict(family="grad", ndim=3, nx=_logint(rng, 30, 80), ny=_logint(rng, 30, 80),
                        nz=_logint(rng, 30, 80), npml=10, nt=rng.randint(30, 100), nsnap=rng.randint(4, 20),
                        fp64=rng.randint(0, 1))
        return dict(family="grad", ndim=2, nx=_logint(rng, 80, 1000), nz=_logint(rng, 60, 300), npml=20,
                    nt=_logint(rng, 60, 400), nsnap=rng.randint(4, 40), fp64=rng.randint(0, 1))
    return dict(family="codec", n=8 * rng.randint(6, 47), tol=rng.choice([2e-4, 7e-4, 1e-3, 1e-2]))


# ----------------------------------------------------------------- inputs ----
def _gen(seed, k=0):
    g = torch.Generator(device="cpu")
    g.manual_seed(int(seed) * 1009 + k)
    return g


def _smooth(shape, seed, k):
    """Smooth random field in [0, 1]: coarse noise, interpolated linearly."""
    coarse = [max(2, n // 16 + 2) for n in shape]
    a = torch.rand(coarse, generator=_gen(seed, k), dtype=torch.float32).to(DEV)
    mode = "trilinear" if len(shape) == 3 else "bilinear"
    return torch.nn.functional.interpolate(a[None, None], size=tuple(shape), mode=mode, align_corners=True)[0, 0]


def _model(shape, seed):
    """vp (a 1800 -> 3300 m/s depth gradient and anomalies), eps, delta <= eps; depth is the last axis."""
    depth = torch.linspace(1800.0, 3300.0, shape[-1], device=DEV)
    vp = (depth + 150.0 * (2.0 * _smooth(shape, seed, 1) - 1.0)).contiguous()
    eps = (0.2 * _smooth(shape, seed, 2)).contiguous()
    dl = torch.minimum(0.1 * _smooth(shape, seed, 3), eps).contiguous()
    return vp, eps, dl


def _records(nrec_x, nrec_y, nt, dt, seed):
    """Reflection hyperbolas of a 20 Hz Ricker with a little noise, (nrec, nt) float32."""
    rng = np.random.default_rng(int(seed) * 7 + 5)
    x = (np.arange(nrec_x) - nrec_x / 2)[None, :] * 20.0
    y = (np.arange(nrec_y) - nrec_y / 2)[:, None] * 20.0
    off = np.sqrt(x * x + y * y).reshape(-1, 1)
    t = np.arange(nt)[None, :] * dt
    out = 1e-3 * rng.standard_normal((off.shape[0], nt))
    for _ in range(4):
        t0, v, a = rng.uniform(0.05, 0.9) * nt * dt, rng.uniform(1800, 3000), rng.uniform(-1, 1)
        s = (PI * 20.0 * (t - np.sqrt(t0 * t0 + (off / v) ** 2))) ** 2
        out += a * (1 - 2 * s) * np.exp(-s)
    return np.ascontiguousarray(out, dtype=np.float32)


def _ndim(c):
    return 3 if "ny" in c else 2


def _shape(c):
    return (c["ny"], c["nx"], c["nz"]) if _ndim(c) == 3 else (c["nx"], c["nz"])


def _geometry(c):
    """(mode, favg, dt_us, source cell, receiver depth) of a single-shot case."""
    if _ndim(c) == 3:
        return vti.MODE_GPU_REF, 15, 800, (c["nx"] // 2, c["ny"] // 2, 2), 3
    return (vti.MODE_CPU_REF if c.get("form") == "cpu" else vti.MODE_GPU_REF), 20, 1000, (c["nx"] // 2, 0, 4), 2


def _cfg_shot(c):
    mode, favg, dt_us, (sx, sy, sz), rz = _geometry(c)
    sv = c.get("sv", 1)
    if _ndim(c) == 3:
        cfg = vti.cfg_ref3d(c["nx"], c["ny"], c["nz"], 10, 10, 10, c["npml"], sv, favg, c["nt"], dt_us)
        return cfg, vti.shot_ref3d(cfg, 0, sx, 0, sy, 0, sz, 0, rec_depth=rz, rec_step=c.get("rec_step", 2))
    cfg = vti.cfg_ref2d(mode, c["nx"], c["nz"], 10, 10, c["npml"], sv, favg, c["nt"], dt_us)
    return cfg, vti.shot_ref2d(cfg, 1, sx, 0, sz, rec_depth=rz)


def _theta(c, seed):
    """Tilt in degrees, -25 .. 25."""
    return (50.0 * _smooth(_shape(c), seed, 4) - 25.0).contiguous()


def _propagator(c, seed):
    cfg, shot = _cfg_shot(c)
    vp, eps, dl = _model(_shape(c), seed)
    p = vti.Propagator(cfg)
    if DEV == "cuda":
        torch.cuda.synchronize()
    p.set_model(vp.data_ptr(), eps.data_ptr(), dl.data_ptr(), on_device=True)
    if c.get("form") == "tti":
        p.set_theta(_theta(c, seed).cpu().numpy(), degrees=True)
    if c["unsplit"]:
        p.set_unsplit(True)
    p.set_shot(shot)
    return p


def _batch_sizes(c):
    """Grid sizes of the batch's shots; the same for every seed."""
    r = random.Random(c["shots"] * 7919 + c["hi"])
    return [(r.randint(c["lo"], c["hi"]), r.randint(c["lo"] * 2 // 3, c["hi"] * 2 // 3), r.randint(10, 25))
            for _ in range(c["shots"])]


def _dct_basis():
    """The orthonormal 8 x 8 x 8 cosine basis, 512 x 512."""
    k = np.arange(8)
    d = np.cos(np.pi * (2 * k[:, None] + 1) * k[None, :] / 16) * np.where(k == 0, math.sqrt(1 / 8), math.sqrt(2 / 8))
    return np.einsum("ai,bj,ck->abcijk", d, d, d).reshape(512, 512).astype(np.float32)


def _snapshot(n, seed):
    """A wavefield snapshot: spherical Ricker wavefronts of several arrivals over a quiet background."""
    ax = torch.arange(n, device=DEV, dtype=torch.float32)
    out = torch.zeros((n, n, n), device=DEV)
    g = _gen(seed, 9)
    for _ in range(4):
        r = torch.rand(6, generator=g).tolist()
        d2 = ((ax - r[0] * n) ** 2).view(n, 1, 1) + ((ax - r[1] * n) ** 2).view(1, n, 1) + \
            ((ax - 0.3 * r[2] * n) ** 2).view(1, 1, n)
        d = torch.sqrt(d2 + 1.0)
        s = (math.pi * (d - (0.15 + 0.4 * r[3]) * n) / (8.0 + 8.0 * r[4])) ** 2
        out += (r[5] + 0.2) * 8.0 / (d + 8.0) * (1 - 2 * s) * torch.exp(-s)
    return out.contiguous()


def prepare(case, seed):
    c, f = dict(case), case["family"]
    if f == "fwd":
        return dict(c=c, p=_propagator(c, seed))
    if f == "rtm":
        p = _propagator(c, seed)
        s = p.shot
        o = p.rtm_defaults()
        o.image_every, o.nsnap = c["every"], c["nsnap"]
        st = dict(c=c, p=p, o=o, obs=_records(s.rec_nx, max(1, s.rec_ny), c["nt"], p.cfg.dt, seed))
        if c["how"] == "learned":
            st["ae"] = vti.Autoencoder(crop=16, batch=1, seed=1)
            st["ae"].set_basis(_dct_basis())
            lo = vti.learned_defaults()
            lo.codec, lo.tol, lo.save_every = 2, 7e-4, c["every"]
            lo.budget = 4 * (c["nt"] // c["every"] + 1) * c["nx"] * c["ny"] * c["nz"]
            st["lo"] = lo
        return st
    if f == "batch":
        cfgs, shots, models, obs = [], [], [], []
        for k, (nx, nz, favg) in enumerate(_batch_sizes(c)):
            cfg = vti.cfg_ref2d(vti.MODE_GPU_REF, nx, nz, 10, 10, 20, 1, favg, c["nt"], 1000)
            cfgs.append(cfg)
            shots.append(vti.shot_ref2d(cfg, 1, nx // 2, 0, 4, rec_depth=2))
            models.append([a.cpu().numpy() for a in _model((nx, nz), int(seed) + 31 * k)])
            obs.append(_records(nx, 1, c["nt"], cfg.dt, int(seed) + 31 * k))
        b = vti.Batch(cfgs, shots, models)
        b.set_unsplit(bool(c["unsplit"]))
        b.autotune(4)
        o = vti.rtm_defaults(2)
        o.nsnap = c["nsnap"]
        return dict(c=c, b=b, o=o, obs=obs)
    if f == "grad":
        cfg, shot = _cfg_shot(c)
        g = vti.Gradient(cfg, fp64=bool(c["fp64"]))
        vp, eps, dl = (a.cpu().numpy() for a in _model(_shape(c), seed))
        g.set_model(vp, eps, dl)
        g.set_shot(shot)
        return dict(c=c, g=g, dobs=_records(shot.rec_nx, max(1, shot.rec_ny), c["nt"], cfg.dt, seed))
    n = c["n"]
    ae = vti.Autoencoder(crop=16, batch=1, seed=1)
    ae.set_basis(_dct_basis())
    nb = (n // 8) ** 3
    return dict(c=c, ae=ae, x=_snapshot(n, seed),
                ent=torch.zeros(min(vti.Autoencoder.bq_max_words(n), n ** 3), dtype=torch.int32, device=DEV),
                boff=torch.zeros(nb, dtype=torch.int32, device=DEV),
                bcnt=torch.zeros(nb, dtype=torch.int16, device=DEV), y=torch.zeros((n, n, n), device=DEV))


def run(state):
    c, f = state["c"], state["c"]["family"]
    if f == "fwd":
        state["p"].run()
        return state["p"].record()
    if f == "rtm":
        p = state["p"]
        p.rtm_reset()
        if c["how"] == "plain":
            p.rtm_shot(state["o"], state["obs"])
        elif c["how"] == "eb":
            p.rtm_shot_eb(state["o"], state["obs"])
        else:
            p.rtm_shot_learned(state["ae"], state["o"], state["lo"], state["obs"])
        return p.rtm_image(finalize=False)
    if f == "batch":
        b = state["b"]
        b.rtm(state["o"], state["obs"])
        return [b.image(s) for s in range(b.n)]
    if f == "grad":
        r = state["g"].run(dobs=state["dobs"], nsnap=c["nsnap"])
        return {k: r[k] for k in ("misfit", "grad_vp", "grad_src", "d")}
    n, ae = c["n"], state["ae"]
    ent, boff, bcnt, y = state["ent"], state["boff"], state["bcnt"], state["y"]
    _, err = ae.bq_encode(state["x"].data_ptr(), 0, n * n, n, n, c["tol"], ent.data_ptr(), ent.numel(),
                             boff.data_ptr(), bcnt.data_ptr())
    ae.bq_decode(ent.data_ptr(), boff.data_ptr(), bcnt.data_ptr(), n, y.data_ptr())
    return {"ent": ent, "boff": boff, "bcnt": bcnt, "err": err, "field": y}


# ------------------------------------------------------------------- work ----
def work(case):
    """Each step reads the state (u, w, P, Q; v in 3D) and the model once and writes the state back once:
    the unsplit minimum in the interior; the split form adds its 4 (2D) or 6 (3D) fields both ways."""
    c, f = case, case["family"]
    if f == "codec":
        n3 = c["n"] ** 3
        return {"bytes": 4.0 * n3 * 2 + 2 * n3, "flops": 2.0 * 2 * 512 * n3}
    if f == "batch":
        cells = sum((nx + 32) * (nz + 32) for nx, nz, _ in _batch_sizes(c))
        nd, split, steps = 2, not c["unsplit"], 3 * c["nt"]
    else:
        nd = _ndim(c)
        cells = float(np.prod([n + 2 * c["npml"] - 8 for n in _shape(c)]))
        split = not c.get("unsplit", 0)
        steps = c["nt"] * (1 if f == "fwd" else 2 if c.get("how") in ("learned", "eb") else 3)
        if c.get("how") == "eb":
            steps += c["nt"]
    per = {2: (4 + 3 + 4), 3: (5 + 3 + 5)}[nd] * 4
    if split:
        per += {2: 4, 3: 6}[nd] * 2 * 4
    if f == "grad" and c["fp64"]:
        per *= 2
    return {"bytes": per * cells * steps, "flops": {2: 80.0, 3: 120.0}[nd] * cells * steps}


# ------------------------------------------------------------------ exact ----
class _Ref:
    """The staggered-grid VTI (or tilted) step in float64 on the padded grid, axes (y,) x, z."""

    def __init__(self, c, model, theta=None, favg=None, src=None, dt=None):
        self.nd = 3 if model[0].dim() == 3 else 2
        mode, fa, dt_us, s, rz = _geometry(c)
        self.cpu_form = mode == vti.MODE_CPU_REF
        favg = favg or fa
        src = src or s
        np_ = c["npml"]
        self.npml, self.nt, self.dh = np_, c["nt"], 10.0
        self.dt = float(np.float32(dt_us / 1e6))
        self.n = tuple(model[0].shape)
        self.nn = tuple(k + 2 * np_ for k in self.n)
        self.vp, self.ep, self.de = (self.pad(a.double()) for a in model)
        self.theta = None if theta is None else self.pad(theta.float().double() * (PI / 180.0))
        vp = self.vp
        if np_ == 0:
            d0 = 0.0
        elif self.cpu_form:
            d0 = 3.0 * float(vp.max()) * math.log(1e5) / (2.0 * np_ * self.dh)
        else:
            d0 = 10.0 * float(vp.reshape(-1)[vp.numel() // 2]) * math.log(1e5) / (2.0 * np_ * self.dh)
        self.tabs = [self.axis_table(k, d0 * self.dt) for k in self.n]
        R = self.R = tuple(slice(4, k - 4) for k in self.nn)
        self.co = [[t[j][4:-4].view([-1 if a == i else 1 for a in range(self.nd)]) for j in range(4)]
                   for i, t in enumerate(self.tabs)]
        # source and receivers, padded cells in axis order
        sx, sy, sz = src
        off = np_ - 1
        self.src = (sx + off, sz + off) if self.nd == 2 else (sy + off, sx + off, sz + off)
        cen = self.src if (self.nd == 3 or self.cpu_form) else (self.src[0] + 1, self.src[1] + 1)
        self.rec_z = rz + off
        step = c.get("rec_step", 2) if self.nd == 3 else 1
        self.rec = tuple(torch.arange(np_, np_ + k, step, device=DEV) for k in self.n[:-1])
        # wavelet: pfac = 10, active for two delays
        t = self.dt * np.arange(1, self.nt + 1)
        x = ((t - 1.0 / favg) * favg) ** 2
        self.amp = np.where(t <= 2.0 / favg, 10.0 * (1 - 2 * PI * PI * x) * np.exp(-PI * PI * x), 0.0)
        k = torch.arange(-3, 4, device=DEV, dtype=torch.float64) ** 2
        self.foot = torch.exp(-(k[:, None] + k[None, :]))
        # taper of eps and delta around the source
        r2 = sum(((torch.arange(m, device=DEV) - cen[i]) ** 2).view([-1 if a == i else 1 for a in range(self.nd)])
                 for i, m in enumerate(self.nn)).double()
        r0 = 15.0 / 4.0 if self.cpu_form else 4.0
        tap = 0.5 * (1 - torch.cos(PI * ((torch.sqrt(r2) - r0) * 4.0 / 44.0)))
        tap = torch.where(r2 <= (14 if self.cpu_form else 16), torch.zeros_like(tap), tap)
        self.tap = torch.where(r2 <= 225, tap, torch.ones_like(tap))
        del r2, tap

    def pad(self, a):
        np_ = self.npml
        return torch.nn.functional.pad(a[None, None], [np_] * (2 * self.nd), mode="replicate")[0, 0] if np_ else a

    def axis_table(self, n, h):
        np_ = self.npml
        i = np.arange(n + 2 * np_, dtype=np.float64)
        lo, hi = i < np_, i >= n + np_
        xv = np.where(lo, np_ - 0.5 - i, np.where(hi, 0.5 + i - n - np_, 0.0)) / max(np_, 1)
        xs = np.where(lo, np_ - i, np.where(hi, (1 if self.cpu_form else 0) + i - n - np_, 0.0)) / max(np_, 1)
        hv, hs = h * xv * xv, h * xs * xs
        c1, a1 = 1 / (1 + hv / 2), 1 / (1 + hs / 2)
        base = c1 if self.cpu_form else a1
        # interior cells: exactly one
        t = [c1, c1 * (1 - hv / 2), a1, base * (1 - hs / 2)]
        return [torch.tensor(np.where(lo | hi, v, 1.0), device=DEV) for v in t]

    def zero(self):
        z = lambda: torch.zeros(self.nn, device=DEV, dtype=torch.float64)  # noqa: E731
        return dict(v=[z() for _ in range(self.nd)], p=[z() for _ in range(self.nd)], q=[z() for _ in range(self.nd)],
                    P=z(), Q=z())

    def diff(self, f, axis, stress):
        """sum_m c_m (f[i+m+1] - f[i-m]) of the updated region (velocity), or (f[i+m] - f[i-m-1]) (stress)."""
        n = self.nn[axis]
        s = 0 if stress else 1
        out = None
        for m, cm in enumerate(C4):
            a, b = list(self.R), list(self.R)
            a[axis] = slice(4 + m + s, n - 4 + m + s)
            b[axis] = slice(4 - m - 1 + s, n - 4 - m - 1 + s)
            d = (f[tuple(a)] - f[tuple(b)]) * cm
            out = d if out is None else out + d
        return out

    def coef(self, sv, vp=None):
        """Per-axis products of the stress update: horizontal and vertical, p and q."""
        R, k = self.R, self.dt / self.dh
        ep, de = (self.ep * self.tap, self.de * self.tap) if sv else (self.ep, self.de)
        v2 = (self.vp if vp is None else vp)[R] ** 2 * k
        e2, sd = 1 + 2 * ep[R], torch.sqrt(1 + 2 * de[R])
        nd = self.nd
        return [v2 * e2] * (nd - 1) + [v2 * sd], [v2 * sd] * (nd - 1) + [v2]

    def step(self, s, co, amp=None):
        """One step in place; amp: the source gain of this step (None: no source)."""
        R, nd, k = self.R, self.nd, self.dt / self.dh
        P, Q = s["P"], s["Q"]
        point = amp is not None and not self.cpu_form and amp != 0.0
        if point:
            P[self.src] += amp
            Q[self.src] += amp
        if self.theta is not None:
            cs, sn = torch.cos(self.theta)[R], torch.sin(self.theta)[R]
            cx, cz = self.co
            g2, g1 = cx[1] * cz[1], cx[0] * cz[0]
            Px, Pz, Qx, Qz = self.diff(P, 0, 0), self.diff(P, 1, 0), self.diff(Q, 0, 0), self.diff(Q, 1, 0)
            s["v"][0][R] = g2 * s["v"][0][R] - g1 * k * (cs * Px - sn * Pz)
            s["v"][1][R] = g2 * s["v"][1][R] - g1 * k * (sn * Qx + cs * Qz)
            u, w = s["v"]
            dx = cs * self.diff(u, 0, 1) - sn * self.diff(u, 1, 1)
            dz = sn * self.diff(w, 0, 1) + cs * self.diff(w, 1, 1)
            a2, a1 = cx[3] * cz[3], cx[2] * cz[2]
            for f, kk in ((s["p"], co[0]), (s["q"], co[1])):
                f[0][R] = a2 * f[0][R] - a1 * kk[0] * dx
                f[1][R] = a2 * f[1][R] - a1 * kk[1] * dz
        else:
            for a in range(nd):
                d = self.diff(Q if a == nd - 1 else P, a, 0)
                s["v"][a][R] = self.co[a][1] * s["v"][a][R] - self.co[a][0] * k * d
            for a in range(nd):
                d = self.diff(s["v"][a], a, 1)
                for f, kk in ((s["p"], co[0]), (s["q"], co[1])):
                    f[a][R] = self.co[a][3] * f[a][R] - self.co[a][2] * kk[a] * d
        if point:   # outside the updated region nothing changes; inside, the stress update rebuilds P and Q
            P[self.src] -= amp
            Q[self.src] -= amp
        P[R] = sum(f[R] for f in s["p"])
        Q[R] = sum(f[R] for f in s["q"])
        if amp is not None and self.cpu_form and amp != 0.0:
            x, z = self.src
            P[x - 3:x + 4, z - 3:z + 4] += amp * self.foot
            Q[x - 3:x + 4, z - 3:z + 4] += amp * self.foot

    def at_rec(self, f):
        if self.nd == 2:
            return f[self.rec[0], self.rec_z]
        return f[self.rec[0][:, None], self.rec[1][None, :], self.rec_z].reshape(-1)

    def interior(self, f):
        return f[tuple(slice(self.npml, k - self.npml) for k in self.nn)]

    def forward(self, sv, each=None):
        s, co = self.zero(), self.coef(sv)
        rec = torch.zeros((self.at_rec(s["P"]).numel(), self.nt), device=DEV, dtype=torch.float64)
        for it in range(self.nt):
            self.step(s, co, float(self.amp[it]))
            r = self.at_rec(s["P"])
            rec[:, it] = r + r if self.cpu_form else r
            if each:
                each(it, s)
        return rec

    def rtm(self, sv, obs, every, both):
        """(image, illumination): both: source + receiver energy, else source energy clamped to 1 while <= 0."""
        snaps, ill = [], torch.zeros(self.n, device=DEV, dtype=torch.float64)

        def each(it, s):
            e = self.interior(s["P"]) ** 2 + self.interior(s["Q"]) ** 2
            ill.add_(e)
            if not both:
                ill[ill <= 0.0] = 1.0
            snaps.append(self.interior(s["P"]).clone() if it % every == 0 else None)

        self.forward(sv, each)
        img = torch.zeros_like(ill)
        g, co = self.zero(), self.coef(False)
        obs = torch.tensor(obs, device=DEV, dtype=torch.float64)
        for it in range(self.nt - 1, -1, -1):
            row = obs[:, it]
            for f in (g["P"], g["Q"]):
                if self.nd == 2:
                    f[self.rec[0], self.rec_z] = row
                else:
                    f[self.rec[0][:, None], self.rec[1][None, :], self.rec_z] = row.view(self.rec[0].numel(), -1)
            self.step(g, co, None)
            if both:
                ill.add_(self.interior(g["P"]) ** 2 + self.interior(g["Q"]) ** 2)
            if it % every == 0:
                img.add_(snaps[it] * self.interior(g["P"]))
        return img, ill

    def flat(self, s):
        return s["v"] + s["p"] + s["q"] + [s["P"], s["Q"]]

    def step_pure(self, t, vpu, amp, sv):
        """The point-source step as a function of the state list, the unpadded vp and the source gain."""
        nd, R, k = self.nd, self.R, self.dt / self.dh
        v, p, q, P, Q = t[:nd], t[nd:2 * nd], t[2 * nd:3 * nd], t[-2], t[-1]
        co = self.coef(sv, self.pad(vpu))
        d = torch.zeros_like(P)
        d[self.src] = 1.0
        P, Q = P + amp * d, Q + amp * d

        def put(f, val):
            out = f.clone()
            out[R] = val
            return out

        v = [put(v[a], self.co[a][1] * v[a][R] - self.co[a][0] * k * self.diff(Q if a == nd - 1 else P, a, 0))
             for a in range(nd)]
        dv = [self.diff(v[a], a, 1) for a in range(nd)]
        p = [put(p[a], self.co[a][3] * p[a][R] - self.co[a][2] * co[0][a] * dv[a]) for a in range(nd)]
        q = [put(q[a], self.co[a][3] * q[a][R] - self.co[a][2] * co[1][a] * dv[a]) for a in range(nd)]
        P, Q = put(P, sum(f[R] for f in p)), put(Q, sum(f[R] for f in q))
        return v + p + q + [P, Q], self.at_rec(P)

    def gradient(self, vpu, sv, dobs):
        t = self.flat(self.zero())
        states, rec = [], []
        with torch.no_grad():
            for it in range(self.nt):
                states.append(t)
                t, r = self.step_pure(t, vpu, float(self.amp[it]), sv)
                rec.append(r)
        d = torch.stack(rec, 1)
        res = d - torch.tensor(dobs, device=DEV, dtype=torch.float64)
        bar = [torch.zeros_like(a) for a in t]
        gv, gs = torch.zeros_like(vpu), torch.zeros(self.nt, device=DEV, dtype=torch.float64)
        for it in range(self.nt - 1, -1, -1):
            x = [a.detach().requires_grad_(True) for a in states[it]]
            m = vpu.detach().requires_grad_(True)
            amp = torch.tensor(float(self.amp[it]), device=DEV, dtype=torch.float64, requires_grad=True)
            y, r = self.step_pure(x, m, amp, sv)
            got = torch.autograd.grad(y + [r], x + [m, amp], bar + [res[:, it]], allow_unused=True)
            bar = [torch.zeros_like(a) if b is None else b for a, b in zip(x, got)]
            gv += got[-2]
            gs[it] = got[-1]
            states[it] = None
        return {"misfit": float(0.5 * (res ** 2).sum()), "grad_vp": gv, "grad_src": gs, "d": d}


def exact(case, seed):
    c, f = case, case["family"]
    if f == "codec" or c.get("how") == "learned":
        return None         # what the codec keeps depends on its quantization, not on the input alone
    if f == "batch":
        out = []
        for k, (nx, nz, favg) in enumerate(_batch_sizes(c)):
            k1 = dict(nx=nx, nz=nz, npml=20, nt=c["nt"])
            ref = _Ref(k1, _model((nx, nz), int(seed) + 31 * k), favg=favg)
            out.append(ref.rtm(True, _records(nx, 1, c["nt"], float(np.float32(1e-3)), int(seed) + 31 * k), 1, False))
        return out
    model = _model(_shape(c), seed)
    ref = _Ref(c, model, _theta(c, seed) if c.get("form") == "tti" else None)
    if f == "fwd":
        return ref.forward(bool(c["sv"]))
    dt = float(np.float32(_geometry(c)[2] / 1e6))
    ny = ref.rec[0].numel() if ref.nd == 3 else 1
    obs = _records(ref.rec[-1].numel(), ny, c["nt"], dt, seed)
    if f == "rtm":
        return ref.rtm(True, obs, c["every"], ref.nd == 3)
    return ref.gradient(model[0].double(), True, obs)
