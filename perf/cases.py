"""Workloads of the MHD step as programs run it, for timing and comparison.

listed() names them, draw(rng) gives one more of the same ranges, prepare()
makes what a program holds before the call (a box with its state uploaded, an
ensemble, a network with its samples), run() is one pass through the public
entry points and work() what that pass cannot do without.  exact() evaluates
the same pass in 64 bits with plain torch operations.

Kinds of a pass:
  step      n steps of one resident box, then the state back in the caller's
            own arrays, as a driver does between two dumps.  calls "each":
            one mhd_step per step (the Fortran drop-in); "batch": mhd_steps.
  noalloc   one mhd_step_noalloc on arrays that stay on the device.
  ensemble  n graph-replayed steps of many uneven boxes, then all states back.
  closure   n closure-corrected steps of a coarse mixed box, then its state.
  train     n Adam iterations of the closure network on resident samples.
  sample    the closure's training data of one snapshot: box-filtered state
            and right-hand side, and the horizontal-mean flux profiles.
"""

import ctypes as C
import importlib
import math

import numpy as np
import torch

DEV = "cuda" if torch.cuda.is_available() else "cpu"
FIELDS = ("ru", "rv", "rw", "ro", "tt", "bx", "by", "bz")


def _pkg():
    return importlib.import_module("rast-3dmhd_amd")


# --------------------------------------------------------------------------
# cases

def listed():
    return [
        # the smallest call: a 16x16x12 box (the size of the reference's own
        # check runs) stepped by one STEP call per step, state read at a dump
        dict(name="step_calls_16x16x12", kind="step", nx=16, ny=16, nz=12, steps=20, calls="each", precision="fp64",
             mag=True, rot=True, ident=0, contrast=3.0, ra=1e4),
        # a program that keeps its arrays on the device and may not allocate
        dict(name="noalloc_64x64x32", kind="noalloc", nx=64, ny=64, nz=32, mag=True, rot=True, contrast=10.0, ra=1e5),
        # the reference CPU configuration's box and number of steps
        dict(name="fp64_64x64x32", kind="step", nx=64, ny=64, nz=32, steps=200, calls="batch", precision="fp64",
             mag=True, rot=True, ident=0, contrast=10.0, ra=1e5),
        # hydrodynamic box of odd sizes that fill neither tiles nor z chunks
        dict(name="fp64_hydro_130x90x41", kind="step", nx=130, ny=90, nz=41, steps=100, calls="batch",
             precision="fp64", mag=False, rot=False, ident=0, contrast=10.0, ra=1e5),
        # optional branch of FLUXES: diffusion of the density perturbations,
        # whose plane means follow the reference's summation order
        dict(name="fp64_density_diffusion_96x96x48", kind="step", nx=96, ny=96, nz=48, steps=20, calls="batch",
             precision="fp64", mag=True, rot=True, ident=1, contrast=10.0, ra=1e5),
        # the accuracy configuration in both forms
        dict(name="fp64_256x256x128", kind="step", nx=256, ny=256, nz=128, steps=100, calls="batch",
             precision="fp64", mag=True, rot=True, ident=0, contrast=10.0, ra=1e5),
        dict(name="mixed_256x256x128", kind="step", nx=256, ny=256, nz=128, steps=200, calls="batch",
             precision="mixed", mag=True, rot=True, ident=0, contrast=10.0, ra=1e5),
        # the bandwidth-bound headline box
        dict(name="mixed_512x512x256", kind="step", nx=512, ny=512, nz=256, steps=100, calls="batch",
             precision="mixed", mag=True, rot=True, ident=0, contrast=30.0, ra=1e6),
        # 64 uneven boxes with their own parameters and dt
        dict(name="ensemble_64_mixed", kind="ensemble", boxes=64, steps=50, precision="mixed", lo=32, hi=96, zlo=32,
             zhi=64, boxseed=4242),
        # the closure-corrected coarse run
        dict(name="closure_128x128x64", kind="closure", nx=128, ny=128, nz=64, steps=50, contrast=10.0, ra=1e5),
        # training of its network
        dict(name="train_64x64x64", kind="train", nx=64, ny=64, nz=64, samples=3, iters=6),
        # the training data of one fine snapshot, filtered by 4
        dict(name="sample_256x256x125", kind="sample", nx=256, ny=256, nz=125, factor=4, contrast=10.0, ra=1e5),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "step", "noalloc", "ensemble", "closure", "train", "sample"])
    if kind == "step":
        n = _log_int(rng, 16, 300)
        nx, ny = max(8, int(n * rng.uniform(0.6, 1.5))), max(8, int(n * rng.uniform(0.6, 1.5)))
        nz = max(8, int(n * rng.uniform(0.4, 0.8)))
        precision = rng.choice(["fp64", "mixed"])
        ident = 1 if precision == "fp64" and nx * ny < 30000 and rng.random() < 0.25 else 0
        zones = nx * ny * nz
        steps = max(10, min(200, int(4e8 / zones)))
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, steps=steps, calls=rng.choice(["each", "batch"]),
                    precision=precision, mag=rng.random() < 0.7, rot=rng.random() < 0.7, ident=ident,
                    contrast=round(rng.uniform(3.0, 12.0), 3), ra=1e4 if n < 48 else 1e5)
    if kind == "noalloc":
        nx, ny, nz = _log_int(rng, 12, 66), _log_int(rng, 12, 66), _log_int(rng, 8, 34)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, mag=rng.random() < 0.7, rot=rng.random() < 0.7,
                    contrast=round(rng.uniform(3.0, 12.0), 3), ra=1e4)
    if kind == "ensemble":
        return dict(kind=kind, boxes=rng.randrange(4, 48), steps=rng.randrange(10, 50),
                    precision=rng.choice(["mixed", "mixed", "fp64"]), lo=24, hi=rng.choice([64, 96, 120]), zlo=24,
                    zhi=64, boxseed=rng.randrange(1, 10000))
    if kind == "closure":
        return dict(kind=kind, nx=_log_int(rng, 24, 160), ny=_log_int(rng, 24, 160), nz=_log_int(rng, 16, 72),
                    steps=rng.randrange(20, 60), contrast=10.0, ra=1e5)
    if kind == "train":
        return dict(kind=kind, nx=_log_int(rng, 16, 96), ny=_log_int(rng, 16, 72), nz=_log_int(rng, 12, 64),
                    samples=rng.randrange(1, 4), iters=rng.randrange(3, 7))
    f = rng.choice([2, 4])
    return dict(kind=kind, nx=f * _log_int(rng, 12, 72), ny=f * _log_int(rng, 12, 72),
                nz=f * _log_int(rng, 6, 36) + 1, factor=f, contrast=10.0, ra=1e5)


# --------------------------------------------------------------------------
# inputs

def _meta(nx, ny, nz, contrast, ra, mag=True, rot=True, tilt=0.0, pm=1.0, ta=1e4, ident=0):
    """The COMMON scalars and metric arrays a driver computes at set-up, and
    the polytrope's columns."""
    cfg = importlib.import_module("rast-3dmhd_amd.config")
    ph = cfg.physics(contrast=contrast, ra=ra, pr=1.0, pm=pm, ta=ta, tilt_deg=tilt)
    par = {k: cfg.f32(v) for k, v in ph.items()}
    mt = cfg.metrics(nx, ny, nz, xmax=par[17], ymax=par[18], zmax=par[19], ngrid=3)
    t, r = cfg.polytrope(mt["zee"], par[3], par[4])
    m = cfg.constants(nx, ny, nz, par, lmag=mag, lrot=rot, izcon=1, itcon=0, tb=float(t[-1]))
    m.update(mt)
    if ident:
        m.update(id=ident, dh=0.5, dv=0.5)
    return m, t, r


def _modes(nx, ny, nz, gen, odd, count=6):
    """[nz][ny][nx]: random horizontal modes |k| <= 4 times cos (odd: sin) of
    pi m zeta, scaled to an RMS of 1."""
    f = dict(dtype=torch.float64, device=DEV)
    k = torch.randint(-4, 5, (2, count), generator=gen).to(**f)
    k[0, :] = torch.where((k[0] == 0) & (k[1] == 0), torch.ones_like(k[0]), k[0])
    ph = torch.rand(count, generator=gen).to(**f) * (2.0 * math.pi)
    amp = (torch.rand(count, generator=gen) + 0.5).to(**f)
    mz = torch.randint(1, 4, (count,), generator=gen).to(**f)
    x = torch.arange(nx, **f) * (2.0 * math.pi / nx)
    y = torch.arange(ny, **f) * (2.0 * math.pi / ny)
    z = torch.arange(nz, **f) * (math.pi / (nz - 1))
    h = torch.cos(k[0][:, None, None] * x + k[1][:, None, None] * y[:, None] + ph[:, None, None])
    zz = mz[:, None] * z
    v = (amp[:, None] * (torch.sin(zz) if odd else torch.cos(zz))).T @ h.reshape(count, -1)
    v = v.reshape(nz, ny, nx)
    return v / v.square().mean().sqrt()


def _state(meta, t, r, seed, mag, mach=0.05, tamp=0.02, bamp=1e-3):
    """Device tensors [nz+2][ny][nx] of a stratified layer with a moderate
    flow and a weak field; ghost planes carry the profile alone."""
    nx, ny, nz = int(meta["npx"]), int(meta["npy"]), int(meta["npz"])
    gen = torch.Generator().manual_seed(int(seed))
    f = dict(dtype=torch.float64, device=DEV)
    col = lambda a: torch.as_tensor(np.asarray(a), **f)[:, None, None]  # noqa: E731
    full = lambda a: a.expand(nz + 2, ny, nx).clone()  # noqa: E731
    q = {"tt": full(col(t)), "ro": full(col(r))}
    q["tt"][1:-1] *= 1.0 + tamp * _modes(nx, ny, nz, gen, True)
    q["ro"][1:-1] *= 1.0 + 0.5 * tamp * _modes(nx, ny, nz, gen, True)
    for c in ("u", "v", "w"):
        a = torch.zeros(nz + 2, ny, nx, **f)
        a[1:-1] = mach * q["ro"][1:-1] * _modes(nx, ny, nz, gen, c == "w")
        if c == "w":
            a[1] = 0.0
            a[nz] = 0.0
        q["r" + c] = a
    for c in ("bx", "by", "bz"):
        a = torch.zeros(nz + 2, ny, nx, **f)
        if mag:
            a[1:-1] = bamp * _modes(nx, ny, nz, gen, c == "bz")
            if c == "bz":
                a[1] = 0.0
                a[nz] = 0.0
        q[c] = a
    return q


def _wrap(a):
    """Periodic x/y ghosts: [K][ny][nx] -> [K][ny+2][nx+2] (the Fortran
    array (nx+2, ny+2, K) in its own byte order)."""
    a = torch.cat([a[:, -1:], a, a[:, :1]], dim=1)
    return torch.cat([a[:, :, -1:], a, a[:, :, :1]], dim=2).contiguous()


def _fields(q, mag):
    """Padded Fortran-order host arrays for an upload."""
    return {k: _wrap(q[k]).cpu().numpy().T for k in (FIELDS if mag else FIELDS[:5])}


def _case_state(case, seed):
    mag = bool(case.get("mag", True))
    meta, t, r = _meta(case["nx"], case["ny"], case["nz"], case["contrast"], case["ra"], mag,
                       bool(case.get("rot", True)), tilt=45.0 if case["contrast"] >= 30.0 else 0.0,
                       pm=2.0 if case["contrast"] >= 30.0 else 1.0, ta=1e6 if case["contrast"] >= 30.0 else 1e4,
                       ident=int(case.get("ident", 0)))
    return meta, _state(meta, t, r, seed, mag), mag


def _specs(case):
    """Boxes of an ensemble: horizontal sizes multiples of 8, the rest uniform
    or log-uniform."""
    rng = np.random.default_rng(case["boxseed"])
    out = []
    for _ in range(case["boxes"]):
        out.append(dict(nx=int(rng.choice(np.arange(case["lo"], case["hi"] + 1, 8))),
                        ny=int(rng.choice(np.arange(case["lo"], case["hi"] + 1, 8))),
                        nz=int(rng.integers(case["zlo"], case["zhi"] + 1)), ra=float(10 ** rng.uniform(4, 5)),
                        ta=float(10 ** rng.uniform(2, 6)), contrast=float(rng.uniform(3, 30))))
    return out


def _ens_states(case, seed):
    for b, s in enumerate(_specs(case)):
        meta, t, r = _meta(s["nx"], s["ny"], s["nz"], s["contrast"], s["ra"], ta=s["ta"])
        yield meta, _state(meta, t, r, 1000 * int(seed) + b, True, mach=0.02, tamp=0.01, bamp=1e-4)


def _net_params(seed):
    g = np.random.default_rng(int(seed) + 99)
    v = []
    for ci, co in ((8, 32), (32, 32), (32, 7)):
        v += [g.standard_normal(co * 27 * ci) * math.sqrt(2.0 / (27 * ci)), np.zeros(co)]
    return np.concatenate(v).astype(np.float32)


def _closure_norm(meta, t, r):
    """Normalisation of the network's inputs and outputs: profiles and
    standard deviations per channel."""
    nz, g = int(meta["npz"]), float(meta["gamma"])
    pin, pout = np.zeros((8, nz)), np.zeros((7, nz))
    pin[0] = r[1:-1]
    pin[4] = np.log(t[1:-1]) / (g - 1.0) - np.log(r[1:-1])
    pout[2] = 1e-4 * np.sin(np.linspace(0.0, math.pi, nz))
    ins = np.array([0.1, 0.05, 0.05, 0.05, 0.05, 1e-3, 1e-3, 1e-3])
    outs = np.array([1e-3, 1e-3, 1e-3, 1e-3, 1e-5, 1e-5, 1e-5])
    return pin, ins, pout, outs


def _samples(case, seed):
    """(inputs, targets) of the network, float32 [nz][ny][nx][8 and 7]."""
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    sh = (case["nz"], case["ny"], case["nx"])
    for _ in range(case["samples"]):
        x = torch.randn(*sh, 8, generator=g, device=DEV)
        t = 0.5 * torch.roll(x, 1, 2)[..., :7] + 0.5 * torch.randn(*sh, 7, generator=g, device=DEV)
        t[0] = 0.0
        t[-1] = 0.0
        yield x, t


class _Kept:
    """A handle that is given back with the state that holds it."""

    def __init__(self, **kw):
        self.__dict__.update(kw)

    def __del__(self):
        for k in ("box", "ens", "net"):
            h = self.__dict__.get(k)
            if h is not None:
                h.close()


_P = C.POINTER(C.c_double)


def _ptr(a):
    return a.ctypes.data_as(_P)


def prepare(case, seed):
    pkg = _pkg()
    kind = case["kind"]
    if kind == "ensemble":
        metas, q = zip(*_ens_states(case, seed))
        ens = pkg.Ensemble(list(metas), precision=case["precision"])
        offs, total = [], 0
        for b, (m, s) in enumerate(zip(metas, q)):
            ens.upload(b, _fields(s, True))
            offs.append(total)
            total += (int(m["npx"]) + 2) * (int(m["npy"]) + 2) * (int(m["npz"]) + 2)
        return _Kept(ens=ens, lib=pkg.load(), steps=case["steps"], offs=offs, out=[np.ones(total) for _ in FIELDS],
                     kind=kind)
    if kind == "train":
        net = pkg.Net(8, 32, 7)
        net.set_params(_net_params(seed))
        for x, t in _samples(case, seed):
            net.add_sample(x.cpu().numpy(), t.cpu().numpy())
        return _Kept(net=net, iters=case["iters"], kind=kind)
    if kind == "noalloc":
        meta, q, mag = _case_state(case, seed)
        d = pkg.make_desc(meta)
        met = [torch.from_numpy(a.copy()).to(DEV) for a in pkg.metric_arrays(meta, d)]
        fs = [_wrap(q[k]) for k in (FIELDS if mag else FIELDS[:5])]
        ptrs = (C.c_void_p * 8)(*([a.data_ptr() for a in fs] + [None] * (8 - len(fs))))
        return _Kept(lib=pkg.load(), desc=d, met=met, dmet=pkg.MhdDevMetrics(*[a.data_ptr() for a in met]), fs=fs,
                     ptrs=ptrs, nit=C.c_int(0), timc=C.c_double(0.0), timt=C.c_double(0.0), dt=C.c_double(),
                     um=C.c_double(), kind=kind)
    meta, q, mag = _case_state(case, seed)
    box = pkg.Box(meta, precision=case.get("precision", "mixed" if kind == "closure" else "fp64"))
    host = _fields(q, mag)
    box.upload(host)
    s = _Kept(box=box, lib=pkg.load(), kind=kind, names=FIELDS if mag else FIELDS[:5])
    if kind == "sample":
        s.factor = case["factor"]
        return s
    s.steps, s.calls = case["steps"], case.get("calls", "batch")
    # the driver's own arrays (COMMON /BIG/), written by every download
    s.out = [host[k].T for k in s.names]
    if kind == "closure":
        _, t, r = _meta(case["nx"], case["ny"], case["nz"], case["contrast"], case["ra"])
        s.net = pkg.Net(8, 32, 7)
        s.net.set_params(_net_params(seed))
        box.set_closure(s.net, *_closure_norm(meta, t, r), 0.0, 0.1)
    return s


# --------------------------------------------------------------------------
# one pass

def run(s):
    if s.kind == "noalloc":
        rc = s.lib.mhd_step_noalloc(C.byref(s.desc), C.byref(s.dmet), s.ptrs, C.byref(s.nit), C.byref(s.timc),
                                    C.byref(s.timt), 0.0, C.byref(s.dt), C.byref(s.um),
                                    C.c_void_p(torch.cuda.current_stream().cuda_stream))
        if rc:
            raise RuntimeError(s.lib.mhd_last_error(None).decode())
        return {"dt": s.dt.value, "umach": s.um.value, "state": s.fs}
    if s.kind == "train":
        first, last = s.net.train(s.iters, 2e-3)
        return {"loss": [first, last], "params": s.net.params()}
    if s.kind == "ensemble":
        dt, um = s.ens.steps(s.steps)
        for b, o in enumerate(s.offs):
            rc = s.lib.mhd_ens_download(s.ens.h, b, *[_ptr(a[o:]) for a in s.out])
            if rc:
                raise RuntimeError(s.lib.mhd_ens_last_error(s.ens.h).decode())
        return {"dt": dt, "umach": um, "state": s.out}
    if s.kind == "sample":
        return {"state": s.box.box_filter(s.factor, 1, "state"), "rhs": s.box.box_filter(s.factor, 1, "rhs"),
                "profiles": s.box.flux_profiles()}
    if s.calls == "each":
        for _ in range(s.steps):
            dt, um = s.box.step()
    else:
        dt, um = s.box.steps(s.steps)
    rc = s.lib.mhd_download(s.box.h, *([_ptr(a) for a in s.out] + [None] * (8 - len(s.out))))
    if rc:
        raise RuntimeError(s.lib.mhd_last_error(s.box.h).decode())
    return {"dt": dt, "umach": um, "state": s.out}


def work(case):
    """Per step: the state read once and written once (mixed: 6 bytes a value,
    4 stored and 2 of residual) and the floating-point operations of three
    right-hand sides and updates; a download writes the state once more."""
    def step(zones, mag, mixed, n):
        nf = 8 if mag else 5
        return dict(bytes=zones * nf * (n * 2 * (6 if mixed else 8) + 8), flops=zones * n * 3 * (590 if mag else 330))

    def add(a, b):
        return {k: a[k] + b[k] for k in a}

    kind = case["kind"]
    net = 2.0 * 27 * (8 * 32 + 32 * 32 + 32 * 7)  # multiply-adds of one voxel's forward pass
    if kind == "ensemble":
        tot = dict(bytes=0, flops=0)
        for s in _specs(case):
            tot = add(tot, step(s["nx"] * s["ny"] * s["nz"], True, case["precision"] == "mixed", case["steps"]))
        return tot
    zones = case["nx"] * case["ny"] * case["nz"]
    if kind == "train":
        # inputs, targets and the two hidden activations; forward, input and weight gradients
        return dict(bytes=case["iters"] * zones * (8 * 2 + 8 * 4 + 2 * 2 * 64), flops=case["iters"] * zones * 3 * net)
    if kind == "sample":
        return dict(bytes=zones * 8 * 8 + zones // case["factor"] ** 3 * 16 * 8, flops=zones * (590 + 40))
    if kind == "noalloc":
        return dict(bytes=zones * (8 if case["mag"] else 5) * 16, flops=zones * 3 * (590 if case["mag"] else 330))
    if kind == "closure":
        w = step(zones, True, True, case["steps"])
        return add(w, dict(bytes=zones * case["steps"] * 28, flops=zones * case["steps"] * net))
    return step(zones, case["mag"], case["precision"] == "mixed", case["steps"])


# --------------------------------------------------------------------------
# the same passes in 64 bits, plain torch

class _Step:
    """One box of the compressible-MHD step on tensors [nz+2][ny][nx]."""

    def __init__(self, meta, q, ghost_flip):
        f = dict(dtype=torch.float64, device=DEV)
        self.m, self.q, self.flip = meta, {k: v.clone() for k, v in q.items()}, ghost_flip
        self.nz, self.mag, self.rot = int(meta["npz"]), bool(int(meta["lmag"])), bool(int(meta["lrot"]))
        a = lambda k: torch.as_tensor(np.asarray(meta[k]), **f)[1:-1]  # noqa: E731
        self.dx, self.d2x, self.ddx_ = (a(k)[None, None, :] for k in ("dxxdx", "d2xxdx2", "ddx"))
        self.dy, self.d2y, self.ddy_ = (a(k)[None, :, None] for k in ("dyydy", "d2yydy2", "ddy"))
        self.dz, self.d2z, self.ddz_ = (a(k)[:, None, None] for k in ("dzzdz", "d2zzdz2", "ddz"))
        self.rk, self.dk = a("rkapa")[:, None, None], a("dkapa")[:, None, None]
        self.names = FIELDS if self.mag else FIELDS[:5]

    def gx(self, f):
        return (torch.roll(f, -1, 2) - torch.roll(f, 1, 2)) * (self.m["hx"] * self.dx)

    def gy(self, f):
        return (torch.roll(f, -1, 1) - torch.roll(f, 1, 1)) * (self.m["hy"] * self.dy)

    def gz(self, f):
        return (f[2:] - f[:-2]) * (self.m["hz"] * self.dz)

    def lx(self, f):
        p, n = torch.roll(f, -1, 2), torch.roll(f, 1, 2)
        return (p - n) * (self.m["hx"] * self.d2x) + (p - 2.0 * f + n) * (self.m["h2x"] * self.dx * self.dx)

    def ly(self, f):
        p, n = torch.roll(f, -1, 1), torch.roll(f, 1, 1)
        return (p - n) * (self.m["hy"] * self.d2y) + (p - 2.0 * f + n) * (self.m["h2y"] * self.dy * self.dy)

    def lz(self, f):
        return ((f[2:] - f[:-2]) * (self.m["hz"] * self.d2z)
                + (f[2:] - 2.0 * f[1:-1] + f[:-2]) * (self.m["h2z"] * self.dz * self.dz))

    def lz_sided(self, f):
        """lz with one-sided forms on the two boundary planes."""
        o, (a, b) = self.lz(f), (self.m["hz"] * self.d2z, self.m["h2z"] * self.dz * self.dz)
        o[0] = (-3.0 * f[1] + 4.0 * f[2] - f[3]) * a[0] + (2.0 * f[1] - 5.0 * f[2] + 4.0 * f[3] - f[4]) * b[0]
        o[-1] = ((3.0 * f[-2] - 4.0 * f[-3] + f[-4]) * a[-1]
                 + (2.0 * f[-2] - 5.0 * f[-3] + 4.0 * f[-4] - f[-5]) * b[-1])
        return o

    def gz_sided(self, f):
        """gz of a quantity that vanishes on the two boundary planes."""
        o, a = self.gz(f), self.m["hz"] * self.dz
        o[0] = (4.0 * f[2] - f[3]) * a[0]
        o[-1] = (f[-4] - 4.0 * f[-3]) * a[-1]
        return o

    def rhs(self, q):
        m = self.m
        ident = int(m.get("id", 0))
        ore, ocv, c43 = m["ore"], m["ocv"], m["c43"]
        tcr, tv, tc = m["c13"] * ore, ocv * ore, ocv / m["repr"]
        i = slice(1, -1)
        ru, rv, rw, ro, tt = (q[k] for k in FIELDS[:5])
        if ident:
            ro = ro.clone()
            ro[0], ro[-1] = ro[2], ro[-3]
        u, v, w, p = ru / ro, rv / ro, rw / ro, ro * tt
        ri, t0 = 1.0 / ro[i], tt[i]
        F = {"ro": -self.gx(ru[i]) - self.gy(rv[i]) - self.gz_sided(rw)}
        if ident:
            rom = ro.mean(dim=(1, 2), keepdim=True)
            d = ro - rom
            F["ro"] += (m["dh"] * (self.lx(d[i]) + self.ly(d[i])) + m["dv"] * self.lz(d)) * (ore / rom[i])

        def adv(a):
            return self.gx((a * u)[i]) + self.gy((a * v)[i]) + self.gz(a * w)

        dxu, dxv, dxw = (self.gx(a[i]) for a in (u, v, w))
        dyu, dyv, dyw = (self.gy(a[i]) for a in (u, v, w))
        dzu, dzv, dzw = (self.gz(a) for a in (u, v, w))
        fu = -self.gx(p[i]) - adv(ru) + ore * (c43 * self.lx(u[i]) + self.ly(u[i]) + self.lz(u))
        fu += tcr * (self.gy(dxv) + self.gx(dzw))
        fv = -self.gy(p[i]) - adv(rv) + ore * (self.lx(v[i]) + c43 * self.ly(v[i]) + self.lz(v))
        fv += tcr * (self.gy(dxu) + self.gy(dzw))
        fw = m["grav"] * ro[i] - self.gz(p) - adv(rw) + ore * (self.lx(w[i]) + self.ly(w[i]) + c43 * self.lz(w))
        fw += tcr * (self.gx(dzu) + self.gy(dzv))
        gzt = self.gz(tt)
        ft = -(u[i] * self.gx(t0) + v[i] * self.gy(t0) + w[i] * gzt)
        ft += tc * ri * (self.rk * (self.lx(t0) + self.ly(t0) + self.lz(tt)) + self.dk * gzt)
        ft += tv * ri * (c43 * (dxu * dxu + dyv * dyv + dzw * dzw - dxu * dzw - dxu * dyv - dyv * dzw)
                         + dxv * dxv + dxw * dxw + dyu * dyu + dzu * dzu + dzv * dzv + dyw * dyw
                         + 2.0 * (dyu * dxv + dzv * dyw + dzu * dxw))
        ft -= ocv * (dxu + dyv + dzw) * t0
        if self.rot:
            fu += m["omz"] * rv[i]
            fv += m["omx"] * rw[i] - m["omz"] * ru[i]
            fw -= m["omx"] * rv[i]
        if self.mag:
            ob, orm = m["obeta"], m["orm"]
            B = [q[k] for k in ("bx", "by", "bz")]
            bx, by, bz = (b[i] for b in B)
            dzw1 = self.gz_sided(w)
            gxb, gyb = [self.gx(b[i]) for b in B], [self.gy(b[i]) for b in B]
            gzb = [self.gz(b) for b in B]
            advb = [u[i] * gxb[c] + v[i] * gyb[c] + w[i] * gzb[c] for c in range(3)]
            jz, jx = gyb[0] - gxb[1], gzb[1] - gyb[2]
            F["bx"] = by * dyu - bx * dyv + bz * dzu - bx * dzw1 - advb[0]
            F["by"] = bx * dxv - by * dxu + bz * dzv - by * dzw1 - advb[1]
            F["bz"] = bx * dxw - bz * dxu + by * dyw - bz * dyv - advb[2]
            F["bx"] += orm * (self.lx(bx) + self.ly(bx) + self.lz_sided(B[0]))
            F["by"] += orm * (self.lx(by) + self.ly(by) + self.lz_sided(B[1]))
            F["bz"] += orm * (self.lx(bz) + self.ly(bz) + self.lz(B[2]))
            fu += ob * (by * jz - bz * gxb[2] + bz * gzb[0])
            fv += ob * (bz * jx - bx * jz)
            fw += ob * (bx * gxb[2] - bx * gzb[0] - by * jx)
            ft += (ob * orm * ocv) * ri * (jz * jz + (gxb[2] - gzb[0]) ** 2 + jx * jx)
        F.update(ru=fu, rv=fv, rw=fw, tt=ft)
        return F

    def bcon(self, q, ro_in):
        m = self.m
        for a, b, c in ((1, 2, 3), (self.nz, self.nz - 1, self.nz - 2)):
            for k in ("ru", "rv"):
                q[k][a] = q["ro"][a] * (m["c43"] * q[k][b] / q["ro"][b] - m["c13"] * q[k][c] / q["ro"][c])
            q["rw"][a] = 0.0
            if self.mag:
                q["bz"][a] = 0.0
        q["tt"][1] = 1.0
        n = self.nz
        dz = m["dzf"] / float(self.dz[-1])
        q["tt"][n] = (m["c43"] * q["tt"][n - 1] - m["c13"] * q["tt"][n - 2]
                      + m["c23"] * dz * m["theta"] / float(self.rk[-1]))
        if self.flip:
            mir = 1 if int(m.get("id", 0)) else 0
            q["ro"][0], q["ro"][-1] = 1.0 / ro_in[2 * mir], 1.0 / ro_in[-1 - 2 * mir]

    def cfl(self, q):
        m, i = self.m, slice(1, -1)
        ro, tt = q["ro"][i], q["tt"][i]
        uu = (q["ru"][i] ** 2 + q["rv"][i] ** 2 + q["rw"][i] ** 2) / (ro * ro)
        um = math.sqrt(float((uu / (m["gamma"] * tt)).max()))
        cs = m["gamma"] * tt
        if self.mag:
            cs = cs + (q["bx"][i] ** 2 + q["by"][i] ** 2 + q["bz"][i] ** 2) * m["obeta"] / ro
        dd = torch.minimum(torch.minimum(self.ddx_, self.ddy_), self.ddz_)
        lim = [float((dd / (uu.sqrt() + cs.sqrt())).min()),
               float((0.5 * dd * dd * m["repr"] * m["cv"] * ro / self.rk).min()),
               float((0.375 * dd * dd * m["re"] * ro).min())]
        if self.mag:
            lim.append(float((0.5 * dd * dd).min()) * m["rm"])
        return m["sf"] * min(lim), um

    def step(self, force=None):
        m, i = self.m, slice(1, -1)
        dt, um = self.cfl(self.q)
        q, z = self.q, None
        for s, (g, zeta) in enumerate(((m["gam1"], m["zeta1"]), (m["gam2"], m["zeta2"]), (m["gam3"], 0.0))):
            F = self.rhs(q)
            for k, a in (force or {}).items():
                F[k] = F[k] + a
            new = {k: v.clone() for k, v in q.items()}
            zn = {}
            for k in self.names:
                new[k][i] = (q[k][i] if z is None else z[k]) + g * dt * F[k]
                if s < 2:
                    zn[k] = new[k][i] + zeta * dt * F[k]
            self.bcon(new, q["ro"])
            q, z = new, zn
        self.q = q
        return dt, um

    def out(self):
        return [_wrap(self.q[k]).cpu().numpy() for k in self.names]


def _weights(vec):
    """[(W [27][ci][co], b)] of a parameter vector W[co][tap][ci], b per layer."""
    out, o = [], 0
    for ci, co in ((8, 32), (32, 32), (32, 7)):
        w = vec[o:o + co * 27 * ci].reshape(co, 27, ci).permute(1, 2, 0)
        o += co * 27 * ci
        out.append((w, vec[o:o + co]))
        o += co
    return out


def _conv(x, w, b):
    """3x3x3 convolution of [nz][ny][nx][ci], periodic in x and y, zero outside in z."""
    xp = torch.nn.functional.pad(x, (0, 0, 0, 0, 0, 0, 1, 1))
    nz = x.shape[0]
    out = b
    for tap in range(27):
        dz, dy, dx = tap // 9, tap // 3 % 3 - 1, tap % 3 - 1
        out = out + torch.roll(xp[dz:dz + nz], (-dy, -dx), (1, 2)) @ w[tap]
    return out


def _network(x, vec):
    (w1, b1), (w2, b2), (w3, b3) = _weights(vec)
    g = torch.nn.functional.gelu
    return _conv(g(_conv(g(_conv(x, w1, b1)), w2, b2)), w3, b3)


def _exact_train(case, seed):
    p = torch.as_tensor(_net_params(seed), dtype=torch.float64, device=DEV)
    data = [(x.double(), t.double()) for x, t in _samples(case, seed)]
    m, v, losses, lr = torch.zeros_like(p), torch.zeros_like(p), [], float(np.float32(2e-3))
    for it in range(case["iters"]):
        x, t = data[it % len(data)]
        p.requires_grad_(True)
        loss = (_network(x, p) - t).square().mean()
        (g,) = torch.autograd.grad(loss, p)
        p = p.detach()
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        p = p - lr * (m / (1.0 - 0.9 ** (it + 1))) / ((v / (1.0 - 0.999 ** (it + 1))).sqrt() + 1e-8)
        losses.append(float(loss))
    return {"loss": [losses[0], losses[-1]], "params": p.cpu().numpy()}


def _exact_closure(case, seed):
    meta, q, _ = _case_state(case, seed)
    _, t, r = _meta(case["nx"], case["ny"], case["nz"], case["contrast"], case["ra"])
    f = dict(dtype=torch.float64, device=DEV)
    pin, ins, pout, outs = (torch.as_tensor(a, **f) for a in _closure_norm(meta, t, r))
    vec = torch.as_tensor(_net_params(seed), **f)
    s, i, g = _Step(meta, q, False), slice(1, -1), float(meta["gamma"])
    for _ in range(case["steps"]):
        ro, tt = s.q["ro"][i], s.q["tt"][i]
        ch = [ro, s.q["ru"][i] / ro, s.q["rv"][i] / ro, s.q["rw"][i] / ro, torch.log(tt) / (g - 1.0) - torch.log(ro),
              s.q["bx"][i], s.q["by"][i], s.q["bz"][i]]
        x = torch.stack([(c - pin[k][:, None, None]) / ins[k] for k, c in enumerate(ch)], dim=-1)
        y = _network(x, vec)
        force = {k: y[..., c] * outs[c] + pout[c][:, None, None]
                 for c, k in enumerate(("ru", "rv", "rw", "tt", "bx", "by", "bz"))}
        dt, um = s.step(force)
    return {"dt": dt, "umach": um, "state": s.out()}


def _exact_sample(case, seed):
    meta, q, _ = _case_state(case, seed)
    s, i, fac, nz = _Step(meta, q, True), slice(1, -1), case["factor"], case["nz"]
    F = s.rhs(s.q)

    def coarse(a):
        h = a.reshape(nz, case["ny"] // fac, fac, case["nx"] // fac, fac).mean(dim=(2, 4))
        w = torch.ones(fac + 1, dtype=torch.float64, device=DEV)
        w[0] = w[-1] = 0.5
        mid = [(h[k - fac // 2:k + fac // 2 + 1] * (w / fac)[:, None, None]).sum(0) for k in range(fac, nz - 1, fac)]
        return torch.stack([h[0]] + mid + [h[-1]])

    order = ("ru", "rv", "rw", "ro", "tt", "bx", "by", "bz")
    m, (ro, tt) = meta, (s.q["ro"][i], s.q["tt"][i])
    u, v, w = (s.q[k][i] / ro for k in ("ru", "rv", "rw"))
    mean = lambda a: a.mean(dim=(1, 2))  # noqa: E731
    ttm = mean(tt)
    fcon = -mean(ro * w * (2.5 * (tt - ttm[:, None, None]) + 0.5 * (u * u + v * v + w * w)))
    g = torch.empty_like(ttm)
    g[1:-1] = ttm[2:] - ttm[:-2]
    g[0] = -3.0 * ttm[0] + 4.0 * ttm[1] - ttm[2]
    g[-1] = 3.0 * ttm[-1] - 4.0 * ttm[-2] + ttm[-3]
    frad = g * m["hz"] * s.dz[:, 0, 0] * s.rk[:, 0, 0] / m["repr"]
    host = lambda a: a.cpu().numpy()  # noqa: E731
    return {"state": host(torch.stack([coarse(s.q[k][i]) for k in order])),
            "rhs": host(torch.stack([coarse(F[k]) for k in order])),
            "profiles": {"ttm": host(ttm), "rom": host(mean(ro)), "fconm": host(fcon), "fradm": host(frad)}}


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_train(case, seed)
    if kind == "closure":
        return _exact_closure(case, seed)
    if kind == "sample":
        return _exact_sample(case, seed)
    if kind == "ensemble":
        parts, dts, ums = [], [], []
        for meta, q in _ens_states(case, seed):
            s = _Step(meta, q, case["precision"] == "fp64")
            for _ in range(case["steps"]):
                dt, um = s.step()
            dts.append(dt)
            ums.append(um)
            parts.append([a.ravel() for a in s.out()])
        return {"dt": np.array(dts), "umach": np.array(ums), "state": [np.concatenate(c) for c in zip(*parts)]}
    zones = case["nx"] * case["ny"] * case["nz"]
    if zones * case.get("steps", 1) > 2e9:
        return None  # minutes of plain tensor operations
    meta, q, _ = _case_state(case, seed)
    s = _Step(meta, q, case.get("precision", "fp64") == "fp64")
    for _ in range(case.get("steps", 1)):
        dt, um = s.step()
    return {"dt": dt, "umach": um, "state": s.out()}
