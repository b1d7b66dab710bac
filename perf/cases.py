"""Performance cases: the calls a user of this library makes, by kind and size.

Each kind is one public entry point:

- model2d: synthetic2d, the traces of 2D shots (forward modelling)
- grad2d:  objfunc_gradient2d, the 2D FWI objective and gradient of one or
           more shots on one grid (one shot per call, or a survey per call)
- batch2d: objfunc_gradient2d_batch, shots on apertures of a wide model, the
           snapshots in FP32 or in 16 bits
- plan2d:  BatchPlan.run, the same through a plan kept over the iterations
           of an inversion
- gn2d:    gn_hessian2d, a Gauss-Newton product
- rtm2d:   rtm2d, a 2D migration image
- prop3d:  Prop3D.forward_shot, 3D modelling on a resident model
- model3d: model_data3d, the whole 3D modelling call
- grad3d:  objfunc_gradient3d, the 3D FWI objective and gradient
- rtm3d:   rtm3d, a 3D migration image

Sizes: 2D sections of 60-1024 x 60-512 points with 20-40 points of absorbing
boundary, 10 m and 1 ms, data at 4 ms; 3D volumes from about 100^3 to
460 x 572 x 572.  The jobs they stand for run 1000-3000 levels; the cases run
fewer of them in 3D, where a level is the same work each time.
"""
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "thesis-source-code_amd"))

import vtiamd  # noqa: E402

DX2D, DX3D, DT, RATE, RATIO = 10.0, 12.5, 1e-3, 4e-3, 4


def listed():
    return [
        # the smallest call: one shot over a small section, as a test of an
        # acquisition makes it; launches and latency count
        dict(name="model2d-small", kind="model2d", nx=96, nz=80, npad=20, nt=501, ns=1),
        # modelling of a survey at the ordinary 2D size, all shots in one call
        dict(name="model2d-survey", kind="model2d", nx=256, nz=256, npad=40, nt=1001, ns=16),
        # one shot's gradient per call, as the reference's drivers are called
        dict(name="grad2d-shot", kind="grad2d", nx=1024, nz=512, npad=40, nt=1001, ns=1),
        # one FWI evaluation: several shots of a survey in one call
        dict(name="grad2d-survey", kind="grad2d", nx=1024, nz=512, npad=40, nt=801, ns=6),
        # shots on ragged apertures of a wide model (streamer-like surveys)
        dict(name="batch2d", kind="batch2d", NX=2048, nz=512, npad=40, nt=801, ns=10, wmin=300, wmax=900, snap="fp32"),
        # the same with 16-bit snapshots, the option for long records
        dict(name="batch2d-s16", kind="batch2d", NX=1531, nz=389, npad=33, nt=801, ns=8, wmin=260, wmax=700, snap="s16"),
        # an inversion of small shots that keeps its plan over the iterations
        dict(name="plan2d-small", kind="plan2d", NX=1024, nz=96, npad=20, nt=601, ns=32, wmin=64, wmax=160,
             snap="fp32"),
        # one Gauss-Newton product of an inner conjugate-gradient loop
        dict(name="gn2d", kind="gn2d", nx=417, nz=301, npad=40, nt=801, ns=1),
        # one shot's migration image
        dict(name="rtm2d", kind="rtm2d", nx=652, nz=376, npad=40, nt=801, ns=1),
        # the largest: 3D modelling on a resident model at survey size
        dict(name="prop3d", kind="prop3d", nx=572, ny=572, nz=460, npad=30, nt=67),
        # a 3D gradient and a 3D image at target-oriented sizes
        dict(name="grad3d", kind="grad3d", nx=239, ny=283, nz=232, npad=30, nt=131),
        dict(name="rtm3d", kind="rtm3d", nx=163, ny=140, nz=128, npad=20, nt=131),
    ]


def draw(rng: random.Random):
    def size(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    kind = rng.choice(["model2d", "model2d", "grad2d", "grad2d", "batch2d", "batch2d", "plan2d", "gn2d", "rtm2d",
                       "prop3d", "model3d", "grad3d", "rtm3d"])
    if kind in ("model2d", "grad2d", "gn2d", "rtm2d"):
        ns = 1 if kind in ("gn2d", "rtm2d") else rng.choice([1, 1, 2, 3, 5])
        return dict(kind=kind, nx=size(60, 1024), nz=size(60, 512), npad=rng.choice([20, 25, 30, 40]),
                    nt=4 * size(75, 250) + 1, ns=ns)
    if kind in ("batch2d", "plan2d"):
        nx = size(500, 2048)
        wmin = size(60, 300)
        return dict(kind=kind, NX=nx, nz=size(80, 512), npad=rng.choice([20, 33, 40]), nt=4 * size(75, 200) + 1,
                    ns=rng.randrange(2, 10), wmin=wmin, wmax=min(nx, 900, wmin + size(40, 500)),
                    snap=rng.choice(["fp32", "fp32", "s16"]))
    top = 430 if kind == "prop3d" else 260
    return dict(kind=kind, nx=size(90, top), ny=size(90, top), nz=size(90, top), npad=rng.choice([15, 20, 30]),
                nt=67 if kind == "prop3d" else 131)


# ---- inputs -----------------------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _ricker(nt, freq, t0):
    a = (np.pi * freq * (np.arange(nt) * DT - t0)) ** 2
    return ((1 - 2 * a) * np.exp(-a)).astype(np.float32)


def _cij(v, eps, dl):
    c33 = v * v
    return tuple(np.ascontiguousarray(c, np.float32) for c in (c33 * (1 + 2 * eps), c33 * np.sqrt(1 + 2 * dl), c33))


def _model2d(rng, nnz, nnx, npad):
    """A velocity gradient with smooth anomalies, and VTI parameters growing with depth."""
    z = np.clip(np.arange(nnz) - npad, 0, nnz - 2 * npad - 1) / max(nnz - 2 * npad - 1, 1)
    coarse = torch.from_numpy(rng.uniform(-1.0, 1.0, (1, 1, nnz // 25 + 2, nnx // 25 + 2)))
    soft = torch.nn.functional.interpolate(coarse, size=(nnz, nnx), mode="bilinear", align_corners=True)[0, 0].numpy()
    v = (1500.0 + 2900.0 * z)[:, None] * (1 + 0.08 * soft)
    dl = np.repeat((0.1 * z)[:, None], nnx, 1)
    return _cij(v, 0.5 * dl + 0.05, dl)


def _events(rng, t, x, amp):
    """Observed traces: a direct wave and hyperbolic reflections, time-major
    (samples, receivers), at the amplitude amp, about that of the modelled
    data.  x: the receivers' offsets in metres."""
    d = np.zeros((t.size, x.size))
    for k in range(6):
        t0 = 0.022 if k == 0 else rng.uniform(0.1, 1.2)
        v = rng.uniform(1500.0, 3500.0)
        a = (np.pi * 12.0 * (t[:, None] - 0.09 - np.sqrt(t0 * t0 + (x[None, :] / v) ** 2))) ** 2
        d += rng.uniform(0.3, 1.0) * rng.choice([-1.0, 1.0]) * (1 - 2 * a) * np.exp(-a)
    return (amp * d).astype(np.float32)


def _geometry2d(case):
    """Shots spread along the section two rows below its top, receivers in every column one row below it."""
    nx, npad, ns = case["nx"], case["npad"], case["ns"]
    sloc = [[npad + (2 * k + 1) * nx // (2 * ns), npad + 2, nx, k * nx] for k in range(ns)]
    rloc = [[npad + i, npad + 1] for _ in range(ns) for i in range(nx)]
    return np.array(sloc, np.int32), np.array(rloc, np.int32)


def _inputs2d(case, seed):
    rng = np.random.default_rng(seed)
    nx, nz, npad, nt = (case[k] for k in ("nx", "nz", "npad", "nt"))
    sloc, rloc = _geometry2d(case)
    s = dict(c=_model2d(rng, nz + 2 * npad, nx + 2 * npad, npad), w=_ricker(nt, rng.uniform(8.0, 14.0), 0.1),
             sloc=sloc, rloc=rloc, rest=(nx, nz, nt, npad, DX2D, DX2D, DT, RATE))
    t = np.arange((nt - 1) // RATIO + 1) * RATE
    if case["kind"] in ("grad2d", "rtm2d"):
        s["data"] = np.concatenate([_events(rng, t, DX2D * (rloc[r0:r0 + nr, 0] - ix), 2e-6)
                                    for ix, _, nr, r0 in sloc], axis=1)
    if case["kind"] == "gn2d":
        d = _model2d(rng, nz + 2 * npad, nx + 2 * npad, npad)
        s["dc"] = tuple((0.02 * (a - b)).astype(np.float32) for a, b in zip(d, s["c"]))
    return s


def _inputs_batch(case, seed):
    rng = np.random.default_rng(seed)
    NX, nz, npad, nt = (case[k] for k in ("NX", "nz", "npad", "nt"))
    shots, rloc, data = [], [], []
    t = np.arange((nt - 1) // RATIO + 1) * RATE
    # the apertures are the survey's, the same for every seed
    geo = random.Random(case["ns"] * 1009 + NX)
    for _ in range(case["ns"]):
        nx = geo.randint(case["wmin"], case["wmax"])
        shots.append([geo.randint(0, NX - nx), nx, npad + nx // 2, npad + 2, nx, len(rloc)])
        rloc += [[npad + i, npad + 1] for i in range(nx)]
        data.append(_events(rng, t, DX2D * (np.arange(nx) - nx // 2), 2e-6).ravel())
    return dict(c=_model2d(rng, nz + 2 * npad, NX + 2 * npad, npad), w=_ricker(nt, rng.uniform(8.0, 14.0), 0.1),
                shots=np.array(shots, np.int32), rloc=np.array(rloc, np.int32), data=np.concatenate(data),
                rest=(NX, nz, nt, npad, DX2D, DX2D, DT, RATE))


def _lmax(nt):
    """The time levels the 3D drivers advance (rounds of 64)."""
    return (nt - 2) // 64 * 64 + 1


def _inputs3d(case, seed):
    """Dipping layers, a source near the middle of the top, a sheet of receivers."""
    rng = np.random.default_rng(seed)
    nx, ny, nz, npad, nt = (case[k] for k in ("nx", "ny", "nz", "npad", "nt"))
    dev = _device()
    z, y, x = (torch.arange(n, device=dev, dtype=torch.float32) for n in (nz, ny, nx))
    depth = z[:, None, None] + rng.uniform(-0.15, 0.15) * (y[None, :, None] - ny / 2) + \
        rng.uniform(-0.15, 0.15) * (x[None, None, :] - nx / 2)
    bounds = torch.tensor(np.sort(rng.uniform(0.1, 0.9, 5)) * nz, device=dev, dtype=torch.float32)
    layer = torch.bucketize(depth, bounds)

    def of(vals):
        return torch.tensor(vals, device=dev, dtype=torch.float32)[layer]

    v, e = of(np.sort(rng.uniform(1500.0, 4300.0, 6))), rng.uniform(0.0, 0.25, 6)
    d = of(np.minimum(rng.uniform(0.0, 0.12, 6), e))
    e = of(e)
    c33 = v * v
    c = [a.cpu().numpy() for a in (c33 * (1 + 2 * e), c33 * torch.sqrt(1 + 2 * d), c33)]
    step = max(1, min(nx, ny) // 100)
    zr = npad + 2
    rec = [(ix, iy) for iy in range(npad, ny - npad, 2 * step) for ix in range(npad, nx - npad, step)]
    src = (nx // 2 + int(rng.integers(-5, 6)), ny // 2 + int(rng.integers(-5, 6)), npad + 4)
    return dict(c=c, w=_ricker(nt, rng.uniform(18.0, 24.0), 0.05), rec=rec, zr=zr, src=src, rng=rng)


def _shell(case):
    """True in the absorbing boundary's shell of the volume, which the packed boundary arrays hold in this order."""
    nx, ny, nz, n = (case[k] for k in ("nx", "ny", "nz", "npad"))
    m = np.ones((nz, ny, nx), bool)
    m[n:nz - n, n:ny - n, n:nx - n] = False
    return m


def _calls3d(case, s):
    nr = len(s["rec"])
    h = DX3D
    live = [1.0] if case["kind"] != "rtm3d" else []
    s["recloc"] = np.array([[ix * h + 0.1, iy * h + 0.1, s["zr"] * h + 0.1] + live for ix, iy in s["rec"]], np.float32)
    s["souloc"] = np.array([[(k * h + 0.1) for k in s["src"]] + [nr, 0]], np.float32)
    if case["kind"] == "model3d":
        return s
    t = np.arange((case["nt"] - 1) // RATIO + 1) * RATE
    x = h * np.array([np.hypot(ix - s["src"][0], iy - s["src"][1]) for ix, iy in s["rec"]])
    s["data"] = np.ascontiguousarray(_events(s["rng"], t, x, 5e-7).T).ravel()
    if case["kind"] == "grad3d":
        s["cij"] = np.stack(s["c"])
        shell = _shell(case)
        pad = [c[shell] for c in s["c"]]
        scale = s["rng"].uniform(0.75, 1.0, pad[0].size).astype(np.float32)
        s["padb"], s["randb"] = np.concatenate(pad), np.concatenate([p * scale for p in pad])
    return s


class _Held:
    """A library object released with the state that holds it."""

    def __init__(self, obj):
        self.obj = obj

    def __del__(self):
        self.obj.close()


_context = []


def _ctx():
    if not _context:
        _context.append(vtiamd.Context(0))
    return _context[0]


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("model2d", "grad2d", "gn2d", "rtm2d"):
        s = _inputs2d(case, seed)
        s["taper"] = vtiamd.init_taper2d(case["nx"], case["nz"], case["npad"])
    elif kind in ("batch2d", "plan2d"):
        s = _inputs_batch(case, seed)
        if kind == "batch2d":
            t = vtiamd.tune_batch2d(_ctx(), s["shots"], s["rloc"], case["NX"], case["nz"], case["nt"], case["npad"],
                                    DX2D, DX2D, DT, RATE)
            s["shape"] = {k: t[k] for k in ("levels", "tile_rows", "max_wave")}
        else:
            s["plan"] = _Held(vtiamd.BatchPlan(_ctx(), s["data"], s["w"], s["shots"], s["rloc"], *s["rest"],
                                               snap=case["snap"]))
    else:
        s = _inputs3d(case, seed)
        if kind == "prop3d":
            nx, ny, nz = case["nx"], case["ny"], case["nz"]
            s["prop"] = _Held(vtiamd.Prop3D(_ctx(), nx, ny, nz, case["npad"], DX3D, DX3D, DX3D, DT))
            s["prop"].obj.set_model(*s.pop("c"))
            s["at"] = s["src"][0] + s["src"][1] * nx + s["src"][2] * nx * ny
            s["idx"] = np.array([ix + iy * nx + s["zr"] * nx * ny for ix, iy in s["rec"]], np.int64)
        else:
            s = _calls3d(case, s)
    s["case"] = case
    return s


def run(s):
    case = s["case"]
    kind, nt = case["kind"], case["nt"]
    if kind == "model2d":
        return vtiamd.synthetic2d(_ctx(), *s["c"], s["w"], s["sloc"], s["rloc"], s["taper"], *s["rest"])
    if kind == "grad2d":
        return vtiamd.objfunc_gradient2d(_ctx(), s["data"], *s["c"], s["w"], s["sloc"], s["rloc"], s["taper"],
                                         *s["rest"])
    if kind == "gn2d":
        return vtiamd.gn_hessian2d(_ctx(), *s["c"], *s["dc"], s["w"], s["sloc"], s["rloc"], s["taper"], *s["rest"])
    if kind == "rtm2d":
        return vtiamd.rtm2d(_ctx(), s["data"], *s["c"], s["w"], s["sloc"], s["rloc"], s["taper"], *s["rest"])
    if kind == "batch2d":
        return vtiamd.objfunc_gradient2d_batch(_ctx(), s["data"], *s["c"], s["w"], s["shots"], s["rloc"], *s["rest"],
                                               snap=case["snap"], **s["shape"])
    if kind == "plan2d":
        return s["plan"].obj.run(*s["c"])
    if kind == "prop3d":
        p = s["prop"].obj
        p.reset(s["at"], np.float32(np.float32(DT) * np.float32(DT)) * s["w"][0])
        return p.forward_shot(_lmax(nt), s["w"], s["at"], s["idx"], RATIO, (nt - 1) // RATIO + 1)
    o, d = (0.0,) * 3, (DX3D,) * 3
    geo = (_ctx(), s["souloc"], [0], s["recloc"], s["w"])
    if kind == "model3d":
        return vtiamd.model_data3d(*geo, *s["c"], nt, case["npad"], o, d, DT, RATE)
    if kind == "grad3d":
        return vtiamd.objfunc_gradient3d(*geo, s["cij"], s["padb"], s["randb"], nt, case["npad"], o, d, DT, RATE,
                                         s["data"])
    return vtiamd.rtm3d(*geo, *s["c"], nt, case["npad"], o, d, DT, RATE, s["data"])


# ---- work -------------------------------------------------------------------

def work(case):
    """Operations: the adds, multiplies and divides of the scheme per point
    and level.  Bytes in 2D, where a shot's fields can stay on the chip: the
    model, the traces and the result once, and each snapshot written and read
    once.  Bytes in 3D, where they cannot: each level reads the two levels
    before it and the coefficients and writes one level (36 per point), with
    the accumulators in the backward pass."""
    kind, nt = case["kind"], case["nt"]
    nnt = (nt - 1) // RATIO + 1
    if kind in ("prop3d", "model3d", "grad3d", "rtm3d"):
        n = case["nx"] * case["ny"] * case["nz"]
        steps = _lmax(nt) - 1
        b, f = {"prop3d": (36, 67), "model3d": (36, 67), "grad3d": (36 + 36 + 84, 67 * 4 + 12),
                "rtm3d": (36 + 68, 67 * 3 + 8)}[kind]
        io = {"prop3d": 0, "model3d": 12, "grad3d": 24, "rtm3d": 16}[kind]
        return {"bytes": n * (b * steps + io), "flops": n * f * steps}
    if kind in ("batch2d", "plan2d"):
        s = _inputs_geometry(case)
        pts = sum(w * (case["nz"] + 2 * case["npad"]) for w in s)
        model = (case["NX"] + 2 * case["npad"]) * (case["nz"] + 2 * case["npad"])
        traces = sum(s) - 2 * case["npad"] * len(s)
        snap = 2 if case["snap"] == "s16" else 4
        return {"bytes": model * (12 + 24) + pts * nnt * 2 * 2 * snap + traces * nnt * 4, "flops": pts * nt * (46 + 62)}
    one = (case["nx"] + 2 * case["npad"]) * (case["nz"] + 2 * case["npad"])
    pts, traces = one * case["ns"], case["nx"] * case["ns"] * nnt * 4
    per, flops, io = {"model2d": (0, 46, 12), "grad2d": (16, 46 + 62, 24), "gn2d": (16, 106 + 60, 36),
                      "rtm2d": (8, 46 + 54, 16)}[kind]
    return {"bytes": one * io + pts * nnt * per + traces, "flops": pts * nt * flops}


def _inputs_geometry(case):
    geo = random.Random(case["ns"] * 1009 + case["NX"])
    widths = []
    for _ in range(case["ns"]):
        nx = geo.randint(case["wmin"], case["wmax"])
        geo.randint(0, case["NX"] - nx)
        widths.append(nx + 2 * case["npad"])
    return widths


# ---- the same results in 64 bits, in plain torch -----------------------------

_W = (-2.84722222222, 1.6, -0.2, 0.02539682539, -0.00178571428)
_DT = float(np.float32(DT))
_DT2 = float(np.float32(np.float32(DT) * np.float32(DT)))


def _f64(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(_device(), torch.float64)


def _second(a, dim, h2):
    """8th-order second difference along a dimension over the points 4 or more from every edge of the last two."""
    n = a.dim()
    inner = [slice(None)] * (n - 2) + [slice(4, -4), slice(4, -4)]

    def at(k):
        i = list(inner)
        i[dim] = slice(4 + k, a.shape[dim] - 4 + k)
        return a[tuple(i)]

    out = _W[0] * at(0)
    for k in range(1, 5):
        out += _W[k] * (at(-k) + at(k))
    return out / h2


def _taper2d(nnz, nnx, npad):
    t = np.ones(npad + 1)
    t[:npad] = 0.95 + 0.05 * np.cos(np.pi * (npad - 1 - np.arange(npad)) / npad)

    def along(n):
        i = np.arange(n)
        return t[np.minimum(np.minimum(i, n - 1 - i), npad)]

    return _f64(along(nnz)[:, None] * along(nnx)[None, :])


class _Wave2:
    """Levels of the 2D scheme for a stack of shots on one grid; D C or, transposed, C D."""

    I = (Ellipsis, slice(4, -4), slice(4, -4))

    def __init__(self, c, taper, ns):
        self.c = [a[self.I] for a in c]
        self.full, self.taper, self.ti = c, taper, taper[self.I]
        shape = (ns,) + tuple(taper.shape)
        self.p, self.q, self.pp, self.qp = (torch.zeros(shape, dtype=torch.float64, device=taper.device)
                                            for _ in range(4))

    def d(self):
        h2 = DX2D * DX2D
        return _second(self.p, -1, h2), _second(self.q, -2, h2)

    def step(self, transposed=False, add=None, extra=None):
        if transposed:
            a, b, e = self.full
            tp = _second(a * self.p + b * self.q, -1, DX2D * DX2D)
            tq = _second(b * self.p + e * self.q, -2, DX2D * DX2D)
            fp, fq = tp, tq
        else:
            tp, tq = self.d()
            a, b, e = self.c
            fp, fq = a * tp + b * tq, b * tp + e * tq
        I = self.I
        pn, qn = torch.zeros_like(self.p), torch.zeros_like(self.q)
        pn[I] = 2 * self.p[I] + _DT2 * fp - self.pp[I] * self.ti
        qn[I] = 2 * self.q[I] + _DT2 * fq - self.qp[I] * self.ti
        if extra is not None:
            pn[I] += extra[0]
            qn[I] += extra[1]
        if add is not None:
            where, val = add
            for f in (pn, qn):
                f.view(-1).index_add_(0, where, val)
        # (a level is tapered when made and again when it becomes the previous one)
        self.pp, self.qp = self.p, self.q
        self.p, self.q = pn * self.taper, qn * self.taper
        return tp, tq


def _exact2d(kind, c, w, src, rec, obs, npad, nt, dc=None):
    """The shots of one grid: src (ns,), rec (ns, nr) flat grid indices, obs (nnt, ns, nr) or None."""
    ns, (nnz, nnx) = len(src), c[0].shape
    n = nnz * nnx
    c = [_f64(a) for a in c]
    taper = _taper2d(nnz, nnx, npad)
    off = torch.arange(ns, device=taper.device) * n
    src = torch.as_tensor(src, device=taper.device) + off
    rec = (torch.as_tensor(rec, device=taper.device) + off[:, None]).reshape(-1)
    nnt = (nt - 1) // RATIO + 1
    w = w.astype(np.float64)
    rtm = kind == "rtm2d"
    if rtm:  # dipoles: the point below takes the other sign
        src, rec = torch.cat([src, src + nnx]), torch.cat([rec, rec + nnx])
        sign = torch.cat([torch.ones(ns), -torch.ones(ns)]).to(taper)
    else:
        sign = torch.ones(ns).to(taper)
    nrec = rec.numel()
    F = _Wave2(c, taper, ns)
    for f in (F.p, F.q):
        f.view(-1)[src] = _DT2 * w[0] * sign
    if kind in ("model2d", "rtm2d"):
        F.p, F.q = F.p * taper, F.q * taper
    B = _Wave2(c, taper, ns) if kind == "gn2d" else None
    dci = [_f64(a)[_Wave2.I] for a in dc] if dc is not None else None
    tr = torch.zeros((nnt, nrec), dtype=torch.float64, device=taper.device)
    snaps = {}
    for it in range(2, nt):
        keep = (it - 1) % RATIO == 0 and kind in ("grad2d", "gn2d")
        tp, tq = F.step(add=(src, _DT2 * w[it - 1] * sign))
        if keep:
            snaps[(it - 1) // RATIO] = (tp.clone(), tq.clone())
        if B is not None:
            B.step(extra=(_DT2 * (dci[0] * tp + dci[1] * tq), _DT2 * (dci[1] * tp + dci[2] * tq)))
        if it % RATIO == 0:
            R = F if B is None else B
            if rtm:
                snaps[it // RATIO] = 0.5 * (F.p + F.q)[_Wave2.I]
            else:
                tr[it // RATIO] = 0.5 * (R.p + R.q).view(-1)[rec]
    if kind == "model2d":
        return tr.reshape(nnt, -1).cpu().numpy()
    if rtm:
        zero = torch.zeros_like(snaps[nnt - 1])
        snaps[0] = zero
        res = _f64(obs).reshape(nnt, -1)
        res = torch.cat([res, -res], 1)
    else:
        snaps[nnt - 1] = F.d()
        snaps[0] = tuple(torch.zeros_like(t) for t in snaps[1])
        res = tr if kind == "gn2d" else tr - _f64(obs).reshape(nnt, -1)
    f = 0.5 * float((res * res).sum())
    res = torch.cat([res, torch.zeros_like(res[:1])])
    L = _Wave2(c, taper, ns)
    for a in (L.p, L.q):
        a.view(-1).index_add_(0, rec, _DT2 * 0.5 * res[nnt - 1])
    if rtm:
        L.p, L.q = L.p * taper, L.q * taper
    I = _Wave2.I
    g = [torch.zeros_like(L.p) for _ in range(1 if rtm else 3)]

    def image(t):
        k = int(t)
        a = t - k
        if rtm:
            g[0][I] += 0.5 * (L.p + L.q)[I] * ((1 - a) * snaps[k] + a * snaps[k + 1])
            return
        dp, dq = ((1 - a) * x + a * y for x, y in zip(snaps[k], snaps[k + 1]))
        g[0][I] += L.p[I] * dp
        g[1][I] += L.p[I] * dq + L.q[I] * dp
        g[2][I] += L.q[I] * dq

    image((nt - 2) / RATIO)
    for it in range(nt - 3, -1, -1):
        t = (it + 1) / RATIO
        k = int(t)
        L.step(transposed=kind == "grad2d",
               add=(rec, _DT2 * 0.5 * ((1 - (t - k)) * res[k] + (t - k) * res[k + 1])))
        image(it / RATIO)
    return f, g


def _damp3d(case):
    n = case["npad"]

    def along(m):
        i = np.arange(m)
        dist = np.where(i < n, n - i, np.where(i > m - n, i - m + n, 0))
        return _f64(0.95 + 0.05 * np.cos(np.pi * dist / n))

    nz, ny, nx = case["nz"], case["ny"], case["nx"]
    return along(nz)[:, None, None] * along(ny)[None, :, None] * along(nx)[None, None, :]


class _Wave3:
    """Levels of the 3D scheme.  With damping, 4-plane blocks are stepped and
    damped from the top down, so a block's stencil reaches planes above it
    that carry the current level's damping once more."""

    def __init__(self, c, damp, shape):
        self.zm = shape[0] // 4 * 4
        self.I = (slice(0, self.zm), slice(4, -4), slice(4, -4))
        self.c = [a[self.I] for a in c]
        self.damp = None if damp is None else damp[self.I]
        self.x, self.z, self.px, self.pz = (torch.zeros(shape, dtype=torch.float64, device=_device())
                                            for _ in range(4))

    def lap(self):
        I, h2 = self.I, DX3D * DX3D
        s = self.x[:self.zm]
        txy = _second(s, -1, h2)
        txy += _second(s, -2, h2)
        q = self.z[I]
        tz = _W[0] * q
        for k in range(1, 5):
            tz[k:] += _W[k] * q[:-k]
            tz[:-k] += _W[k] * q[k:]
        if self.damp is not None:
            e = q * (self.damp - 1)
            for r in range(4):
                for k in range(r + 1, 5):
                    tz[4 + r::4] += _W[k] * e[4 + r - k:self.zm - k:4]
        return txy, tz / h2

    def step(self, lap, at=(), val=None):
        I = self.I
        txy, tz = lap
        a, b, c = self.c
        nx = _DT2 * (a * txy + b * tz) + 2 * self.x[I] - self.px[I]
        nz = _DT2 * (b * txy + c * tz) + 2 * self.z[I] - self.pz[I]
        self.px[I], self.pz[I] = nx, nz
        for where, vx, vz in at:
            self.px.view(-1).index_add_(0, where, vx)
            self.pz.view(-1).index_add_(0, where, vz)
        if self.damp is not None:
            for f in (self.px, self.pz, self.x, self.z):
                f[I] *= self.damp
        self.x, self.px = self.px, self.x
        self.z, self.pz = self.pz, self.z


def _exact3d(case, s):
    kind, nt = case["kind"], case["nt"]
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    shape, lmax, nnt = (nz, ny, nx), _lmax(nt), (nt - 1) // RATIO + 1
    dev = _device()
    src = torch.tensor([s["src"][0] + s["src"][1] * nx + s["src"][2] * nx * ny], device=dev)
    true = torch.tensor([ix + iy * nx + s["zr"] * nx * ny for ix, iy in s["rec"]], device=dev)
    w = _DT2 * s["w"].astype(np.float64)
    third, two = 0.3333333333, 0.6666666666
    damp = _damp3d(case)

    def forward(c, damp, record):
        F = _Wave3(c, damp, shape)
        F.x.view(-1)[src] = w[0]
        F.z.view(-1)[src] = w[0]
        tr = torch.zeros((nnt, true.numel()), dtype=torch.float64, device=dev)
        for it in range(2, lmax + 1):
            v = torch.full((1,), w[it - 1], dtype=torch.float64, device=dev)
            F.step(F.lap(), [(src, v, v)])
            if record and it % RATIO == 0 and it // RATIO < nnt:
                tr[it // RATIO] = two * F.x.view(-1)[true] + third * F.z.view(-1)[true]
        return F, tr

    c = [_f64(a) for a in s["c"]]
    if kind in ("prop3d", "model3d"):
        return forward(c, damp, True)[1].T.contiguous()
    if kind == "grad3d":
        _, tr = forward(c, damp, True)
        res = tr - _f64(s["data"].reshape(-1, nnt).T)
        shell = torch.from_numpy(_shell(case)).to(dev)
        c = [a.clone() for a in c]
        for a, b in zip(c, s["randb"].reshape(3, -1)):
            a[shell] = _f64(b)
    else:
        res = _f64(s["data"].reshape(-1, nnt).T)
    F, _ = forward(c, None, False)
    F.x, F.px, F.z, F.pz = F.px, F.x, F.pz, F.z
    L = _Wave3(c, damp, shape)
    L.x.view(-1)[true] = two * _DT2 * res[nnt - 1]
    L.z.view(-1)[true] = third * _DT2 * res[nnt - 1]
    I = F.I
    g = [torch.zeros(shape, dtype=torch.float64, device=dev) for _ in range(3 if kind == "grad3d" else 1)]
    for lev in range(2, lmax + 1):
        it = nt - 1 - lev
        t = (it + 1) / RATIO
        k = int(t)
        r = res[nnt - 1] if k >= nnt - 1 else (1 - (t - k)) * res[k] + (t - k) * res[k + 1]
        txy, tz = F.lap()
        if kind == "grad3d":
            g[0][I] += L.x[I] * txy
            g[1][I] += L.x[I] * tz + L.z[I] * txy
            g[2][I] += L.z[I] * tz
        sx, sz = F.x[I].clone(), F.z[I].clone()
        v = torch.full((1,), w[it + 1], dtype=torch.float64, device=dev)
        F.step((txy, tz), [(src, v, v)])
        L.step(L.lap(), [(true, two * _DT2 * r, third * _DT2 * r)])
        if kind == "rtm3d":  # the current levels, the receiver side's after its damping
            g[0][I] += (two * sx + third * sz) * (two * L.px[I] + third * L.pz[I])
    if kind == "rtm3d":
        return g[0]
    return 0.5 * float((res * res).sum()), torch.stack(g)


def exact(case, seed):
    kind, nt, npad = case["kind"], case["nt"], case["npad"]
    if kind in ("prop3d", "model3d", "grad3d", "rtm3d"):
        s = _inputs3d(case, seed)
        if kind != "prop3d":
            s = _calls3d(case, s)
        out = _exact3d(case, s)
        if kind == "model3d":
            return out.reshape(-1)
        return (torch.tensor(out[0]), out[1]) if kind == "grad3d" else out
    if kind in ("batch2d", "plan2d"):
        s = _inputs_batch(case, seed)
        nnt = (nt - 1) // RATIO + 1
        f, g, at = 0.0, torch.zeros((3,) + s["c"][0].shape, dtype=torch.float64, device=_device()), 0
        for c0, nx, ix, iz, nr, r0 in s["shots"].tolist():
            nnx = nx + 2 * npad
            c = [np.ascontiguousarray(a[:, c0:c0 + nnx]) for a in s["c"]]
            rec = s["rloc"][r0:r0 + nr].astype(np.int64)
            obs = s["data"][at:at + nnt * nr].reshape(nnt, 1, nr)
            at += nnt * nr
            fk, gk = _exact2d("grad2d", c, s["w"], np.array([ix + iz * nnx]), (rec[:, 0] + rec[:, 1] * nnx)[None],
                              obs, npad, nt)
            f += fk
            for a, b in zip(g, gk):
                a[:, c0:c0 + nnx] += b[0]
        return torch.tensor(f, dtype=torch.float64), g
    s = _inputs2d(case, seed)
    nx, nnx, ns = case["nx"], case["nx"] + 2 * npad, case["ns"]
    src = s["sloc"][:, 0].astype(np.int64) + s["sloc"][:, 1].astype(np.int64) * nnx
    rec = (s["rloc"][:, 0].astype(np.int64) + s["rloc"][:, 1].astype(np.int64) * nnx).reshape(ns, nx)
    out = _exact2d(kind, s["c"], s["w"], src, rec, s.get("data"), npad, nt, s.get("dc"))
    if kind == "model2d":
        return out
    f, g = out
    g = [a.sum(0) for a in g]
    if kind == "rtm2d":
        return g[0]
    g = torch.stack(g)
    return (torch.tensor(f, dtype=torch.float64), g) if kind == "grad2d" else g
