"""The reconstructions this framework is used for, as cases that can be timed.

Four kinds of work, each through the public entry points of `risa_amd.device`:

* "chain": raw uint16 detector frames in HBM to images, a call of `Chain` (plain
  FP32, or the mixed-precision chain whose filtered sinogram is FP16);
* "stages": one frame through the four stage handles, call by call, as an
  online pipeline with one frame in flight runs them;
* "forward" and "backward": filtered backprojection of parallel sinograms and
  its hand-written adjoint (sinogram and filter-tap gradients), one training
  step of learnable taps;
* "uneven": a batch of backprojections of different geometry in one launch.

Geometries are the two configurations of the package (c0: 432 x 500 fan, one
plane; c1: 768 x 1000 fan, two planes), the sizes of the benchmark and of the
tests, and sizes around them.  `exact` restates each path in float64 with
torch and numpy alone.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

DEV = "cuda"
I0 = 60000.0          # counts of an unattenuated detector sample
MU_MAX = 0.05         # largest attenuation coefficient of an ellipse, 1/mm
WIDTH = 190.0         # reconstructed field, mm
X4_SCALE = 256.0      # FP16 sinograms store 256 * value
WINDOWS = ("ramp", "sheppLogan", "cosine", "hamming", "hanning")


# ------------------------------------------------------------------- cases --
def listed():
    return [
        # one frame of the small configuration: the latency of a single call
        dict(name="frame_c0", kind="chain", base="c0", mode="plain", frames=1, P=500, D=256, N=256, window=0, module=0),
        # the small configuration's whole job in one call
        dict(name="job_c0", kind="chain", base="c0", mode="plain", frames=100, P=500, D=256, N=256, window=0, module=0),
        # an online pipeline's single production frame, stage by stage
        dict(name="stages_c1", kind="stages", base="c1", P=1000, D=512, N=512, window=1),
        # production rate, FP32: a call of frames of both detector planes
        dict(name="plain_c1", kind="chain", base="c1", mode="plain", frames=256, P=1000, D=512, N=512, window=1, module=0),
        # production rate, mixed precision, the benchmark's call size
        dict(name="mixed_c1", kind="chain", base="c1", mode="mixed", frames=512, P=1000, D=512, N=512, window=1, module=0),
        # a short mixed call, as the streaming stage makes when few frames are queued
        dict(name="mixed_short", kind="chain", base="c1", mode="mixed", frames=8, P=1000, D=512, N=512, window=1, module=0),
        # frames as the scanner sends them (27 modules of 16 detectors), a ragged count
        dict(name="mixed_rofex", kind="chain", base="c0", mode="mixed", frames=30, P=500, D=256, N=256, window=3, module=1),
        # one training step's two directions at the benchmark's size
        dict(name="forward_c4", kind="forward", slices=16, P=720, D=512, N=512, window=0, rotation=0.0, mask=1),
        dict(name="backward_c4", kind="backward", slices=16, P=720, D=512, N=512, window=0, rotation=0.0, mask=1),
        # the same at ragged sizes: a detector count without a 512-point
        # transform, and one that no transform of radix 2, 3 and 5 divides
        dict(name="forward_ragged", kind="forward", slices=6, P=360, D=500, N=384, window=2, rotation=13.0, mask=1),
        dict(name="backward_ragged", kind="backward", slices=5, P=181, D=303, N=320, window=1, rotation=0.0, mask=0),
        # 96 reconstructions of uneven geometry, FP32 and FP16 sinograms
        dict(name="uneven_96", kind="uneven", jobs=96, Nmin=256, Nmax=768, Pmin=360, Pmax=1000, Dmin=256, Dmax=768, layout=96),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("plain", "mixed", "mixed", "plain", "stages", "forward", "backward", "uneven"))
    if kind in ("plain", "mixed", "stages"):
        base = rng.choice(("c0", "c1"))
        P = rng.randint(300, 1000)
        D = rng.randint(200, 560)
        c = dict(kind="chain", base=base, mode=kind, P=P, D=D, N=rng.randint(max(200, D // 2), 560),
                 window=rng.randrange(5), module=0)
        if kind == "stages":
            del c["mode"], c["module"]
            return dict(c, kind="stages")
        c["module"] = int(rng.random() < 0.25)
        c["frames"] = _log(rng, 1, 96 if kind == "plain" else 192)
        return c
    if kind in ("forward", "backward"):
        N = _log(rng, 128, 640)
        slices = _log(rng, 1, 20)
        # more detectors than pixels: a few slices (that adjoint walks every ray)
        D = rng.randint(N // 2, N + N // 4 if slices <= 4 else N)
        return dict(kind=kind, slices=slices, P=rng.randint(120, 800), D=D, N=N, window=rng.randrange(5),
                    rotation=round(rng.uniform(-45.0, 45.0), 2), mask=int(rng.random() < 0.7))
    return dict(kind="uneven", jobs=_log(rng, 6, 80), Nmin=rng.randint(128, 256), Nmax=rng.randint(320, 768),
                Pmin=rng.randint(180, 400), Pmax=rng.randint(500, 1000), Dmin=rng.randint(160, 256),
                Dmax=rng.randint(384, 768), layout=rng.randrange(1 << 20))


# ------------------------------------------------------------------ inputs --
def _generator(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 1000003 + salt) & 0x7FFFFFFF)
    return g


def _phantoms(seed, count):
    """count phantoms of 16 random ellipses: (cx, cy, a, b, phi, mu), each [count][16]."""
    u = torch.rand((6, count, 16), generator=_generator(seed, 1), device=DEV)
    R = 0.5 * WIDTH
    rad, ang = 0.8 * R * u[0].sqrt(), 2 * math.pi * u[1]
    return (rad * ang.cos(), rad * ang.sin(), (0.05 + 0.35 * u[2]) * R, (0.05 + 0.35 * u[3]) * R, math.pi * u[4],
            MU_MAX * u[5])


def _line_integrals(phantoms, px, py, ux, uy):
    """Attenuation along the lines (px, py) + l (ux, uy), [count][lines]."""
    total = torch.zeros((phantoms[0].shape[0],) + px.shape, device=DEV)
    for e in range(phantoms[0].shape[1]):
        cx, cy, a, b, phi, mu = (v[:, e].reshape((-1,) + (1,) * px.dim()) for v in phantoms)
        c, s = phi.cos(), phi.sin()
        dx, dy = px - cx, py - cy
        qx, qy = (dx * c + dy * s) / a, (dy * c - dx * s) / b
        vx, vy = (ux * c + uy * s) / a, (uy * c - ux * s) / b
        A, B, C = vx * vx + vy * vy, 2 * (qx * vx + qy * vy), qx * qx + qy * qy - 1
        total += mu * (B * B - 4 * A * C).clamp_min(0).sqrt() / A
    return total


def _sinograms(case, seed, count):
    """Parallel-beam attenuation sinograms [count][P][D] with counting noise."""
    P, D = case["P"], case["D"]
    th = torch.arange(P, device=DEV)[:, None] * (math.pi / P) + case.get("rotation", 0.0) * math.pi / 180
    s = (torch.arange(D, device=DEV)[None, :] - D // 2) * (WIDTH / D)
    p = _line_integrals(_phantoms(seed, count), s * th.cos(), s * th.sin(), -th.sin() + 0 * s, th.cos() + 0 * s)
    counts = torch.poisson(I0 * torch.exp(-p), generator=_generator(seed, 2))
    return -(counts.clamp_min(1.0) / I0).log()


def _geometry(case):
    import risa_amd

    base = risa_amd.geom_from_config(risa_amd.config_path(case.get("base", "c0")))
    more = {}
    if "rotation" in case:
        more = dict(rotationOffset=case["rotation"], fusedMasking=case["mask"])
    return base.replace(numberOfParallelProjections=case["P"], numberOfParallelDetectors=case["D"],
                        numberOfPixels=case["N"], filterType=case["window"], **more)


def _references(g):
    """A flat field (host arrays, as the handles take them): counts of 8 averaged frames, no dark current."""
    rng = np.random.default_rng(901)
    ref = I0 + rng.standard_normal((g.numberOfPlanes,) + g.fan_shape) * math.sqrt(I0 / 8)
    return ref.astype(np.float32), np.zeros((g.numberOfPlanes, g.numberOfFanDetectors), np.float32)


def _frames(g, seed, count):
    """Raw uint16 fan frames [count][P_f][D_f], up to 8 distinct phantoms, every frame its own noise."""
    Pf, Df = g.fan_shape
    th = (torch.arange(Pf, device=DEV) * (360.0 / Pf) - g.sourceOffset)[:, None] * (math.pi / 180)
    ga = (torch.arange(Df, device=DEV) * (2 * math.pi / Df) + math.pi / 2)[None, :]
    sx, sy = 0.5 * g.sourceDiameter[0] * th.cos(), 0.5 * g.sourceDiameter[0] * th.sin()
    dx, dy = 0.5 * g.detectorDiameter * ga.cos() - sx, 0.5 * g.detectorDiameter * ga.sin() - sy
    length = (dx * dx + dy * dy).sqrt()
    expected = I0 * torch.exp(-_line_integrals(_phantoms(seed, min(count, 8)), sx + 0 * dx, sy + 0 * dx, dx / length,
                                               dy / length))
    gen = _generator(seed, 3)
    raw = torch.empty((count, Pf, Df), dtype=torch.int16, device=DEV)
    for f in range(count):
        n = torch.poisson(expected[f % expected.shape[0]], generator=gen).clamp_max(65535.0)
        raw[f] = n.to(torch.int32).to(torch.int16)   # the low 16 bits
    return raw.view(torch.uint16)


def _planes(g, count):
    return np.arange(count, dtype=np.int32) % g.numberOfPlanes


def _uneven_specs(case):
    rng = random.Random(case["layout"])
    specs = []
    for i in range(case["jobs"]):
        specs.append(dict(N=rng.randint(case["Nmin"], case["Nmax"]), P=rng.randint(case["Pmin"], case["Pmax"]),
                          D=rng.randint(case["Dmin"], case["Dmax"]), f16=i % 2, mask=int(i % 3 != 0),
                          rotation=round(rng.uniform(-45.0, 45.0), 3)))
    return specs


def _filtered_like(spec, seed, i):
    """A sinogram as a ramp filter leaves it (zero mean, sharpened), FP32 or FP16 times X4_SCALE."""
    x = _sinograms(spec, seed + 7919 * i, 1)[0]
    y = x - 0.5 * (x.roll(1, 1) + x.roll(-1, 1))
    y = 0.25 * y / WIDTH * spec["D"]
    return (y * X4_SCALE).half() if spec["f16"] else y


# A program keeps its handles (tables, tuned tile shapes, scratch buffers) for
# as long as the geometry stays the same; so do the states of one case.
_handles = {}


def _kept(case, make):
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _handles:
        if len(_handles) >= 4:
            _handles.clear()
        _handles[key] = make()
    return _handles[key]


def prepare(case, seed):
    from risa_amd import device

    kind = case["kind"]
    if kind == "uneven":
        specs = _uneven_specs(case)
        images = torch.empty(sum(s["N"] ** 2 for s in specs), device=DEV)   # the jobs' images, end to end
        jobs, at = [], 0
        for i, s in enumerate(specs):
            jobs.append(dict(sino=_filtered_like(s, seed, i), img=images[at:at + s["N"] ** 2], N=s["N"], P=s["P"],
                             D=s["D"], dtype=s["f16"], in_scale=X4_SCALE if s["f16"] else 1.0,
                             rotationOffset=s["rotation"], mask=s["mask"], maskingValue=0.0))
            at += s["N"] ** 2
        batch = device.BatchedBackprojection(jobs)
        batch.autotune()
        return dict(kind=kind, batch=batch, images=images, jobs=jobs)
    g = _geometry(case)
    if kind == "chain":
        def make():
            ref, dark = _references(g)
            chain = device.Chain(g, ref, dark, mode=int(case["mode"] == "mixed"), max_frames=case["frames"])
            if case["module"]:
                chain.set_input_layout(1)
            return chain

        n = case["frames"]
        return dict(kind=kind, chain=_kept(case, make), raw=_frames(g, seed, n), planes=_planes(g, n),
                    image=torch.empty((n,) + g.img_shape, device=DEV))
    if kind == "stages":
        def make():
            ref, dark = _references(g)
            bp = device.Backprojection(g)
            bp.autotune()
            return device.Attenuation(g, ref, dark), device.Fan2Para(g), device.Filter(g), bp

        return dict(kind=kind, handles=_kept(case, make), raw=_frames(g, seed, 1)[0],
                    fan=torch.empty(g.fan_shape, device=DEV), sinogram=torch.empty(g.par_shape, device=DEV),
                    image=torch.empty(g.img_shape, device=DEV))

    def make():
        bp = device.Backprojection(g)
        bp.autotune_batch(case["slices"])
        return device.Filter(g), bp

    filt, bp = _kept(case, make)
    S = case["slices"]
    x = _sinograms(case, seed, S)
    state = dict(kind=kind, filter=filt, bp=bp, slices=S, x=x, sinogram=torch.empty_like(x))
    if kind == "forward":
        state["image"] = torch.empty((S,) + g.img_shape, device=DEV)
    else:
        # the gradient of a squared difference: image-like values and noise
        state["image"] = torch.randn((S,) + g.img_shape, generator=_generator(seed, 4), device=DEV) * 1e-2
        state["taps"] = torch.empty(case["D"] // 2 + 1, device=DEV)
    return state


# --------------------------------------------------------------------- run --
def run(state):
    kind = state["kind"]
    if kind == "chain":
        return state["chain"](state["raw"], state["planes"], state["image"])
    if kind == "stages":
        attenuation, rebinning, filt, bp = state["handles"]
        attenuation(state["raw"], 0, state["fan"])
        rebinning(state["fan"], 0, state["sinogram"])
        filt(state["sinogram"], 1)
        return bp(state["sinogram"], state["image"])
    if kind == "forward":
        state["sinogram"].copy_(state["x"])
        state["filter"](state["sinogram"], state["slices"])
        return state["bp"].batch(state["sinogram"], state["slices"], state["image"])
    if kind == "backward":
        state["bp"].adjoint_batch(state["image"], state["slices"], state["sinogram"])
        state["filter"].grad_taps(state["x"], state["sinogram"], state["slices"], state["taps"])
        state["filter"].adjoint(state["sinogram"], state["slices"])
        return state["sinogram"], state["taps"]
    state["batch"]()
    return state["images"]


# -------------------------------------------------------------------- work --
FLOP_PER_UPDATE = 10   # coordinate, two weights, two multiply-adds


def _inside(N, mask):
    return int(math.pi / 4 * N * N) if mask else N * N


def work(case):
    kind = case["kind"]
    if kind == "uneven":
        specs = _uneven_specs(case)
        return dict(bytes=float(sum((2 if s["f16"] else 4) * s["P"] * s["D"] + 4 * s["N"] ** 2 for s in specs)),
                    flops=float(sum(FLOP_PER_UPDATE * _inside(s["N"], s["mask"]) * s["P"] for s in specs)))
    P, D, N = case["P"], case["D"], case["N"]
    fft = 10.0 * D * math.log2(D)   # a row's transform, response and inverse
    if kind in ("chain", "stages"):
        Pf, Df, planes = (500, 432, 1) if case["base"] == "c0" else (1000, 768, 2)
        n = case.get("frames", 1)
        planes = min(planes, n)
        return dict(bytes=float(n * (2 * Pf * Df + 4 * N * N) + planes * 4 * Pf * Df),
                    flops=float(n * (FLOP_PER_UPDATE * _inside(N, True) * P + fft * P)))
    S = case["slices"]
    updates = S * P * (FLOP_PER_UPDATE * _inside(N, case["mask"]) + fft)
    if kind == "forward":
        return dict(bytes=float(S * 4 * (P * D + N * N)), flops=float(updates))
    return dict(bytes=float(S * 4 * (2 * P * D + N * N) + 4 * (D // 2 + 1)), flops=float(updates + S * P * fft))


# ------------------------------------------------- the same in 64 bits --
def _taps(D, window, cutoff=1.0):
    i = np.arange(1, D // 2 + 1)
    w = 2 * math.pi * i / D
    v = 2.0 * i / D
    name = WINDOWS[window]
    if name == "sheppLogan":
        v = v * np.sin(w / (2 * cutoff)) / (w / (2 * cutoff))
    elif name == "cosine":
        v = v * np.cos(w / (2 * cutoff))
    elif name == "hamming":
        v = v * (0.54 + 0.46 * np.cos(w / cutoff))
    elif name == "hanning":
        v = v * (1 + np.cos(w / cutoff)) / 2
    h = np.concatenate([[0.0], v / D])
    if D % 2 == 0:
        h[-1] = 0.0   # the Nyquist tap drops: float(pi) > pi
    return torch.from_numpy(h).to(DEV)


def _filter64(x, taps):
    D = x.shape[-1]
    return torch.fft.irfft(torch.fft.rfft(x) * taps, n=D) * D


def _angles(P, rotation):
    return [i * math.pi / P + rotation / 180.0 * math.pi for i in range(P)]


def _disk(N, mask):
    c = torch.arange(N, device=DEV, dtype=torch.float64) - (N - 1) * 0.5
    inside = (c[None, :] ** 2 + c[:, None] ** 2 <= N * N * 0.25) if mask else torch.ones((N, N), dtype=torch.bool, device=DEV)
    y, x = torch.nonzero(inside, as_tuple=True)
    return x, y, c[x], c[y]


def _bins(px, py, th, scale, D):
    """Padded sample index (0 and D + 1 are outside) and fraction of every pixel."""
    t = (px * math.cos(th) + py * math.sin(th)) * scale
    k = t.floor()
    f = t - k
    k = k.long() + int(D * 0.5)
    return (k + 1).clamp(0, D + 1), (k + 2).clamp(0, D + 1), f


def _backproject64(sino, N, rotation, mask):
    S, P, D = sino.shape
    x, y, px, py = _disk(N, mask)
    rows = torch.zeros((P, D + 2, S), dtype=torch.float64, device=DEV)
    rows[:, 1:D + 1] = sino.permute(1, 2, 0)
    acc = torch.zeros((px.numel(), S), dtype=torch.float64, device=DEV)
    for a, th in enumerate(_angles(P, rotation)):
        k0, k1, f = _bins(px, py, th, D / N, D)
        acc.addcmul_(rows[a][k0], (1 - f)[:, None]).addcmul_(rows[a][k1], f[:, None])
    img = torch.zeros((S, N, N), dtype=torch.float64, device=DEV)
    img[:, y, x] = (acc * (math.pi / P / (D / N))).T
    return img


def _project64(img, P, D, rotation, mask):
    """The transpose of _backproject64."""
    S, N, _ = img.shape
    x, y, px, py = _disk(N, mask)
    v = img[:, y, x].T.double().contiguous()
    out = torch.zeros((P, D + 2, S), dtype=torch.float64, device=DEV)
    for a, th in enumerate(_angles(P, rotation)):
        k0, k1, f = _bins(px, py, th, D / N, D)
        out[a].index_add_(0, k0, v * (1 - f)[:, None]).index_add_(0, k1, v * f[:, None])
    return out[:, 1:D + 1].permute(2, 0, 1) * (math.pi / P / (D / N))


def _area_mask(g):
    """Attenuation.cu:327-381: the relevant detectors of every source angle."""
    Pf, D = g.fan_shape
    mask = np.ones((Pf, D))
    lo, hi = (g.lowerLimOffset + g.sourceOffset) / 360.0, (g.upperLimOffset + g.sourceOffset) / 360.0

    def half_up(v):   # round half away from zero, to an unsigned 32-bit number
        return int(math.copysign(math.floor(abs(v) + 0.5), v)) & 0xFFFFFFFF

    ya, yc = half_up(lo * Pf), half_up(hi * Pf)
    m = (ya - yc) / (g.xa - g.xd)
    ye = half_up(yc + (g.xe - g.xc) * m)

    def clear(x, y0, y1):
        flat = mask.reshape(-1)
        at = x + np.arange(y0, min(y1, Pf + 1), dtype=np.int64) * D
        flat[at[at < flat.size]] = 0.0

    for x in range(0, g.xa + 1):
        clear(x, ya, half_up(ye + m * x))
    for x in range(g.xa, g.xc + 1):
        clear(x, half_up(ya + m * (x - g.xa)), half_up(ye + m * x))
    for x in range(g.xc, g.xd + 1):
        clear(x, half_up(ya + m * (x - g.xa)), yc)
    for x in range(g.xb, g.xf + 1):
        clear(x, ya, half_up(ya + m * (x - g.xb)))
    flat = mask.reshape(-1)
    flat[:max(0, int(lo * D * Pf))] = 0.0
    flat[max(0, int(hi * Pf * D)):] = 0.0
    return mask


def _ring_angle(alpha, dx, dz, diameter):
    """cuda_kernels_fan2para.h:38-62: an in-plane source angle on the tilted source ring, in alpha's type."""
    real = alpha.dtype.type

    def r(v):   # the reference keeps its angles in one type and evaluates the roots in double
        return np.asarray(v).astype(real)

    dx, dz = real(dx), real(dz)
    L, R, ca = r(np.sqrt(dx * dx + dz * dz)), real(0.5 * diameter), np.cos(alpha)
    d = np.float64

    def acos(v):
        return np.arccos(np.clip(r(v), real(-1), real(1)))

    eps = acos((L * L + R * dx * ca).astype(d) / (d(L) * np.sqrt(d(L * L + R * R) + 2.0 * R * dx * ca.astype(d))))
    p1 = acos(d(L * L - R * dx) / (d(L) * np.sqrt(d(L * L + R * R) - 2.0 * d(R) * d(dx))))
    p2 = acos(d(L * L + R * dx) / (d(L) * np.sqrt(d(L * L + R * R) + 2.0 * d(R) * d(dx))))
    gam = real(0.5 * d(p1 - p2))
    ae = acos((eps * ca + gam).astype(d) / np.sqrt((eps * eps).astype(d) + 2.0 * eps.astype(d) * gam * ca + d(gam * gam)))
    return np.where(alpha.astype(d) <= math.pi, ae, r(2.0 * math.pi - ae.astype(d)))


def _goals(g, plane, real):
    """Goal angles (theta, gamma) of the two rays of every internal sample (j, i), j < 2 P, evaluated in `real`."""
    P2, D = 2 * g.numberOfParallelProjections, g.numberOfParallelDetectors
    d, two_pi = np.float64, 2 * math.pi

    def r(v):
        return np.asarray(v).astype(real)

    alpha = r((two_pi / 360) * r(np.arange(P2) * (360.0 / P2)).astype(d) + math.pi / 2)
    alpha = np.where(alpha.astype(d) > two_pi, r(alpha.astype(d) - two_pi), alpha)
    alpha[0] = 0
    alpha = alpha[:, None]
    s = r(-0.5 * g.imageWidth + ((0.5 + np.arange(D)) * g.imageWidth) / D)[None, :]
    rD, rT = real(g.detectorDiameter / 2), real(g.sourceDiameter[plane] / 2)
    turn = np.arcsin(s / rT)
    with np.errstate(invalid="ignore"):
        eps = np.arcsin(s / rD)
    goals = []
    for ray in (0, 1):
        t = alpha - turn if ray == 0 else r((alpha + turn).astype(d) - math.pi)
        t = np.where(t < 0, r(t.astype(d) + two_pi), t)
        t = _ring_angle(t, g.deltaX[plane], g.deltaZ[plane], 2 * d(rT))
        gg = r((eps + alpha).astype(d) - 1.5 * math.pi) if ray == 0 else r((alpha - eps).astype(d) - 0.5 * math.pi)
        gg = np.where(gg < 0, r(gg.astype(d) + two_pi), gg)
        goals.append((t, np.where(gg.astype(d) > two_pi, r(gg.astype(d) - two_pi), gg)))
    return goals, np.abs(s / rD) <= 1


def _rebin_rays(g, plane):
    """The two rays of every internal sample: (valid, four flat fan indices, f_theta, f_gamma).

    Which rays and samples a point takes is decided in single precision, as the
    reference's host code decides it (Fan2Para.cu:286-480); the weights are
    float64."""
    Pf, Df = g.fan_shape
    d, two_pi = np.float64, 2 * math.pi

    def axes(real):
        v = (np.arange(Pf) * (360.0 / Pf) - d(real(g.sourceOffset))).astype(real)
        v = np.where(v < 0, (v.astype(d) + 360.0).astype(real), v)
        theta = ((two_pi / 360) * v.astype(d)).astype(real)
        return theta, ((two_pi / 360) * (np.arange(Df) * (360.0 / Df)).astype(real).astype(d)).astype(real)

    theta32, gamma32 = axes(np.float32)
    theta, gamma = axes(d)
    order = np.argsort(theta32, kind="stable")
    goals32, in_range = _goals(g, plane, np.float32)
    goals, _ = _goals(g, plane, d)
    half = (360.0 - g.sourceAngle[plane]) / 2
    lim1, lim2 = np.float32(half / 180 * math.pi), np.float32((360.0 - half) / 180 * math.pi)
    rays = []
    for (t32, g32), (t, gg) in zip(goals32, goals):
        valid = in_range & (t32 > lim1) & (t32 < lim2)
        ta = order[np.minimum(np.searchsorted(theta32[order], t32), Pf - 1)]
        tb = (ta - 1) % Pf
        gx = np.searchsorted(gamma32, g32)   # the first gamma >= the goal; past the end: (D_f - 1, 0)
        ga, gb = gx % Df, (gx - 1) % Df
        # the goal at the turn its single-precision value has
        t = t + two_pi * np.rint((t32 - t) / two_pi)
        gg = gg + two_pi * np.rint((g32 - gg) / two_pi)
        ft = (t - theta[tb]) / (theta[ta] - theta[tb])
        fg = (gg - gamma[gb]) / (gamma[ga] - gamma[gb])
        flat = [np.where(valid, a * Df + b, 0) for a in (tb, ta) for b in (gb, ga)]
        rays.append((torch.from_numpy(np.broadcast_to(valid, t.shape).copy()).to(DEV),
                     [torch.from_numpy(f).to(DEV) for f in flat],
                     torch.from_numpy(np.where(valid, ft, 0.0)).to(DEV), torch.from_numpy(np.where(valid, fg, 0.0)).to(DEV)))
    return rays


def _fold_odd(out, second, D):
    """Odd D: output i > h takes sample 2h - i, i < h takes 2h - 1 - i, and h - 1 also takes D - 1
    (cuda_kernels_fan2para.h:164-176)."""
    h = D // 2
    i = torch.arange(D, device=DEV)
    src = torch.where(i > h, 2 * h - i, 2 * h - 1 - i)
    keep = i != h
    out[:, :, keep] += second[:, :, src[keep]]
    out[:, :, h - 1] += second[:, :, D - 1]
    return out


def _rebin64(g, fan, rays):
    """fan [F][P_f D_f] -> [F][P][D]: each sample the mean of its valid rays, folded onto 180 degrees."""
    P, D = g.par_shape
    z = []
    for valid, (i00, i01, i10, i11), ft, fg in rays:
        lo = fan[:, i00] + ft * (fan[:, i10] - fan[:, i00])
        hi = fan[:, i01] + ft * (fan[:, i11] - fan[:, i01])
        z.append(torch.where(valid, lo + fg * (hi - lo), torch.zeros((), dtype=torch.float64, device=DEV)))
    count = rays[0][0].double() + rays[1][0].double()
    Z = 0.5 * (z[0] + z[1]) / count.clamp_min(1.0)
    return Z[:, :P] + Z[:, P:].flip(2) if D % 2 == 0 else _fold_odd(Z[:, :P].clone(), Z[:, P:], D)


def _chain64(case, raw, planes):
    g = _geometry(case)
    P, D = g.par_shape
    Pf, Df = g.fan_shape
    ref, dark = _references(g)
    mask = torch.from_numpy(_area_mask(g)).to(DEV)
    taps = _taps(D, case["window"])
    order = None
    if case.get("module"):
        # Reordering.cu:180-204: 27 modules x P_f x 16 -> [P_f][432]; past those samples, sample 0
        i = torch.arange(Pf * Df, device=DEV)
        p, r = i // 432, i % 432
        order = torch.where(i < Pf * 432, r % 16 + p * 16 + (r // 16) * 16 * Pf, torch.zeros_like(i))
    tables = {k: _rebin_rays(g, k) for k in sorted(set(int(k) for k in planes))}
    images = []
    for f0 in range(0, raw.shape[0], 16):
        sinos = []
        for f in range(f0, min(raw.shape[0], f0 + 16)):
            k = int(planes[f])
            counts = (raw[f].view(torch.int16).to(torch.int32) & 0xFFFF).double().reshape(-1)
            if order is not None:
                counts = counts[order]
            den = torch.from_numpy(ref[k].astype(np.float64) - dark[k]).to(DEV).clamp_min(1e-5)
            att = -torch.log(counts.reshape(Pf, Df).clamp_min(1e-5) / den) * mask
            sinos.append(_rebin64(g, att.reshape(1, -1), tables[k])[0])
        images.append(_backproject64(_filter64(torch.stack(sinos), taps), case["N"], g.rotationOffset, True))
    return torch.cat(images)


def exact(case, seed):
    kind = case["kind"]
    if kind == "uneven":
        images = []
        for i, s in enumerate(_uneven_specs(case)):
            x = _filtered_like(s, seed, i).double()
            x = x / X4_SCALE if s["f16"] else x
            images.append(_backproject64(x[None], s["N"], s["rotation"], bool(s["mask"])).reshape(-1))
        return torch.cat(images)
    if kind in ("chain", "stages"):
        g = _geometry(case)
        n = case.get("frames", 1)
        img = _chain64(case, _frames(g, seed, n), _planes(g, n))
        return img if kind == "chain" else img[0]
    taps = _taps(case["D"], case["window"])
    x = _sinograms(case, seed, case["slices"]).double()
    if kind == "forward":
        return _backproject64(_filter64(x, taps), case["N"], case["rotation"], bool(case["mask"]))
    D = case["D"]
    img = torch.randn((case["slices"], case["N"], case["N"]), generator=_generator(seed, 4), device=DEV) * 1e-2
    back = _project64(img, case["P"], D, case["rotation"], bool(case["mask"]))
    X, G = torch.fft.rfft(x), torch.fft.rfft(back)
    grad = (G.conj() * X).real.sum((0, 1))
    w = torch.full_like(grad, 2.0)
    w[0] = 1.0
    if D % 2 == 0:
        w[-1] = 1.0
    return _filter64(back, taps), grad * w
