"""The work that programs on this framework have it do, as cases that can be timed.

Sizes and value distributions follow the repository's workloads and benchmark
(planes of points with 7.56 and 10 um pitch, 632.8 nm, 0.35 m, a plane
generator that leaves copies of point 0, pixels jittered by up to 0.4875
pitch, distances of 2 to 50 cm).  FP64 fields stay complex128.  Fields of the
FP32-split formulation, whose pairs are FP32, are kept by their users as
complex64, and a hologram's phases are an FP32 parameter as torch's are.
"""
import math

import numpy as np
import torch

import __graft_entry__

holo = __graft_entry__.load_package()
from holo_amd import hologram as hologram_module  # noqa: E402
from holo_amd import torch_ops, workloads  # noqa: E402

LAM = workloads.LAMBDA_HENE
EXACT_PAIRS = 1e11  # about 8 s of plain torch


def listed():
    return [
        # the smallest program: 32 x 32 points on a 64 x 64 plane, one FP64 call; its latency
        dict(name="f64_smallest", kind="field", precision="f64", src="lattice", nx=32, ny=32,
             mx=64, my=64, z=0.35, sign=1, obliquity=False),
        # an object of a thousand points in depth onto a projector: few sources, many targets
        dict(name="f64_object", kind="field", precision="f64", src="object", nx=1031, ny=1,
             mx=720, my=1280, z=0.35, sign=1, obliquity=False),
        # object plane -> projector -> image plane, each field normalised to polar form
        dict(name="f64_chain", kind="chain", precision="f64", nx=256, ny=256, mx=512, my=512,
             z=0.35),
        # the reference's own call, on host arrays: a small plane, forwards, polar result
        dict(name="f64_host", kind="host", precision="f64", nx=96, ny=80, mx=200, my=150, z=0.35,
             sign=1),
        # a small plane kept as a plan and evaluated again and again: launches count
        dict(name="f32_small", kind="plan", precision="f32", src="lattice", nx=64, ny=64, mx=64,
             my=64, z=0.35, sign=1, obliquity=False),
        # the full projector plane, the benchmark's FP32-split case
        dict(name="f32_plane", kind="plan", precision="f32", src="lattice", nx=1024, ny=1024,
             mx=1024, my=1024, z=0.35, sign=1, obliquity=False),
        # planes of the reference's generator with point counts that are no product
        dict(name="f32_generator", kind="plan", precision="f32", src="generator", nx=300001, ny=1,
             mx=200003, my=1, z=0.35, sign=-1, obliquity=False),
        # near field: the short distances of the reference's sweeps
        dict(name="f32_near", kind="plan", precision="f32", src="lattice", nx=512, ny=512, mx=512,
             my=512, z=0.1, sign=1, obliquity=False),
        # jittered pixels (the reference's -r): no lattice
        dict(name="f32_jittered", kind="plan", precision="f32", src="jittered", nx=400, ny=400,
             mx=512, my=512, z=0.35, sign=1, obliquity=False),
        # one call on new positions, with the obliquity factor: the plan is part of it
        dict(name="f32_one_shot", kind="field", precision="f32", src="lattice", nx=512, ny=512,
             mx=512, my=512, z=0.35, sign=-1, obliquity=True),
        # a phase-only hologram's training step: forward field, loss, adjoint
        dict(name="hologram_step", kind="hologram", precision="f32", nx=1024, ny=1024, mx=512,
             my=512, z=0.35),
        # Monte Carlo: 1024 draws per target from the full plane
        dict(name="mc_plane", kind="mc", precision="f32", src="lattice", nx=1024, ny=1024,
             mx=1024, my=1024, z=0.35, K=1024, shared=False, sign=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sides(rng, most):
    """Two sides from 16 up, odd ones among them, with at most `most` points."""
    a = _log(rng, 16, 1024)
    b = min(_log(rng, max(16, a // 3), min(3 * a, 1024)), max(16, most // a))
    return a, b


def draw(rng):
    kind = rng.choice(["f64", "f64", "object", "chain", "host", "plan", "plan", "plan",
                       "generator", "jittered", "one_shot", "hologram", "mc", "mc_shared"])
    sign = rng.choice([1, -1])
    if kind == "object":
        n = _log(rng, 1, 4096)
        mx, my = _sides(rng, 1 << 20)
        return dict(kind="field", precision="f64", src="object", nx=n, ny=1, mx=mx, my=my,
                    z=rng.uniform(0.1, 0.5), sign=sign, obliquity=rng.random() < 0.2)
    # the largest drawn call has 3e10 pairs in FP64 and off the lattice, 4e11 on it
    fast = kind in ("plan", "generator", "one_shot", "hologram")
    nx, ny = _sides(rng, 1 << 20)
    pairs = 4e11 if fast else 3e10
    mx, my = _sides(rng, max(256, int(min(1 << 20, pairs / (nx * ny)))))
    far = rng.uniform(0.2, 0.5)
    if kind == "f64":
        src = rng.choice(["lattice", "generator", "jittered"])
        if src == "generator":
            nx, ny, mx, my = nx * ny + rng.randrange(8), 1, mx * my + rng.randrange(8), 1
        return dict(kind="field", precision="f64", src=src, nx=nx, ny=ny, mx=mx, my=my,
                    z=math.exp(rng.uniform(math.log(0.02), math.log(0.5))), sign=sign,
                    obliquity=rng.random() < 0.3)
    if kind == "chain":
        return dict(kind="chain", precision="f64", nx=nx, ny=ny, mx=mx, my=my, z=far)
    if kind == "host":
        nx, ny, mx, my = min(nx, 160), min(ny, 160), min(mx, 256), min(my, 256)
        return dict(kind="host", precision="f64", nx=nx, ny=ny, mx=mx, my=my, z=far, sign=sign)
    if kind == "plan":
        z = far if rng.random() < 0.6 else math.exp(rng.uniform(math.log(0.02), math.log(0.2)))
        while z < 0.2 and nx * ny * mx * my > 7e10:
            nx, mx = max(16, nx // 2), max(16, mx // 2)
        return dict(kind="plan", precision="f32", src="lattice", nx=nx, ny=ny, mx=mx, my=my, z=z,
                    sign=sign, obliquity=rng.random() < 0.3)
    if kind == "generator":
        return dict(kind="plan", precision="f32", src="generator", nx=nx * ny + rng.randrange(9),
                    ny=1, mx=mx * my + rng.randrange(9), my=1, z=far, sign=sign, obliquity=False)
    if kind == "jittered":
        return dict(kind="plan", precision="f32", src="jittered", nx=nx, ny=ny, mx=mx, my=my,
                    z=math.exp(rng.uniform(math.log(0.05), math.log(0.5))), sign=sign,
                    obliquity=rng.random() < 0.3)
    if kind == "one_shot":
        return dict(kind="field", precision="f32", src=rng.choice(["lattice", "generator"]),
                    nx=nx, ny=ny, mx=mx, my=my, z=far, sign=sign, obliquity=rng.random() < 0.5)
    if kind == "hologram":
        return dict(kind="hologram", precision="f32", nx=nx, ny=ny, mx=mx, my=my, z=far)
    K = _log(rng, 16, 4096)
    mx, my = _sides(rng, max(256, int(min(1 << 20, 1e9 / K))))
    return dict(kind="mc", precision="f32", src=rng.choice(["lattice", "jittered"]), nx=nx, ny=ny,
                mx=mx, my=my, z=far, K=K, shared=kind == "mc_shared", sign=sign)


# ---- inputs -----------------------------------------------------------------------


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(_device())


def _plane(nx, ny, pitch, z):
    """The product lattice of workloads.grid, made on the device."""
    d = _device()
    ix = (torch.arange(nx, dtype=torch.float64, device=d) - (nx - 1) / 2.0) * pitch
    iy = (torch.arange(ny, dtype=torch.float64, device=d) - (ny - 1) / 2.0) * pitch
    u = torch.empty((nx, ny, 3), dtype=torch.float64, device=d)
    u[..., 0], u[..., 1], u[..., 2] = ix[:, None], iy[None, :], z
    return u.reshape(-1, 3)


def _uniform(gen, n):
    return torch.rand(n, dtype=torch.float64, device=_device(), generator=gen)


def _geometry(case, gen):
    """Sources at z = 0 (objects at depths about it), targets at the plane z."""
    nx, ny, mx, my, z = case["nx"], case["ny"], case["mx"], case["my"], case["z"]
    src = case.get("src", "lattice")
    if src == "generator":
        u = _dev(workloads.reference_plane(nx * ny, math.sqrt(nx * ny) * 10e-6, 0.0))
        v = _dev(workloads.reference_plane(mx * my, math.sqrt(mx * my) * 7.56e-6, z))
        return u, v
    v = _plane(mx, my, 7.56e-6, z)
    if src == "object":  # a circle of points, each at its own depth
        t = _uniform(gen, nx) * (2 * math.pi)
        u = torch.stack([2e-3 * torch.cos(t), 2e-3 * torch.sin(t),
                         (_uniform(gen, nx) - 0.5) * 0.02], dim=1)
        return u.contiguous(), v
    u = _plane(nx, ny, 10e-6, 0.0)
    if src == "jittered":
        u[:, :2] += (torch.rand((nx * ny, 2), dtype=torch.float64, device=_device(),
                                generator=gen) - 0.5) * (2 * 0.4875 * 10e-6)
    return u, v


def _inputs(case, seed):
    gen = torch.Generator(device=_device()).manual_seed(int(seed))
    u, v = _geometry(case, gen)
    n, m = u.shape[0], v.shape[0]
    if case["kind"] == "hologram":  # FP32 phases, a bright spots' target image
        theta = (_uniform(gen, n) * (2 * math.pi)).to(torch.float32)
        image = _uniform(gen, m) ** 8
        return u, v, torch.ones(n, dtype=torch.float32, device=u.device), theta, image / image.mean()
    return u, v, _uniform(gen, n), _uniform(gen, n) * (2 * math.pi), None


def prepare(case, seed):
    u, v, amp, phase, image = _inputs(case, seed)
    s = dict(case=case, u=u, v=v, amp=amp, phase=phase,
             precision=holo.FP64 if case["precision"] == "f64" else holo.FP32_SPLIT)
    kind = case["kind"]
    if kind == "host":
        s.update(x=torch.stack([amp, phase], dim=1).cpu().numpy(), u=u.cpu().numpy(),
                 v=v.cpu().numpy(), ctx=holo.Context(0))
        return s
    s["ctx"] = holo.Context(0)
    if kind == "plan":
        s["plan"] = s["ctx"].plan(u)
    elif kind == "chain":
        s["w"] = _plane(case["nx"], case["ny"], 10e-6, 0.0)
    elif kind == "hologram":
        s.update(prop=torch_ops.Propagator(u, v, +1, LAM, holo.FP32_SPLIT, ctx=s["ctx"]),
                 theta=phase.requires_grad_(True), image=image)
    return s


def run(s):
    case, ctx, kind = s["case"], s["ctx"], s["case"]["kind"]
    if kind == "field":
        y = ctx.transform_full(s["amp"], s["phase"], s["u"], s["v"], case["sign"], LAM,
                               s["precision"], obliquity=case["obliquity"])
        return y if case["precision"] == "f64" else y.to(torch.complex64)
    if kind == "plan":
        y = s["plan"].transform(s["amp"], s["phase"], s["v"], case["sign"], LAM, s["precision"],
                                obliquity=case["obliquity"])
        return y.to(torch.complex64)
    if kind == "chain":
        y = ctx.transform_full(s["amp"], s["phase"], s["u"], s["v"], +1, LAM, s["precision"])
        ya, yp, _ = ctx.normalize_polar(y)
        z = ctx.transform_full(ya, yp, s["v"], s["w"], -1, LAM, s["precision"])
        za, zp, zmax = ctx.normalize_polar(z)
        return {"y_amp": ya, "y_phase": yp, "z_amp": za, "z_phase": zp, "z_max": zmax}
    if kind == "host":
        polar, _ = holo.time_transform(s["x"], s["u"], s["v"], holo.Direction(case["sign"]),
                                       lam=LAM, precision=s["precision"], ctx=ctx)
        return polar
    if kind == "hologram":
        theta = s["theta"]
        theta.grad = None
        z = s["prop"](s["amp"], theta)
        hologram_module.intensity_loss(z, s["image"]).backward()
        return {"field": z.detach().to(torch.float32), "grad": theta.grad}
    y = ctx.transform_mc(s["amp"], s["phase"], s["u"], s["v"], case["K"], 7, case["sign"], LAM,
                         s["precision"], shared=case["shared"])
    return y.to(torch.complex64)


def work(case):
    """Every pair once, 29 operations each as the reference counts them; positions, weights and
    results moved once."""
    n, m = case["nx"] * case["ny"], case["mx"] * case["my"]
    pairs = m * case["K"] if case["kind"] == "mc" else n * m
    w = 8 if case["kind"] == "hologram" else 16
    out = 16 if case["precision"] == "f64" else 8
    b = (24 + w) * n + (24 + out) * m
    if case["kind"] == "chain":
        pairs, b = 2 * pairs, 2 * b
    if case["kind"] == "hologram":
        pairs, b = 2 * pairs, b + 8 * m + 4 * n
    return {"bytes": float(b), "flops": 29.0 * pairs}


# ---- the same in plain torch, 64 bits -----------------------------------------------


def _sum(u, w, v, sign, obliquity):
    """sum_n w_n exp(i sign 2 pi d / lambda) / d at every target."""
    out = torch.empty(v.shape[0], dtype=torch.complex128, device=v.device)
    step = max(1, int(6e7) // u.shape[0])
    wr, wi = w.real.contiguous(), w.imag.contiguous()
    for a in range(0, v.shape[0], step):
        t = v[a:a + step]
        d2 = (t[:, None, 0] - u[None, :, 0]) ** 2
        d2 += (t[:, None, 1] - u[None, :, 1]) ** 2
        dz = t[:, None, 2] - u[None, :, 2]
        d2 += dz ** 2
        d = d2.sqrt_()
        arg = d * (sign * 2 * math.pi / LAM)
        g = 1.0 / d
        if obliquity:
            g *= dz.abs() * g
        c = torch.cos(arg) * g
        s = arg.sin_() * g
        out[a:a + step] = torch.complex(c @ wr - s @ wi, c @ wi + s @ wr)
    return out


def _philox(c0, c1, c2, c3, k0, k1):
    """Philox4x32-10 on int64 tensors that hold 32-bit words."""
    low = 0xFFFFFFFF

    def mul(a, b):  # the 64-bit product of a constant and a word, as (high, low)
        bl, bh = b & 0xFFFF, b >> 16
        p0, p1 = a * bl, a * bh
        t = p0 + ((p1 & 0xFFFF) << 16)
        return (p1 >> 16) + (t >> 32), t & low

    for _ in range(10):
        h0, l0 = mul(0xD2511F53, c0)
        h1, l1 = mul(0xCD9E8D57, c2)
        c0, c1, c2, c3 = h1 ^ c1 ^ k0, l1, h0 ^ c3 ^ k1, l0
        k0, k1 = (k0 + 0x9E3779B9) & low, (k1 + 0xBB67AE85) & low
    return c0, c1, c2, c3


def _indices(lo, hi, n):
    return (hi * n + ((lo * n) >> 32)) >> 32


def _mc(case, u, w, v):
    n, m, K = u.shape[0], v.shape[0], case["K"]
    k = torch.arange((K + 1) // 2, device=v.device)
    out = torch.empty(m, dtype=torch.complex128, device=v.device)
    zero = torch.zeros((), dtype=torch.int64, device=v.device)
    step = max(1, int(3e7) // K)
    for a in range(0, m, step):
        t = v[a:a + step]
        rows = torch.arange(a, min(m, a + step), device=v.device)
        if case["shared"]:
            who, c2 = rows // 1024, zero + 0x80000000
        else:
            who, c2 = rows, zero
        x, y, z, q = _philox(k[None, :] + 0 * who[:, None], who[:, None] + 0 * k[None, :], c2,
                             zero + 0x4D43, 7, 0)
        i = torch.stack([_indices(x, y, n), _indices(z, q, n)], dim=2).reshape(t.shape[0], -1)[:, :K]
        p = u[i]
        d = ((t[:, None, :] - p) ** 2).sum(-1).sqrt_()
        arg = d * (case["sign"] * 2 * math.pi / LAM)
        out[a:a + step] = (w[i] * torch.polar(1.0 / d, arg)).sum(1) * (n / K)
    return out


def _polar(y):
    top = y.abs().max()
    y = y / top if top >= 1e-6 else y
    return y.abs(), y.angle(), top


def exact(case, seed):
    pairs = work(case)["flops"] / 29
    if pairs > EXACT_PAIRS:
        return None
    u, v, amp, phase, image = _inputs(case, seed)
    w = torch.polar(amp.double(), phase.double())
    kind = case["kind"]
    if kind in ("field", "plan"):
        return _sum(u, w, v, case["sign"], case["obliquity"])
    if kind == "chain":
        ya, yp, _ = _polar(_sum(u, w, v, +1, False))
        za, zp, zmax = _polar(_sum(v, torch.polar(ya, yp), _plane(case["nx"], case["ny"], 10e-6, 0.0),
                                   -1, False))
        return {"y_amp": ya, "y_phase": yp, "z_amp": za, "z_phase": zp, "z_max": zmax.reshape(1)}
    if kind == "host":
        a, p, _ = _polar(_sum(u, w, v, case["sign"], False))
        return torch.stack([a, p], dim=1)
    if kind == "hologram":
        z = torch.view_as_real(_sum(u, w, v, +1, False)).requires_grad_(True)
        hologram_loss = torch.mean(((z ** 2).sum(1) / (z ** 2).sum(1).mean() - image) ** 2)
        (g,) = torch.autograd.grad(hologram_loss, z)
        b = _sum(v, torch.view_as_complex(g.contiguous()), u, -1, False)
        return {"field": z.detach(), "grad": amp.double() * (w.conj() * b).imag}
    return _mc(case, u, w, v)
