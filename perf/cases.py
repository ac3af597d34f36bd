"""Timing cases of the framework: what its users have it do, through its public entry points.

A case is a dict of plain values.  ``kind`` names the call:

    radon            Plan.radon of a stack of images (R, A layout)
    backprojection   Plan.backprojection of a stack of sinograms
    fbp              Plan.fbp of a stack of sinograms
    osem             Plan.em: ordered-subsets EM of one or more slices
    osem_batch       Batch.em: OSEM of slices of different sizes in one call
    grad             autograd.radon and its gradient for a weighted least-squares loss
    mesh_radon       Plan.mesh(...).radon on arbitrary detector and angle tables
    line_radon       DdaPlan.radon (line traversal, pyraft's default projector)
    line_backprojection  DdaPlan.backprojection (its normalised backprojection)
    numpy_fbp        pyraft_amd.fbp_gpu on a host sinogram, as a pyraft program calls it (the
                     image has the detector's size)

Images and sinograms are sums of random ellipses (the sinograms in closed form).  The EM
data are Poisson counts of a region of interest: the body reaches past the field, so that
no ray is empty (a view of nothing has no stable ratio of measured to expected counts).
``n`` is the image side, ``rays`` the detector bins, ``angles`` the views, ``slices`` the
images of one call; ``arc`` is the angular range, ``half`` the detector's half width and
``shift`` the offset of its centre from the rotation axis (the image spans [-1, 1]^2).
"""
import math

import numpy
import torch

import pyraft_amd
from pyraft_amd import autograd, batch, device

IMG = (-1.0, 1.0, 1.0, -1.0)


def _case(kind, n, rays, angles, slices=1, **more):
    out = dict(kind=kind, n=n, rays=rays, angles=angles, slices=slices, arc=math.pi, half=1.0, shift=0.0)
    out.update(more)
    return out


def listed():
    return [
        # the reference's own demonstration size: one slice, launch and call latency
        dict(_case("radon", 256, 256, 180), name="radon_256"),
        # the same size, filtered backprojection (a preview of one slice)
        dict(_case("fbp", 256, 256, 180), name="fbp_256"),
        # a few slices of a detector that is neither a power of two nor the image's size
        dict(_case("fbp", 363, 517, 271, slices=3, half=1.42), name="fbp_odd"),
        # a full-resolution parallel-beam slice, forward: simulation, the residual of a solver
        dict(_case("radon", 2048, 2048, 1500), name="radon_2048"),
        # the same slice backwards, on a plan that was tuned as a production program does
        dict(_case("backprojection", 2048, 2048, 1500, tune=True), name="backprojection_2048"),
        # iterative reconstruction of one slice: two iterations of 16 subsets
        dict(_case("osem", 1024, 1024, 720, subsets=16, niter=2), name="osem_1024"),
        # slices of several scans in one call, sizes and views uneven
        dict(_case("osem_batch", 768, 768, 500, slices=12, subsets=8, niter=1), name="osem_batch"),
        # one training step of a learned reconstruction: projector, loss, gradient
        dict(_case("grad", 512, 512, 720, slices=64), name="grad_64x512"),
        # non-uniform detector and angle tables, a stack of slices
        dict(_case("mesh_radon", 768, 768, 600, slices=8), name="mesh_radon_8x768"),
        # pyraft's default projector, a full-resolution slice
        dict(_case("line_radon", 2048, 2048, 1500), name="line_radon_2048"),
        # pyraft's default backprojection, an ordinary slice
        dict(_case("line_backprojection", 1024, 1024, 721), name="line_backprojection_1024"),
        # a pyraft program's call: host arrays in and out, plan and filter made on the way
        dict(_case("numpy_fbp", 1024, 1024, 720), name="numpy_fbp_1024"),
    ]


# updates (interpolated accumulates) of the largest drawn call of each kind
_LIMIT = {"radon": 6.2e9, "backprojection": 6.2e9, "fbp": 6.2e9, "osem": 3.0e9, "osem_batch": 6.0e9, "grad": 2.4e10,
          "mesh_radon": 2.8e9, "line_radon": 6.2e9, "line_backprojection": 6.2e9, "numpy_fbp": 1.5e9}


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(sorted(_LIMIT))
    while True:
        n = _log_int(rng, 64, 2048)
        angles = _log_int(rng, 24, 1500)
        rays = n if rng.random() < 0.5 else min(2048, _log_int(rng, max(48, 0.7 * n), 1.5 * n))
        slices = 1 if rng.random() < 0.4 else _log_int(rng, 2, 64)
        more = {}
        if kind not in ("line_radon", "line_backprojection", "mesh_radon", "numpy_fbp", "osem_batch"):
            more["arc"] = rng.choice([math.pi, math.pi, 2.0 * math.pi, 2.0])
            more["half"] = rng.choice([1.0, 1.0, 1.42])
            more["shift"] = rng.choice([0.0, 0.0, 0.0, 0.03])
        if kind == "numpy_fbp":
            slices, rays = 1, n
        if kind == "osem":
            more["subsets"] = rng.choice([1, 4, 8, 16])
            more["niter"] = rng.choice([1, 2])
            more["half"] = 1.0 - more["shift"]  # every ray crosses the image
            slices = min(slices, 4)
        if kind == "osem_batch":
            more["subsets"] = rng.choice([4, 8])
            more["niter"] = 1
            slices = max(2, min(slices, 16))
        if angles < 40 * more.get("subsets", 0):
            continue  # subsets of a few views are no use to anyone
        c = _case(kind, n, rays, angles, slices=slices, **more)
        if n * n * angles * slices * 2.0 * c.get("niter", 0.5) <= _LIMIT[kind] and n * slices <= 40000:
            return c


# ------------------------------------------------------------------ inputs

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _ellipses(seed, count=16, whole=False):
    """(value, a, b, x0, y0, rotation) rows: a body that fills most of the field (or reaches
    past all of it: `whole`) and what it holds."""
    r = numpy.random.default_rng(seed)
    rad, phi = 0.62 * numpy.sqrt(r.random(count)), r.uniform(0.0, 2.0 * math.pi, count)
    inside = numpy.stack([r.uniform(0.1, 1.0, count), r.uniform(0.03, 0.35, count), r.uniform(0.03, 0.35, count),
                          rad * numpy.cos(phi), rad * numpy.sin(phi), r.uniform(0.0, math.pi, count)], 1)
    lo, hi = (1.6, 1.8) if whole else (0.8, 0.95)
    body = [[0.5, r.uniform(lo, hi), r.uniform(lo, hi), 0.0, 0.0, r.uniform(0.0, math.pi)]]
    return numpy.concatenate([body, inside])


def _image(ell, n, top_first):
    """The ellipses' density at the pixel centres; row 0 at y = -1 (or y = 1: top_first)."""
    dev = _device()
    x = torch.linspace(-1.0, 1.0, n, device=dev)
    y = (-x if top_first else x)[:, None]
    out = torch.zeros((n, n), device=dev)
    for v, a, b, x0, y0, rot in ell:
        c, s = math.cos(rot), math.sin(rot)
        p = ((x - x0) * c + (y - y0) * s) / a
        q = ((y - y0) * c - (x - x0) * s) / b
        out += v * (p * p + q * q <= 1.0)
    return out


def _images(case, seed, top_first=False):
    return torch.stack([_image(_ellipses(1000 * seed + i), case["n"], top_first) for i in range(case["slices"])])


def _sinogram(ell, rays, angles, th0, arc, tmin, tmax, last=False):
    """Line integrals of the ellipses, (rays, angles); `last`: the arc's end is an angle too."""
    dev = _device()
    th = th0 + torch.arange(angles, device=dev, dtype=torch.float64) * (arc / max(1, angles - (1 if last else 0)))
    t = torch.linspace(tmin, tmax, rays, device=dev, dtype=torch.float64)[:, None]
    out = torch.zeros((rays, angles), device=dev, dtype=torch.float64)
    for v, a, b, x0, y0, rot in ell:
        a2 = (a * torch.cos(th - rot)) ** 2 + (b * torch.sin(th - rot)) ** 2
        tau = t - x0 * torch.cos(th) - y0 * torch.sin(th)
        out += 2.0 * v * a * b * torch.sqrt((a2 - tau * tau).clamp_min(0.0)) / a2
    return out.float()


def _detector(case):
    return case["shift"] - case["half"], case["shift"] + case["half"]


def _sino_corners(case):
    tmin, tmax = _detector(case)
    return (0.0, tmax, case["arc"], tmin)


def _sinograms(case, seed, whole=False):
    tmin, tmax = _detector(case)
    return torch.stack([_sinogram(_ellipses(1000 * seed + i, whole=whole), case["rays"], case["angles"], 0.0,
                                  case["arc"], tmin, tmax) for i in range(case["slices"])])


def _counts(sino, seed):
    gen = torch.Generator(device=sino.device)
    gen.manual_seed(seed)
    return torch.poisson(sino * (100.0 / sino.mean()), generator=gen)


def _batch_sizes(case):
    """Slices around the case's size: sides and views spread over a factor of about three."""
    r = numpy.random.default_rng(case["n"] * 1000003 + case["angles"] * 1009 + case["slices"])
    n = [max(48, int(case["n"] * f)) for f in r.choice([0.34, 0.5, 0.67, 1.0, 1.0, 1.33], case["slices"])]
    a = [max(case["subsets"], int(case["angles"] * f)) for f in r.uniform(0.5, 1.5, case["slices"])]
    return n, a


def _mesh_tables(case, seed):
    r = numpy.random.default_rng(seed)
    return (numpy.sort(r.uniform(-1.0, 1.0, case["rays"])), numpy.sort(r.uniform(0.0, math.pi, case["angles"])))


def _inputs(case, seed):
    """The call's data alone (what `exact` starts from as well)."""
    kind = case["kind"]
    if kind == "radon":
        return dict(x=_images(case, seed))
    if kind in ("backprojection", "fbp"):
        return dict(s=_sinograms(case, seed))
    if kind == "osem":
        return dict(s=_counts(_sinograms(case, seed, whole=True), seed))
    if kind == "osem_batch":
        n, a = _batch_sizes(case)
        one = [_sinogram(_ellipses(1000 * seed + i, whole=True), n[i], a[i], 0.0, math.pi, -1.0, 1.0)
               for i in range(len(n))]
        return dict(s=[_counts(v, seed + i) for i, v in enumerate(one)])
    if kind == "grad":
        x, s = _images(case, seed), _sinograms(case, seed + 1)
        w = 0.5 + torch.rand(s.shape[-2:], device=s.device,
                             generator=torch.Generator(device=s.device).manual_seed(seed))
        return dict(x=x, s=s, w=w)
    if kind == "mesh_radon":
        t, th = _mesh_tables(case, seed)
        return dict(x=_images(case, seed), t=t, theta=th)
    if kind == "line_radon":
        return dict(x=_images(case, seed, top_first=True))
    if kind == "line_backprojection":
        # ray r at t = 1 - 2 r / (R - 1), angle a at pi a / (A - 1)
        return dict(s=torch.stack([_sinogram(_ellipses(1000 * seed + i), case["rays"], case["angles"], 0.0, math.pi,
                                             1.0, -1.0, last=True) for i in range(case["slices"])]))
    if kind == "numpy_fbp":
        return dict(s=_sinograms(case, seed)[0].double().cpu().numpy())
    raise ValueError("unknown kind %s" % kind)


def prepare(case, seed):
    state = dict(_inputs(case, seed), case=case)
    kind = case["kind"]
    n, rays, angles = case["n"], case["rays"], case["angles"]
    if kind in ("radon", "backprojection", "fbp", "osem", "grad"):
        state["plan"] = device.Plan(n, rays, angles, IMG, _sino_corners(case))
        if case.get("tune"):
            state["plan"].tune()
    elif kind == "osem_batch":
        sizes, views = _batch_sizes(case)
        state["plan"] = batch.Batch(sizes, nangles=views)
        state["s"] = state["plan"].pack_sinos(state["s"])
    elif kind == "mesh_radon":
        state["plan"] = device.Plan.mesh(n, state["t"], state["theta"])
    elif kind in ("line_radon", "line_backprojection"):
        state["plan"] = device.DdaPlan(n, rays, angles)
    elif kind == "numpy_fbp":
        state["s"] = pyraft_amd.image(state["s"], top_left=(0.0, 1.0), bottom_right=(math.pi, -1.0))
    if kind == "grad":
        state["x"].requires_grad_(True)
    return state


def run(state):
    case = state["case"]
    kind, plan = case["kind"], state.get("plan")
    if kind in ("radon", "mesh_radon", "line_radon"):
        return plan.radon(state["x"])
    if kind in ("backprojection", "line_backprojection"):
        return plan.backprojection(state["s"])
    if kind == "fbp":
        return plan.fbp(state["s"])
    if kind == "osem":
        return plan.em(state["s"], case["niter"], case["subsets"])
    if kind == "osem_batch":
        return plan.unpack_images(plan.em(state["s"], case["niter"], case["subsets"]))
    if kind == "grad":
        p = autograd.radon(state["x"], plan)
        r = p - state["s"]
        loss = 0.5 * (state["w"] * r * r).sum()
        g, = torch.autograd.grad(loss, state["x"])
        return p.detach(), g
    return pyraft_amd.fbp_gpu(state["s"])


def work(case):
    """Each input read once, each output written once; 4 operations per interpolated
    accumulate (difference, multiply, two adds)."""
    kind = case["kind"]
    n, rays, angles, slices = case["n"], case["rays"], case["angles"], case["slices"]
    img, sino, upd = n * n * slices, rays * angles * slices, float(n) * n * angles * slices
    size, passes = 4.0, 1.0
    if kind == "osem":
        passes = 2.0 * case["niter"]
    elif kind == "osem_batch":
        sizes, views = _batch_sizes(case)
        img, sino = sum(v * v for v in sizes), sum(v * a for v, a in zip(sizes, views))
        upd = float(sum(v * v * a for v, a in zip(sizes, views)))
        passes = 2.0 * case["niter"]
    elif kind == "grad":
        return {"bytes": 4.0 * (2 * img + 2 * sino + rays * angles), "flops": 8.0 * upd}
    elif kind == "numpy_fbp":
        size = 8.0
    return {"bytes": size * (img + sino), "flops": 4.0 * upd * passes}


# ------------------------------------------------------------------ the same in 64 bits

def _div(a, b):
    """a / b rounded once: which samples lie on the image is decided by these quotients (by a
    number, torch multiplies with the reciprocal on the GPU)."""
    return a / torch.full((), b, dtype=torch.float64, device=a.device)


def _axis(n):
    return torch.arange(n, device=_device(), dtype=torch.float64) * (2.0 / (n - 1)) - 1.0


def _detector_table(case):
    tmin, tmax = _detector(case)
    return tmin + torch.arange(case["rays"], device=_device(), dtype=torch.float64) * ((tmax - tmin) /
                                                                                       (case["rays"] - 1))


def _angle_table(case):
    return [j * (case["arc"] / case["angles"]) for j in range(case["angles"])]


def _samples(n, t, theta):
    """Interpolation cells of every (sample, ray): flat index of the lower tap in the image
    or (columns) its transpose, weight, validity, and the step length."""
    c, s, tan = math.cos(theta), math.sin(theta), math.tan(theta)
    h = 2.0 / (n - 1)
    x = (-1.0 + torch.arange(n, device=t.device, dtype=torch.float64) * h)[:, None]
    by_columns = abs(c) < 1.0 / math.sqrt(2.0)
    u = _div((_div(t, s) - _div(x, tan) if by_columns else _div(t, c) - x * tan) - (-1.0), h)
    m = torch.floor(u)
    ok = (m >= 0) & (m <= n - 2)
    w = torch.where(ok, u - m, 0.0)
    lo = torch.where(ok, m, 0.0).long() + torch.arange(n, device=t.device)[:, None] * n
    return lo, w, ok, by_columns, h / abs(s if by_columns else c)


def _radon64(x, t, thetas):
    S, n = x.shape[0], x.shape[-1]
    rows, cols = x.reshape(S, -1), x.transpose(1, 2).reshape(S, -1)
    out = torch.empty((S, t.numel(), len(thetas)), device=x.device, dtype=torch.float64)
    for j, th in enumerate(thetas):
        lo, w, ok, by_columns, step = _samples(n, t, th)
        src, shape = (cols if by_columns else rows), (S,) + lo.shape
        a = src.index_select(1, lo.reshape(-1)).reshape(shape)
        b = src.index_select(1, lo.reshape(-1) + 1).reshape(shape)
        out[:, :, j] = ((a * (1.0 - w) + b * w) * ok).sum(1) * step
    return out


def _transpose64(q, n, t, thetas):
    """The exact transpose of _radon64."""
    S = q.shape[0]
    rows = torch.zeros((n * n, S), device=q.device, dtype=torch.float64)
    cols = torch.zeros_like(rows)
    for j, th in enumerate(thetas):
        lo, w, ok, by_columns, step = _samples(n, t, th)
        dst = cols if by_columns else rows
        v = (q[:, :, j].t() * step)[None]  # (1, R, S)
        wl, wu = ((1.0 - w) * ok)[..., None], (w * ok)[..., None]
        dst.index_add_(0, lo.reshape(-1), (v * wl).reshape(-1, S))
        dst.index_add_(0, lo.reshape(-1) + 1, (v * wu).reshape(-1, S))
    return rows.t().reshape(S, n, n) + cols.t().reshape(S, n, n).transpose(1, 2)


def _backprojection64(q, n, tmin, dt, thetas, dth):
    S, R = q.shape[0], q.shape[1]
    x = _axis(n)
    out = torch.zeros((S, n, n), device=q.device, dtype=torch.float64)
    for j, th in enumerate(thetas):
        u = _div(x * math.cos(th) + x[:, None] * math.sin(th) - tmin, dt)
        m = torch.floor(u)
        ok = (m >= 0) & (m <= R - 2)
        w = torch.where(ok, u - m, 0.0)
        i = torch.where(ok, m, 0.0).long()
        row = q[:, :, j].contiguous()
        a = row.index_select(1, i.reshape(-1)).reshape(S, n, n)
        b = row.index_select(1, i.reshape(-1) + 1).reshape(S, n, n)
        out += (a * (1.0 - w) + b * w) * ok
    return out * dth


def _filter64(s, tmin, tmax):
    """Re(ifft(fft(s) fftshift(|w| cos(pi w dt)))) along the rays."""
    R = s.shape[1]
    dt = (tmax - tmin) / (R - 1)
    w = torch.linspace(-0.5 / dt, 0.5 / dt, R, device=s.device, dtype=torch.float64)
    h = torch.roll(w.abs() * torch.cos(math.pi * w * dt), R // 2)
    return torch.fft.ifft(torch.fft.fft(s, dim=1) * h[:, None], dim=1).real


def _osem64(s, n, case, subsets, niter):
    t, thetas = _detector_table(case), _angle_table(case)
    A, dth = len(thetas), case["arc"] / len(thetas)
    tmin, tmax = _detector(case)
    dt = (tmax - tmin) / (case["rays"] - 1)
    x = torch.ones((s.shape[0], n, n), device=s.device, dtype=torch.float64)
    cuts = [((b * A) // subsets, ((b + 1) * A) // subsets) for b in range(subsets)]
    weights = [_backprojection64(torch.ones_like(s[:1, :, a:b]), n, tmin, dt, thetas[a:b], dth) for a, b in cuts]
    for _ in range(niter):
        for (a, b), wt in zip(cuts, weights):
            p = _radon64(x, t, thetas[a:b])
            rho = torch.where(p > 0, s[:, :, a:b] / torch.where(p > 0, p, 1.0), 0.0)
            up = x * _backprojection64(rho, n, tmin, dt, thetas[a:b], dth) / torch.where(wt > 0, wt, 1.0)
            x = torch.where(wt > 0, up, x)
    return x


def _line_length(d, theta, h):
    """Length of a line at distance d from the centre of a square pixel of side h."""
    c, s = abs(math.cos(theta)), abs(math.sin(theta))
    p, q, top = 0.5 * h * (c + s), 0.5 * h * abs(c - s), h / max(c, s)
    if p - q < 1e-12 * h:
        return top * (d.abs() < p)
    return top * ((p - d.abs()) / (p - q)).clamp(0.0, 1.0)


def _line_radon64(x, rays, angles):
    S, n = x.shape[0], x.shape[-1]
    h = 2.0 / (n - 1)
    k = torch.arange(n, device=x.device, dtype=torch.float64)
    t = 1.0 - torch.arange(rays, device=x.device, dtype=torch.float64) * (2.0 / (rays - 1))
    rows, cols = x.reshape(S, -1), x.transpose(1, 2).reshape(S, -1)
    out = torch.empty((S, rays, angles), device=x.device, dtype=torch.float64)
    for a in range(angles):
        th = a * (math.pi / (angles - 1))
        c, s = math.cos(th), math.sin(th)
        by_rows = abs(c) >= abs(s)  # one row at a time: the columns the ray crosses there
        if by_rows:
            pos = ((t - (1.0 - k * h)[:, None] * s) / c + 1.0) / h
        else:
            pos = (1.0 - (t - (k * h - 1.0)[:, None] * c) / s) / h
        src, lead = (rows if by_rows else cols), max(abs(c), abs(s)) * h
        m = torch.floor(pos)
        acc = 0.0
        for e in (0, 1):
            ok = (m + e >= 0) & (m + e <= n - 1)
            i = torch.where(ok, m + e, 0.0).long() + torch.arange(n, device=x.device)[:, None] * n
            ln = _line_length((pos - m - e) * lead, th, h) * ok
            acc = acc + (src.index_select(1, i.reshape(-1)).reshape((S,) + i.shape) * ln).sum(1)
        out[:, :, a] = acc
    return out


def _line_backprojection64(q, n, rays, angles):
    S = q.shape[0]
    h, dt = 2.0 / (n - 1), 2.0 / (rays - 1)
    x = _axis(n)
    out = torch.zeros((S, n, n), device=q.device, dtype=torch.float64)
    norm = torch.zeros((n, n), device=q.device, dtype=torch.float64)
    for a in range(angles):
        th = a * (math.pi / (angles - 1))
        tc = x * math.cos(th) - x[:, None] * math.sin(th)  # row i at y = 1 - i h
        half = 0.5 * h * (abs(math.cos(th)) + abs(math.sin(th))) / dt
        rc = (1.0 - tc) / dt
        first = torch.ceil(rc - half)
        row = q[:, :, a].contiguous()
        for e in range(int(math.floor(2.0 * half)) + 1):
            r = first + e
            ok = (r >= 0) & (r <= rays - 1)
            i = torch.where(ok, r, 0.0).long()
            ln = _line_length((rc - r) * dt, th, h) * ok
            norm += ln
            out += row.index_select(1, i.reshape(-1)).reshape(S, n, n) * ln
    return out / norm


def exact(case, seed):
    kind = case["kind"]
    n, rays, angles = case["n"], case["rays"], case["angles"]
    data = _inputs(case, seed)
    dth = case["arc"] / angles
    tmin, tmax = _detector(case)
    if kind == "radon":
        return _radon64(data["x"].double(), _detector_table(case), _angle_table(case))
    if kind == "mesh_radon":
        t = torch.as_tensor(data["t"], device=data["x"].device)
        return _radon64(data["x"].double(), t, [float(v) for v in data["theta"]])
    if kind == "line_radon":
        return _line_radon64(data["x"].double(), rays, angles)
    if kind == "line_backprojection":
        return _line_backprojection64(data["s"].double(), n, rays, angles)
    if kind == "backprojection":
        return _backprojection64(data["s"].double(), n, tmin, (tmax - tmin) / (rays - 1), _angle_table(case), dth)
    if kind in ("fbp", "numpy_fbp"):
        s = torch.as_tensor(data["s"], device=_device()).float().double()
        f = _filter64(s if s.dim() == 3 else s[None], tmin, tmax)
        out = _backprojection64(f, n, tmin, (tmax - tmin) / (rays - 1), _angle_table(case), dth)
        return out if kind == "fbp" else out[0].cpu().numpy()
    if kind == "osem":
        return _osem64(data["s"].double(), n, case, case["subsets"], case["niter"])
    if kind == "osem_batch":
        out = []
        for s in data["s"]:
            side, views = s.shape
            one = dict(case, rays=side, angles=views)
            out.append(_osem64(s.double()[None], side, one, case["subsets"], case["niter"])[0])
        return out
    t, thetas = _detector_table(case), _angle_table(case)
    p = _radon64(data["x"].double(), t, thetas)
    return p, _transpose64(data["w"].double() * (p - data["s"].double()), n, t, thetas)
