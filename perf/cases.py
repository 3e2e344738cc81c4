"""Performance cases of the projector framework.

Each case is one call (or one step) that a program using the framework makes
through its public entry points, over the range the repository's own
configurations, tests and benchmark cover: parallel, fan-flat and fan-arc
images from 64^2 to 512^2 (single slices, small batches, planned batches of
up to 16, uneven batches of up to 64), cone-flat, cone-arc and helical
volumes, in both directions, plus filtered backprojection and the
data-consistency step built from it.

Kinds:
  step2d    projector2d: A x, residual against a measured sinogram, gradient
            of ||A x - y||^2 through autograd (one slice or a small batch);
  fbp2d     projector2d.filtered_backprojection of a sinogram;
  plan2d    the same gradient step on a BatchedProjector2d, eager;
  graph2d   the same gradient step captured with GraphStep and replayed;
  fid2d     the data-consistency step x - w FBP(A x - y) on a PlannedFBP2d;
  uneven    the gradient step on an UnevenBatch2d with the kernels its tuner
            picks for such batches (running sums in both directions);
  step3d    projector3d / projectorsp gradient step through autograd;
  fbp3d     projector3d.filtered_backprojection.

Images are ellipse / ellipsoid phantoms under noise, as a sampler's iterates
are; sinograms are the phantoms' line integrals with detector noise.
"""
import math
import random

import numpy as np
import torch

PIX, DET, SID, SDD = 0.7, 1.2858, 595.0, 1085.6  # mm, the fan scanner of the benchmark
DEV = "cuda"


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _two(kind, scan, w, h, det, views, batch):
    return {"kind": kind, "scan": scan, "w": w, "h": h, "det": det, "views": views, "batch": batch}


def _three(kind, scan, w, h, dz, cols, rows, views, batch):
    return {"kind": kind, "scan": scan, "w": w, "h": h, "dz": dz, "cols": cols, "rows": rows,
            "views": views, "batch": batch}


def listed():
    named = {
        # the smallest image the tests use: launches and latency
        "arc-64-step": _two("step2d", "arc", 64, 64, 92, 60, 1),
        # the reference's own CPU configuration
        "para-256-step": _two("step2d", "para", 256, 256, 367, 180, 1),
        # a ragged rectangle, filtered backprojection of a small batch
        "flat-203x152-fbp": _two("fbp2d", "flat", 203, 152, 301, 240, 3),
        # one full-size clinical slice through the drop-in module
        "arc-512-step": _two("step2d", "arc", 512, 512, 736, 720, 1),
        # a sampler's inner loop over a small batch, replayed as a graph
        "arc-256-graph-b8": _two("graph2d", "arc", 256, 256, 368, 360, 8),
        # the headline: 16 slices, planned
        "arc-512-plan-b16": _two("plan2d", "arc", 512, 512, 736, 720, 16),
        # the sampler's data-consistency step on the same batch
        "arc-512-fidelity-b16": _two("fid2d", "arc", 512, 512, 736, 720, 16),
        # 64 slices of different size, view count and detector
        "arc-uneven-64": {"kind": "uneven", "scan": "arc", "count": 64, "n_lo": 256, "n_hi": 512,
                          "v_lo": 96, "v_hi": 720, "shape_seed": 2025},
        # a small odd cone-beam volume
        "cone-flat-96-step": _three("step3d", "flat", 96, 81, 50, 131, 75, 100, 1),
        # cone-beam filtered backprojection at a preview size
        "cone-arc-160-fbp": _three("fbp3d", "arc", 160, 144, 96, 243, 128, 201, 1),
        # the benchmark's cone-beam volume
        "cone-flat-256-step-b2": _three("step3d", "flat", 256, 256, 256, 512, 384, 360, 2),
        # one turn of the benchmark's helical scan
        "helical-512-step-b4": _three("step3d", "spiral", 512, 512, 64, 736, 64, 1152, 4),
    }
    return [dict(c, name=n) for n, c in named.items()]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step2d", "step2d", "fbp2d", "plan2d", "graph2d", "fid2d", "uneven",
                       "step3d", "step3d", "fbp3d"])
    if kind == "uneven":
        lo = rng.randint(64, 256)
        return {"kind": kind, "scan": rng.choice(["para", "flat", "arc"]), "count": _log(rng, 4, 48),
                "n_lo": lo, "n_hi": rng.randint(lo + 1, 512), "v_lo": 60, "v_hi": rng.randint(96, 720),
                "shape_seed": rng.randrange(1 << 20)}
    if kind in ("step3d", "fbp3d"):
        scan = rng.choice(["flat", "arc"] if kind == "fbp3d" else ["flat", "arc", "spiral"])
        w = _log(rng, 48, 200)
        h = max(32, int(w * rng.uniform(0.75, 1.25)))
        dz = max(16, int(w * rng.uniform(0.2, 0.9)))
        cols, rows = int(math.hypot(w, h) * rng.uniform(1.0, 1.6)), max(12, int(dz * rng.uniform(0.8, 1.5)))
        return _three(kind, scan, w, h, dz, cols, rows, _log(rng, 60, 400),
                      rng.choice([1, 1, 2, 3, 4]) if kind == "step3d" else rng.choice([1, 2]))
    w = _log(rng, 64, 512)
    h = w if rng.random() < 0.5 else max(32, int(w * rng.uniform(0.7, 1.0)))
    scan = rng.choice(["para", "flat", "arc"] if kind != "fid2d" else ["flat", "arc"])
    batch = {"step2d": [1, 1, 2, 4], "fbp2d": [1, 2, 3, 4], "plan2d": [4, 7, 8, 16],
             "graph2d": [2, 4, 8, 16], "fid2d": [4, 8, 13, 16]}[kind]
    return _two(kind, scan, w, h, int(max(w, h) * rng.uniform(1.2, 1.6)), _log(rng, 60, 720), rng.choice(batch))


# ---------------------------------------------------------------------------
# geometry: what the constructors are given, and its meaning in 64 bits
# ---------------------------------------------------------------------------
def _fan_args(scan, w, h, det):
    """Constructor arguments of one 2D scan: the benchmark's pixel and bin at
    512 pixels and 736 bins, the same field of view at other sizes."""
    d = DET * 736.0 / det * (SID / SDD if scan == "para" else 1.0)
    return dict(image_size=(w, h), num_det=det, pix_size=PIX * 512.0 / max(w, h), det_size=d,
                iso_source=SID, source_detector=SDD, scan_type=scan)


def _cone_args(c):
    """Constructor arguments of one 3D scan: 256 mm of object at the cone
    scanner's distances, the helical scanner's own sizes."""
    w, h, dz, cols, rows = (c[k] for k in ("w", "h", "dz", "cols", "rows"))
    if c["scan"] == "spiral":
        k = 512.0 / max(w, h)
        return dict(image_size=(w, h, dz), num_det=(cols, rows), pix_size=(0.7 * k, 0.7 * k, 1.0 * k),
                    det_size=(1.2858 * 736.0 / cols, 1.82454 * k * dz / rows), iso_source=SID,
                    source_detector=SDD, scan_type="arc")
    k = 256.0 / max(w, h)
    return dict(image_size=(w, h, dz), num_det=(cols, rows), pix_size=k,
                det_size=(512.0 / cols, 1.5 * k * dz / rows), iso_source=1000.0,
                source_detector=1500.0, scan_type=c["scan"])


def _f(v):
    """A parameter as the projector keeps it: rounded to 32 bits."""
    return float(np.float32(v))


class _Geo:
    """One scan in 64 bits; 2D scans are 3D ones without z."""

    def __init__(self, c, w=None, h=None, det=None, views=None):
        self.dim = 3 if "dz" in c else 2
        self.scan = c["scan"]
        if self.dim == 2:
            a = _fan_args(c["scan"], w or c["w"], h or c["h"], det or c["det"])
            (self.W, self.H), self.C = a["image_size"], a["num_det"]
            self.dx = self.dy = _f(a["pix_size"])
            col = a["det_size"]
        else:
            a = _cone_args(c)
            (self.W, self.H, self.Dz), (self.C, self.R) = a["image_size"], a["num_det"]
            p = a["pix_size"] if isinstance(a["pix_size"], tuple) else (a["pix_size"],) * 3
            self.dx, self.dy, self.dz = (_f(v) for v in p)
            col, self.row = a["det_size"][0], _f(a["det_size"][1])
        self.arc = a["scan_type"] == "arc"
        self.args, self.sid, self.sdd = a, _f(a["iso_source"]), _f(a["source_detector"])
        self.col_arg = col / a["source_detector"] if self.arc else col
        self.col = _f(self.col_arg)
        self.V = views or c["views"]
        turn = math.pi if self.scan == "para" else 2 * math.pi
        self.angles = (np.arange(self.V) * (turn / self.V)).astype(np.float32)
        self.z = np.zeros(self.V, dtype=np.float32)
        if self.scan == "spiral":  # the source passes the volume once
            self.z = np.linspace(-0.5, 0.5, self.V, dtype=np.float32) * np.float32(self.Dz * self.dz)

    def pitch(self):
        """Bin pitch: radians (arc), at the isocentre (flat), or as it is (parallel)."""
        return self.sid / self.sdd * self.col if self.scan == "flat" else self.col

    def view(self, v):
        """(source, axis choice, flip, column edges on the axis in walk
        order, column-centre magnifications) of one view."""
        thf = self.angles[v]
        th = float(thf)
        cf, sf = np.float32(math.cos(th)), np.float32(math.sin(th))
        xaxis = bool(np.float32(cf * cf) > np.float32(0.5))
        flip = not (cf >= 0) if xaxis else not (sf >= 0)
        s, c = math.sin(th), math.cos(th)
        sx, sy = -s * self.sid, c * self.sid
        k = torch.arange(self.C + 1, dtype=torch.float64, device=DEV)
        off = (self.C / 2 - k) if flip else (k - self.C / 2)
        mid = (off[1:] + off[:-1]) / 2
        if self.scan == "para":
            return None, xaxis, flip, off * self.col / (c if xaxis else s), None, th
        if self.arc:
            t = torch.tan(off * self.col + th)
            e = sx + sy * t if xaxis else sy + sx / t
            dcx, dcy = torch.sin(mid * self.col + th) * self.sdd + sx, -torch.cos(mid * self.col + th) * self.sdd + sy
        else:
            u, m = off * self.pitch(), mid * self.pitch()
            px, py, dcx, dcy = u * c, u * s, m * c, m * s
            e = (sx * py - sy * px) / (py - sy) if xaxis else (sy * px - sx * py) / (px - sx)
        mag = sy / (sy - dcy) if xaxis else sx / (sx - dcx)
        return (sx, sy), xaxis, flip, e, mag, th

    def rows_z(self, v):
        r = torch.arange(self.R + 1, dtype=torch.float64, device=DEV) - self.R / 2
        return r * self.row * (self.sid / self.sdd if self.scan == "flat" else 1.0) + float(self.z[v])


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _ellipsoids(rng, n, dim):
    out = []
    for _ in range(n):
        r, phi = math.sqrt(rng.random()) * 0.6, rng.uniform(0, 2 * math.pi)
        out.append((r * math.cos(phi), r * math.sin(phi), rng.uniform(-0.5, 0.5) if dim == 3 else 0.0,
                    rng.uniform(0.05, 0.4), rng.uniform(0.05, 0.4), rng.uniform(0.1, 0.6),
                    rng.uniform(0, math.pi), rng.uniform(0.1, 1.0)))
    return out


def _image(geo, batch, rng, gen):
    """[batch, 1, (Dz,) H, W]: phantoms (attenuation per mm) under noise of a
    tenth of their peak, and the phantoms' ellipsoids in mm."""
    half = (geo.W * geo.dx / 2, geo.H * geo.dy / 2, geo.Dz * geo.dz / 2 if geo.dim == 3 else 1.0)
    xs = (torch.arange(geo.W, device=DEV) - geo.W / 2 + 0.5) * geo.dx
    ys = (geo.H / 2 - torch.arange(geo.H, device=DEV) - 0.5) * geo.dy
    zs = (torch.arange(geo.Dz, device=DEV) - geo.Dz / 2 + 0.5) * geo.dz if geo.dim == 3 else torch.zeros(1, device=DEV)
    Z, Y, X = zs[:, None, None], ys[:, None], xs
    out, every = [], []
    for _ in range(batch):
        img = torch.zeros(len(zs), geo.H, geo.W, device=DEV)
        own = []
        for cx, cy, cz, a, b, d, t, val in _ellipsoids(rng, 10, geo.dim):
            e = (cx * half[0], cy * half[1], cz * half[2], a * half[0], b * half[1], d * half[2], t, 0.01 * val)
            u, w = (X - e[0]) * math.cos(t) + (Y - e[1]) * math.sin(t), (Y - e[1]) * math.cos(t) - (X - e[0]) * math.sin(t)
            q = (u / e[3]) ** 2 + (w / e[4]) ** 2
            if geo.dim == 3:
                q = q + ((Z - e[2]) / e[5]) ** 2
            img += e[7] * (q <= 1)
            own.append(e)
        img += 0.002 * torch.randn(img.shape, device=DEV, generator=gen)
        out.append(img if geo.dim == 3 else img[0])
        every.append(own)
    return torch.stack(out)[:, None].contiguous(), every


def _sinogram(geo, every, gen):
    """[batch, 1, V, (R,) C]: line integrals of the ellipsoids through the
    cell centres, plus the noise of about 1e5 photons."""
    th = torch.from_numpy(geo.angles).to(DEV).double()[:, None, None]
    off = (torch.arange(geo.C, device=DEV) + 0.5 - geo.C / 2).double()
    s, c = torch.sin(th), torch.cos(th)
    z0 = torch.from_numpy(geo.z).to(DEV).double()[:, None, None]
    zero = torch.zeros_like(th)
    if geo.scan == "para":
        src, d = (off * geo.col * c, off * geo.col * s, zero), (s + 0 * off, -c + 0 * off, zero)
    else:
        src = (-s * geo.sid, c * geo.sid, z0)
        if geo.arc:
            g = off * geo.col + th
            hit = (torch.sin(g) * geo.sdd + src[0], -torch.cos(g) * geo.sdd + src[1])
        else:
            hit = (off * geo.pitch() * c, off * geo.pitch() * s)
        dz = zero
        if geo.dim == 3:
            r = (torch.arange(geo.R, device=DEV) + 0.5 - geo.R / 2).double()[:, None] * geo.row
            dz = r * (geo.sid / geo.sdd if geo.scan == "flat" else 1.0)
        d = (hit[0] - src[0], hit[1] - src[1], dz)
    src, d = tuple(t.float() for t in src), tuple(t.float() for t in d)
    length = torch.sqrt(d[0] ** 2 + d[1] ** 2 + d[2] ** 2)
    rows = geo.R if geo.dim == 3 else 1
    out = torch.empty(len(every), 1, geo.V, rows, geo.C, device=DEV)
    for b, own in enumerate(every):
        y = 1e-3 * torch.randn(geo.V, rows, geo.C, device=DEV, generator=gen)
        for ex, ey, ez, a, bb, az, t, val in own:
            ct, st = math.cos(t), math.sin(t)
            px, py = src[0] - ex, src[1] - ey
            qx, qy = (px * ct + py * st) / a, (py * ct - px * st) / bb
            ux, uy = (d[0] * ct + d[1] * st) / a, (d[1] * ct - d[0] * st) / bb
            uu, qu, qq = ux * ux + uy * uy, ux * qx + uy * qy, qx * qx + qy * qy
            if geo.dim == 3:
                qz, uz = (src[2] - ez) / az, d[2] / az
                uu, qu, qq = uu + uz * uz, qu + uz * qz, qq + qz * qz
            y += 2 * val * torch.sqrt(torch.clamp(qu * qu - uu * (qq - 1), min=0)) / uu * length
        out[b, 0] = y
    return (out if geo.dim == 3 else out[:, :, :, 0]).contiguous()


def _uneven_geos(case):
    r = np.random.RandomState(case["shape_seed"])
    geos = []
    for _ in range(case["count"]):
        n = int(r.randint(case["n_lo"], case["n_hi"] + 1))
        geos.append(_Geo(case, w=n, h=n, det=int(math.ceil(1.44 * n)), views=int(r.randint(case["v_lo"], case["v_hi"] + 1))))
    return geos


def _inputs(case, seed):
    """[(geometry, image or None, sinogram)] of a case, from the seed alone."""
    rng, gen = random.Random(seed), torch.Generator(device=DEV).manual_seed(seed)
    geos = _uneven_geos(case) if case["kind"] == "uneven" else [_Geo(case)]
    got = []
    for geo in geos:
        x, every = _image(geo, case.get("batch", 1), rng, gen)
        got.append((geo, x, _sinogram(geo, every, gen)))
    return got


def prepare(case, seed):
    from pridediff_amd import load_radontorch
    from pridediff_amd.batched import BatchedProjector2d, GraphStep, UnevenBatch2d, data_consistency_grad
    from pridediff_amd.deeprecon.torch.projector import projector2d, projector3d, projectorsp
    from pridediff_amd.fbp import PlannedFBP2d

    kind = case["kind"]
    got = _inputs(case, seed)
    make = {True: projectorsp, False: projector3d if "dz" in case else projector2d}[case["scan"] == "spiral"]
    projs = [make(**g.args).to(DEV) for g, _, _ in got]
    angs = [torch.from_numpy(g.angles).to(DEV) for g, _, _ in got]
    s = {"kind": kind, "P": projs[0], "ang": angs[0], "x": got[0][1].requires_grad_(True), "y": got[0][2], "extra": ()}
    if case["scan"] == "spiral":
        spos = np.zeros((4, got[0][0].V), dtype=np.float32)
        spos[0] = got[0][0].z
        s["extra"] = (torch.from_numpy(spos).to(DEV),)
    if kind == "uneven":
        rt = load_radontorch()
        ub = UnevenBatch2d(projs, angs)
        ub.plan.set_variant(rt.ADJ_BLOCK_PREFIX | rt.FWD_PREFIX)
        s.update(op=ub.projection, x=ub.pack_images([x[0, 0] for _, x, _ in got]).detach().requires_grad_(True),
                 y=ub.pack_sinos([y[0, 0] for _, _, y in got]))
    elif kind in ("plan2d", "graph2d", "fid2d"):
        bp = BatchedProjector2d(projs[0], angs[0], case["batch"])
        s["op"] = bp.projection
        if kind == "graph2d":
            s["step"] = GraphStep(lambda a, b: data_consistency_grad(bp.projection, a, b), s["x"], s["y"])
        if kind == "fid2d":
            s["fbp"] = PlannedFBP2d(projs[0], angs[0], case["batch"], plan=bp)
            s["w"] = torch.full((1,), 0.5, device=DEV)
    return s


def run(s):
    from pridediff_amd.fbp import fidelity_step_fused

    kind = s["kind"]
    if kind in ("fbp2d", "fbp3d"):
        with torch.no_grad():
            return s["P"].filtered_backprojection(s["y"], s["ang"])
    if kind == "fid2d":
        with torch.no_grad():
            return fidelity_step_fused(s["fbp"], s["x"].detach(), s["y"], s["w"])
    if kind == "graph2d":
        return s["step"].replay(s["x"], s["y"])
    x = s["x"]
    x.grad = None
    ax = s["op"](x) if "op" in s else s["P"].projection(x, s["ang"], *s["extra"])
    r = ax - s["y"]
    torch.autograd.backward(r, grad_tensors=2.0 * r)
    return ax, x.grad


# ---------------------------------------------------------------------------
# what the path cannot do without
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: each input read once, each output written once.  Operations: per
    view each pixel meets, on average, one bin more than its width in bins;
    a multiply-add for each meeting and instance (3D: times the rows or
    slices met), plus the filter's matrix product in the reconstructions."""
    geos = _uneven_geos(case) if case["kind"] == "uneven" else [_Geo(case)]
    b = case.get("batch", 1)
    img = sum(g.W * g.H * (g.Dz if g.dim == 3 else 1) for g in geos) * b
    sino = sum(g.V * g.C * (g.R if g.dim == 3 else 1) for g in geos) * b
    gather = sum(2.0 * g.V * g.W * g.H * 2 * (g.Dz * 2 if g.dim == 3 else 1) for g in geos) * b
    gemm = 2.0 * sino * geos[0].C
    kind = case["kind"]
    if kind in ("fbp2d", "fbp3d"):
        return {"bytes": 4.0 * (img + sino), "flops": gather + gemm}
    if kind == "fid2d":
        return {"bytes": 4.0 * (2 * img + sino), "flops": 2 * gather + gemm}
    return {"bytes": 4.0 * (2 * img + (sino if kind == "graph2d" else 2 * sino)), "flops": 2 * gather}


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _at(table, t):
    """The running integral `table` [..., n + 1] (linear between its entries)
    at positions t [..., m] in [0, n]."""
    i = t.floor().clamp(0, table.shape[-1] - 2).long()
    shape = table.shape[:-1] + t.shape[-1:]
    lo = torch.gather(table, -1, i.expand(shape))
    return lo + (torch.gather(table, -1, (i + 1).expand(shape)) - lo) * (t - i)


def _running(x):
    return torch.nn.functional.pad(torch.cumsum(x, -1), (1, 0))


def _view(geo, v, x, weights):
    """View v of the projection of x [B, (Dz,) H, W] in detector order.
    weights: "fp" (projection), "bp" (the backprojection's transpose) or
    "bpw" (the same with the filtered backprojection's distance weight)."""
    src, xaxis, flip, e, mag, th = geo.view(v)
    s, c = math.sin(th), math.cos(th)
    if xaxis:
        lines = (geo.H / 2 - torch.arange(geo.H, dtype=torch.float64, device=DEV) - 0.5) * geo.dy
        n, step, img = geo.W, geo.dx, x
    else:
        lines = (torch.arange(geo.W, dtype=torch.float64, device=DEV) - geo.W / 2 + 0.5) * geo.dx
        n, step, img = geo.H, geo.dy, x.transpose(-1, -2).flip(-1)
    if src is None:
        a0, p = -n / 2 * step + lines * (s / c if xaxis else c / s), torch.full_like(lines, step)
    else:
        sa, sp = (src[0], src[1]) if xaxis else (src[1], src[0])
        a0, a1 = ((sa * lines - sp * q) / (lines - sp) for q in (-n / 2 * step, n / 2 * step))
        p, m = (a1 - a0) / n, sp / (sp - lines)
    if weights == "bpw":
        q = (torch.arange(n, dtype=torch.float64, device=DEV) - n / 2 + 0.5) * step
        X, Y = (q[None], lines[:, None]) if xaxis else (lines[:, None], q[None])
        if geo.scan == "flat":
            dist = (geo.sid / (geo.sid - (src[0] * X + src[1] * Y) / geo.sid)) ** 2
        else:
            dist = 1 / ((src[0] - X) ** 2 + (src[1] - Y) ** 2)
        img = img * dist
    t = ((e[None] - a0[:, None]) / p[:, None]).clamp(0, n)
    width = e[1:] - e[:-1]
    kbp = geo.pitch() * (geo.sid if geo.arc else 1.0)
    perp = geo.dy if xaxis else geo.dx
    if geo.dim == 2:
        got = torch.diff(_at(_running(img), t), dim=-1)  # [B, line, bin], in pixels
        if weights != "fp":
            out = kbp * got.sum(-2)
        else:
            mid = (e[1:] + e[:-1]) / 2
            w = perp / (width * (abs(sp) / torch.sqrt((mid - sa) ** 2 + sp * sp))) if src else perp / geo.col
            out = (got * p[:, None]).sum(-2) * w
    else:
        sz = float(geo.z[v])
        zr = mag[:, None] * (geo.rows_z(v)[None] - sz) + sz                       # [bin, row edge]
        z0 = m * (-geo.Dz / 2 * geo.dz - sz) + sz                                  # [line]
        tz = ((zr[None] - z0[:, None, None]) / (m * geo.dz)[:, None, None]).clamp(0, geo.Dz)
        got = torch.diff(_at(_running(img.transpose(-2, -3)), t[:, None]), dim=-1)  # [B, line, slice, bin]
        got = torch.diff(_at(_running(got.transpose(-1, -2)), tz), dim=-1)          # [B, line, bin, row]
        if weights != "fp":
            out = kbp * got.sum(1)
        else:
            a, b = ((e[1:] + e[:-1]) / 2 - sa)[:, None], (zr[:, 1:] + zr[:, :-1]) / 2
            w = perp / (width[:, None] * torch.diff(zr, dim=-1) * abs(sp) / torch.sqrt(a * a + b * b + sp * sp))
            out = (got * (p * m * geo.dz)[:, None, None]).sum(1) * w
        out = out.transpose(-1, -2)
    return out.flip(-1) if flip else out


def _project(geo, x):
    return torch.stack([_view(geo, v, x, "fp") for v in range(geo.V)], 1)


def _transpose(geo, y, weights):
    """The transpose of _view over all views, by its own gradient."""
    shape = (y.shape[0],) + ((geo.Dz,) if geo.dim == 3 else ()) + (geo.H, geo.W)
    x = torch.zeros(shape, dtype=torch.float64, device=DEV, requires_grad=True)
    out = torch.zeros_like(x)
    for v in range(geo.V):
        with torch.enable_grad():
            got = _view(geo, v, x, weights)
        out = out + torch.autograd.grad(got, x, y[:, v])[0]
    return out.detach()


def _fbp(geo, y):
    k = torch.arange(-(geo.C - 1), geo.C, dtype=torch.float64, device=DEV)
    d = geo.col_arg * (geo.args["iso_source"] / geo.args["source_detector"] if geo.scan == "flat" else 1.0)
    taps = torch.where(k.long() % 2 != 0, -1 / (math.pi * d * k) ** 2, torch.zeros_like(k))
    taps[geo.C - 1] = 1 / (4 * d * d)
    j = torch.arange(geo.C, device=DEV)
    R = geo.args["iso_source"]
    u = (torch.arange(geo.C, dtype=torch.float64, device=DEV) - geo.C / 2 + 0.5) * geo.col_arg
    if geo.dim == 2:
        if geo.scan == "flat":
            u = u * R / geo.args["source_detector"]
            w = R / torch.sqrt(u * u + R * R)
        else:
            w = torch.cos(u) if geo.scan == "arc" else torch.ones_like(u)
    else:
        r = (torch.arange(geo.R, dtype=torch.float64, device=DEV) - geo.R / 2 + 0.5)[:, None]
        r = r * geo.args["det_size"][1] * R / geo.args["source_detector"]
        u = u * R / geo.args["source_detector"] if geo.scan == "flat" else torch.tan(u) * R
        w = R / torch.sqrt(r * r + u * u + R * R)
    filtered = (y * w) @ taps[j[:, None] - j[None] + geo.C - 1]
    step = abs(float(geo.angles[-1]) - float(geo.angles[0])) / (geo.V - 1)
    return _transpose(geo, filtered, "bp" if geo.scan == "para" else "bpw") * step / 2


def exact(case, seed):
    geos = _uneven_geos(case) if case["kind"] == "uneven" else [_Geo(case)]
    # elements that the 64-bit evaluation goes through, and what it takes in 20 s
    cost = sum(g.V * case.get("batch", 1) * (max(g.W, g.H) * (g.C * (g.R + 2 * g.Dz) + 2 * g.W * g.Dz) if g.dim == 3
                                             else max(g.W, g.H) * (g.C + g.W) + 2e5) for g in geos)
    if cost > 2.2e10:
        return None
    kind = case["kind"]
    grads, sinos = [], []
    with torch.no_grad():
        for geo, x, y in _inputs(case, seed):
            x, y = x[:, 0].double(), y[:, 0].double()
            if kind in ("fbp2d", "fbp3d"):
                return _fbp(geo, y)[:, None]
            ax = _project(geo, x)
            if kind == "fid2d":
                return (x - 0.5 * _fbp(geo, ax - y))[:, None]
            sinos.append(ax)
            grads.append(_transpose(geo, 2 * (ax - y), "fp"))
    if kind == "uneven":
        return torch.cat([a.reshape(-1) for a in sinos]), torch.cat([g.reshape(-1) for g in grads])
    if kind == "graph2d":
        return grads[0][:, None]
    return sinos[0][:, None], grads[0][:, None]
