"""The work that a user of ctlib_amd has it do, as cases that can be timed and checked.

A case is a dict of plain values.  `listed()` gives the named ones, `draw(rng)` one more of the same
ranges, `prepare` what a program holds before the call, `run` one pass through the public entry
points, `work` the bytes and operations that the pass cannot do without and `exact` the result in
64 bits from plain torch.

Geometries are those of ctlib_amd.phantom scaled to the case's sizes: the fan-beam scanner of source
distance 5.95 and detector distance 4.906 seeing a field of 3.379, and the parallel one of extent 1.
Images are ellipse phantoms, sinograms their analytic line integrals with counting noise.
"""
import math

import torch

import ctlib_amd
from ctlib_amd import autograd, batch, recon

S2R, D2R = 5.95, 4.906
FIELD = 512 * 0.0066            # image extent of the fan-beam geometries
ED_DETECTOR = 736 * 0.0072      # detector extents: equal distance, equal angle, parallel
EA_DETECTOR = 888 * 0.0011
PARA_DETECTOR = 367 / 256
SCAN = {"ed": 0, "ea": 1, "para": 2}
TO_SINO = ("projection", "backprojection_t")
TO_IMAGE = ("projection_t", "backprojection", "fbp")
WEIGHTED = ("backprojection", "backprojection_t", "fbp", "backprojection_sv")
I0 = 5e4                        # photons per ray


def _dd(name, op, scan, size, views, dets, batch, dtype="f32", train=False, **more):
    width, height = size
    return dict(name=name, op=op, scan=scan, width=width, height=height, views=views, dets=dets, batch=batch,
                dtype=dtype, train=train, **more)


def listed():
    return [
        # the smallest call: one parallel-beam slice, as in a loop over slices; launches and latency count
        _dd("para256_projection_b1", "projection", "para", (256, 256), 180, 367, 1),
        # quick-look reconstruction of one small slice
        _dd("para256_fbp_b1", "fbp", "para", (256, 256), 180, 367, 1),
        # iterative reconstruction of one clinical slice: y = A x and A^T (y - m)
        _dd("ed512_residual_b1", "residual_step", "ed", (512, 512), 736, 736, 1),
        # the data term of a training step at the largest batch: loss and gradient
        _dd("ed512_least_squares_b32", "least_squares", "ed", (512, 512), 736, 736, 32),
        # analytic reconstruction of a batch
        _dd("ed512_fbp_b8", "fbp", "ed", (512, 512), 736, 736, 8),
        # a backprojection layer of a network, forward and backward
        _dd("ed512_backprojection_train_b8", "backprojection", "ed", (512, 512), 736, 736, 8, train=True),
        # a projection layer on the equal-angle scanner, forward and backward
        _dd("ea512_projection_train_b16", "projection", "ea", (512, 512), 1024, 888, 16, train=True),
        # unrolled gradient descent with learned steps at high resolution: a training step of two iterations
        _dd("ed1024_unrolled_b4", "unrolled", "ed", (1024, 1024), 1440, 1536, 4, iters=2),
        # gradient checks and reference computations: fp64, odd sizes, a shifted detector
        _dd("ea_ragged_fbp_train_f64_b3", "fbp", "ea", (421, 300), 211, 333, 3, dtype="f64", train=True, shift=0.25),
        # per-view images, the input of view-weighting networks
        _dd("ed512_views_b1", "backprojection_sv", "ed", (512, 512), 736, 736, 1),
        # a mixed worklist of slices, each with its own geometry, through the batch handle
        dict(name="hetero_b16", op="hetero", slices=16, pick=3999, dtype="f32"),
        # graph weights over the 7 x 7 patches of a 128 x 128 image
        dict(name="laplacian_16384x49", op="laplacian", points=16384, dim=49, k=16, dtype="f32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(case):
    """Relative time of a pass: operations, dearer in fp64 and with pixel weights."""
    return work(case)["flops"] * (1.7 if case["dtype"] == "f64" else 1.0) * (1.8 if case["op"] in WEIGHTED else 1.0)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.random()
        if kind < 0.08:
            case = dict(op="laplacian", points=_log_int(rng, 500, 16384), dim=_log_int(rng, 3, 256),
                        k=_log_int(rng, 8, 128), dtype="f32")
        elif kind < 0.16:
            case = dict(op="hetero", slices=rng.randint(4, 24), pick=rng.randrange(1 << 30), dtype="f32")
        else:
            op = rng.choice(TO_SINO + TO_IMAGE + TO_IMAGE + TO_SINO
                            + ("residual_step", "least_squares", "least_squares", "unrolled", "backprojection_sv"))
            scan = "ed" if op == "backprojection_sv" else rng.choice(("ed", "ed", "ea", "para"))
            width = _log_int(rng, 96, 1024)
            if rng.random() < 0.4:
                width = max(64, width // 64 * 64)
            height = width if rng.random() < 0.6 else max(64, int(width * rng.uniform(0.6, 1.0)))
            case = _dd(None, op, scan, (width, height), _log_int(rng, 60, 1440),
                       min(1536, int(width * rng.uniform(1.0, 1.8))), _log_int(rng, 1, 32),
                       dtype="f64" if rng.random() < 0.2 else "f32",
                       train=op in TO_SINO + TO_IMAGE and rng.random() < 0.4)
            del case["name"]
            if op == "unrolled":
                case["iters"] = rng.randint(1, 3)
            if rng.random() < 0.3:
                case["shift"] = round(rng.uniform(-2.0, 2.0), 2)
            if op == "backprojection_sv" and work(case)["bytes"] > 2e9:
                continue
        if _cost(case) <= most:
            return case


# ---- inputs -------------------------------------------------------------------------------------


def _options(case):
    """The options vector of the case, float32 on the host."""
    V, D, W, H = case["views"], case["dets"], case["width"], case["height"]
    side = max(W, H)
    if case["scan"] == "para":
        d_det = PARA_DETECTOR / D
        o = [V, D, W, H, 1.0 / side, d_det, 0.0, math.pi / V, case.get("shift", 0.0) * d_det, 2]
    else:
        d_det = (ED_DETECTOR if case["scan"] == "ed" else EA_DETECTOR) / D
        o = [V, D, W, H, FIELD / side, d_det, 0.0, 2 * math.pi / V, S2R, D2R, case.get("shift", 0.0) * d_det,
             SCAN[case["scan"]]]
    return torch.tensor(o, dtype=torch.float32)


def _ellipses(B, options, gen):
    """[B, 10, 6] (cx, cy, a, b, angle, value) in image units, as the phantoms draw them."""
    half = torch.tensor([float(options[2]), float(options[3])], dtype=torch.float64) * float(options[4]) / 2
    u = torch.rand(B, 10, 6, generator=gen, dtype=torch.float64)
    e = torch.empty_like(u)
    e[..., 0:2] = (u[..., 0:2] * 1.4 - 0.7) * half
    e[..., 2:4] = (u[..., 2:4] * 0.35 + 0.05) * half
    e[..., 4] = u[..., 4] * math.pi
    e[..., 5] = u[..., 5] * (1.0 if float(options[-1]) == 2 else 0.02)
    return e


def _image(ell, options, device):
    W, H, d = int(options[2]), int(options[3]), float(options[4])
    x = (torch.arange(W, device=device, dtype=torch.float64) - W / 2 + 0.5) * d
    y = (H / 2 - torch.arange(H, device=device, dtype=torch.float64) - 0.5) * d
    out = torch.zeros(len(ell), 1, H, W, device=device, dtype=torch.float64)
    for cx, cy, a, b, phi, rho in ell.to(device).permute(1, 2, 0)[..., None, None]:
        dx, dy = x[None, None, :] - cx, y[None, :, None] - cy
        u = (dx * phi.cos() + dy * phi.sin()) / a
        v = (dy * phi.cos() - dx * phi.sin()) / b
        out[:, 0] += rho * (u * u + v * v <= 1)
    return out


def _rays(options, device):
    """A point and the unit direction of the ray through the middle of every bin, [V, D] each."""
    o = options.double()
    V, D = int(o[0]), int(o[1])
    ang = (torch.arange(V, device=device, dtype=torch.float64) * float(o[7]) + float(o[6]))[:, None]
    r = torch.arange(D, device=device, dtype=torch.float64)[None, :] - D / 2 + 0.5
    if float(o[-1]) == 2:
        t = r * float(o[5]) + float(o[8])
        return t * ang.cos(), t * ang.sin(), (-ang.sin()).expand(V, D), ang.cos().expand(V, D)
    sx, sy = -ang.sin() * float(o[8]), ang.cos() * float(o[8])
    if float(o[-1]) == 0:
        mag = float(o[8]) / (float(o[8]) + float(o[9]))
        t = mag * (r * float(o[5]) + float(o[10]))
        dx, dy = t * ang.cos() - sx, t * ang.sin() - sy
        n = torch.sqrt(dx * dx + dy * dy)
        return sx.expand(V, D), sy.expand(V, D), dx / n, dy / n
    beta = r * float(o[5]) + float(o[10]) + ang
    return sx.expand(V, D), sy.expand(V, D), beta.sin(), -beta.cos()


def _sinogram(ell, options, device, gen):
    """Line integrals of the ellipses with the noise of I0 photons per ray, [B, 1, V, D]."""
    px, py, dx, dy = _rays(options, device)
    out = torch.zeros(len(ell), 1, *px.shape, device=device, dtype=torch.float64)
    for s, one in enumerate(ell.tolist()):
        for cx, cy, a, b, phi, rho in one:
            c, n = math.cos(phi), math.sin(phi)
            ux, uy = ((px - cx) * c + (py - cy) * n) / a, ((py - cy) * c - (px - cx) * n) / b
            wx, wy = (dx * c + dy * n) / a, (dy * c - dx * n) / b
            A, h = wx * wx + wy * wy, ux * wx + uy * wy
            disc = h * h - A * (ux * ux + uy * uy - 1)
            out[s, 0] += 2 * rho * disc.clamp_min(0).sqrt() / A
    noise = torch.randn(out.shape, generator=gen, device=device, dtype=torch.float32)
    return out + noise * torch.exp(out / 2) / math.sqrt(I0)


def _hetero_options(case):
    """Image sizes 256, 384 or 512, 96 to 1152 views, 512, 736 or 1024 bins, all scan types."""
    gen = torch.Generator().manual_seed(case["pick"])

    def pick(values):
        return values[int(torch.randint(len(values), (1,), generator=gen))]

    opts = []
    for _ in range(case["slices"]):
        size = pick((256, 384, 512))
        views = int(torch.randint(96, 1153, (1,), generator=gen))
        opts.append(_options(dict(views=views, dets=pick((512, 736, 1024)), width=size, height=size,
                                  scan=pick(("ed", "ea", "para")))))
    return opts


def _step(options):
    """A stable step of gradient descent: 1 over (longest ray) x (sum of a pixel's weights)."""
    o = options.double()
    side = max(float(o[2]), float(o[3])) * float(o[4])
    bin_width = float(o[5]) * (float(o[8]) / (float(o[8]) + float(o[9])) if float(o[-1]) == 0 else 1.0)
    if float(o[-1]) == 1:
        bin_width *= float(o[8])
    step = 1.0 / (1.5 * side * float(o[0]) * float(o[4]) ** 2 / bin_width)
    return float(torch.tensor(step, dtype=torch.float32))


def _inputs(case, seed):
    """Named input tensors of the case on the GPU, and its options."""
    device = torch.device("cuda")
    gen = torch.Generator().manual_seed(seed)
    noise = torch.Generator(device=device).manual_seed(seed)
    if case["op"] == "laplacian":
        # patches vary around a smooth mean, as image patches do
        x = torch.rand(case["points"], 1, generator=noise, device=device)
        return {"points": x + 0.2 * torch.randn(case["points"], case["dim"], generator=noise, device=device)}, None
    if case["op"] == "hetero":
        opts = _hetero_options(case)
        xs, ms = [], []
        for o in opts:
            ell = _ellipses(1, o, gen)
            xs.append(_image(ell, o, device).float())
            ms.append(_sinogram(ell, o, device, noise).float())
        return {"xs": xs, "ms": ms}, opts
    o = _options(case)
    dtype = torch.float64 if case["dtype"] == "f64" else torch.float32
    ell = _ellipses(case["batch"], o, gen)
    got = {}
    sino = case["op"] not in TO_SINO
    if sino or case["train"]:
        got["sino"] = _sinogram(ell, o, device, noise).to(dtype)
    if not sino or case["train"] or case["op"] in ("residual_step", "least_squares", "unrolled"):
        got["image"] = _image(ell, o, device).to(dtype)
    if case["op"] in ("residual_step", "least_squares"):
        got["image"] *= 0.9  # an iterate of a running reconstruction
    return got, o


def prepare(case, seed):
    got, o = _inputs(case, seed)
    state = dict(got, case=case, options=o)
    if case["op"] == "hetero":
        state["handle"] = batch.HeteroBatch(o, device="cuda:0")
    elif case["op"] == "unrolled":
        state["model"] = recon.UnrolledGD(o, iters=case["iters"], alpha0=_step(o)).cuda()
    elif case["op"] == "least_squares":
        got["image"].requires_grad_(True)
    elif case.get("train"):
        got["image" if case["op"] in TO_SINO else "sino"].requires_grad_(True)
    return state


def run(state):
    case, o, op = state["case"], state["options"], state["case"]["op"]
    if op == "laplacian":
        w = ctlib_amd.laplacian(state["points"], case["k"])
        return {"indices": w._indices(), "values": w._values()}
    if op == "hetero":
        y, grad = state["handle"].run(state["xs"], state["ms"])
        return {"y": y, "grad": grad}
    if op == "residual_step":
        y, grad = ctlib_amd.residual_step(state["image"], state["sino"], o)
        return {"y": y, "grad": grad}
    if op == "least_squares":
        loss = autograd.least_squares(state["image"], state["sino"], o)
        (grad,) = torch.autograd.grad(loss, state["image"])
        return {"loss": loss.detach(), "grad": grad}
    if op == "unrolled":
        model = state["model"]
        x = model(state["sino"])
        (grad,) = torch.autograd.grad(0.5 * ((x - state["image"]) ** 2).sum(), model.alpha)
        return {"image": x.detach(), "alpha_grad": grad}
    name, other = ("image", "sino") if op in TO_SINO else ("sino", "image")
    if case["train"]:
        y = getattr(autograd, op)(state[name], o)
        (grad,) = torch.autograd.grad(y, state[name], state[other])
        return {"out": y.detach(), "grad": grad}
    return {"out": getattr(ctlib_amd, op)(state[name], o)}


# ---- what a pass cannot do without --------------------------------------------------------------


def work(case):
    """One sweep of a slice meets, per view and swept line, pixels + bins overlaps of 2 operations each."""
    es = 8 if case["dtype"] == "f64" else 4
    op = case["op"]
    if op == "laplacian":
        n, d, k = case["points"], case["dim"], case["k"]
        return {"bytes": n * d * es + n * k * (16 + 4), "flops": 2.0 * n * n * d}
    if op == "hetero":
        nbytes = flops = 0
        for o in _hetero_options(case):
            V, D, W, H = (int(v) for v in o[:4])
            nbytes += es * 2 * (V * D + W * H)
            flops += 2 * 2.0 * V * H * (W + D)
        return {"bytes": nbytes, "flops": flops}
    V, D, W, H, B = (case[k] for k in ("views", "dets", "width", "height", "batch"))
    sino, img = V * D, W * H
    sweep = 2.0 * V * (W * H + (W + H) / 2 * D)
    ramp = 2.0 * V * D * (D / 2)  # the taps at even offsets are zero
    sweeps, moved, ramps = 1, sino + img, 0
    if op == "backprojection_sv":
        moved = sino + V * img
    elif op == "residual_step":
        sweeps, moved = 2, 2 * (sino + img)
    elif op == "least_squares":
        sweeps, moved = 2, sino + 2 * img
    elif op == "unrolled":
        # forward and adjoint per iteration, and again for the gradient of every iterate but the first
        sweeps, moved = 2 * (2 * case["iters"] - 1), sino + 2 * img
    elif case["train"]:
        sweeps, moved = 2, 2 * (sino + img)
    if op == "fbp":
        ramps = 2 if case["train"] else 1
    return {"bytes": es * B * moved, "flops": B * (sweeps * sweep + ramps * ramp)}


# ---- the same in 64 bits ------------------------------------------------------------------------


class _Exact:
    """The distance-driven operators of one options vector in float64 torch: per view, both edge grids
    are mapped to the sweep axis and the piecewise-constant line (or bin row) is integrated between the
    edges of the other grid."""

    def __init__(self, options, device):
        o = options.double()
        self.dev = device
        self.V, self.D, self.W, self.H = (int(v) for v in o[:4])
        self.d_img, self.d_det, self.ang0, self.d_ang = (float(v) for v in o[4:8])
        self.scan = int(o[-1])
        if self.scan == 2:
            self.R, self.shift, self.mag = 0.0, float(o[8]), 1.0
        else:
            self.R, self.shift = float(o[8]), float(o[10])
            self.mag = self.R / (self.R + float(o[9])) if self.scan == 0 else 1.0

    def _view(self, v):
        """Sweep axis (x?), ascending?, bin edges, bin factors, pixel edges [lines, n + 1], pixel weights."""
        f64 = dict(device=self.dev, dtype=torch.float64)
        ang = v * self.d_ang + self.ang0
        xmode = abs(ang - round(ang / math.pi) * math.pi) * 4 / math.pi <= 1
        cs, sn = math.cos(ang), math.sin(ang)
        sx, sy = -sn * self.R, cs * self.R
        t = (torch.arange(self.D + 1, **f64) - self.D / 2) * self.d_det + self.shift
        if self.scan == 0:
            px, py = self.mag * t * cs, self.mag * t * sn
            e = (sx * py - sy * px) / (py - sy) if xmode else (sy * px - sx * py) / (px - sx)
        elif self.scan == 1:
            e = sx + torch.tan(t + ang) * sy if xmode else sy + sx / torch.tan(t + ang)
        else:
            e = t / (cs if xmode else sn)
        up = bool(e[-1] > e[0])
        n, lines = (self.W, self.H) if xmode else (self.H, self.W)
        p = (torch.arange(n + 1, **f64) - n / 2) * self.d_img
        if xmode:
            line = (self.H / 2 - torch.arange(lines, **f64) - 0.5) * self.d_img
            if self.scan == 2:
                pe = p[None, :] + sn / cs * line[:, None]
            else:
                pe = (sx * line[:, None] - sy * p[None, :]) / (line[:, None] - sy)
        else:
            line = (torch.arange(lines, **f64) - self.W / 2 + 0.5) * self.d_img
            if self.scan == 2:
                pe = p[None, :] + cs / sn * line[:, None]
            else:
                pe = (sy * line[:, None] - sx * p[None, :]) / (line[:, None] - sx)
        mid = ((p[1:] + p[:-1]) / 2)[None, :]
        x, y = (mid, line[:, None]) if xmode else (line[:, None], mid)
        if self.scan == 0:
            weight = 1 / (1 - (sx * x + sy * y) / self.R ** 2) ** 2
        elif self.scan == 1:
            weight = 1 / ((x - sx) ** 2 + (y - sy) ** 2)
        else:
            weight = torch.ones(1, 1, **f64)
        weight = weight / (pe[:, 1:2] - pe[:, 0:1])
        if self.scan == 2:
            post, post_t = torch.full((self.D,), self.d_img / self.d_det, **f64), None
        else:
            near, far = (sx, sy) if xmode else (sy, sx)
            kap = abs(far) / torch.sqrt((e - near) ** 2 + far ** 2)
            c = (kap[1:] + kap[:-1]) / 2
            post = self.d_img / c / (e[1:] - e[:-1]).abs()
            post_t = self.d_img / c if self.scan == 1 else None
        return xmode, up, e, post, post_t, pe, weight

    def to_sino(self, x, weighted=False, quirk=False):
        """projection; weighted: the transpose of backprojection (quirk: as backprojection_t scales it)."""
        x = x[:, 0].double()
        cols = x.flip(1).transpose(1, 2).contiguous()
        out = torch.empty(len(x), 1, self.V, self.D, device=self.dev, dtype=torch.float64)
        for v in range(self.V):
            xmode, up, e, post, post_t, pe, weight = self._view(v)
            src = x if xmode else cols
            if weighted:
                src = src * weight
            n = src.shape[2]
            s = (pe[:, -1:] - pe[:, :1]) / n
            tau = ((e[None, :] - pe[:, :1]) / s).clamp(0, n)
            j = tau.floor().clamp_max(n - 1).long()[None].expand(len(x), -1, -1)
            cum = torch.cumsum(src, 2) - src
            F = cum.gather(2, j) + (tau[None] - j) * src.gather(2, j)
            S = (s * F).sum(1).diff(dim=1)
            if not up:
                S = -S
            if not weighted:
                S = S * post
            elif quirk and post_t is not None:
                S = S * post_t
            out[:, 0, v] = S
        return out

    def _view_image(self, y, v, weighted, quirk=False):
        xmode, up, e, post, post_t, pe, weight = self._view(v)
        g = y[:, v]
        if not weighted:
            g = g * post
        elif quirk and post_t is not None:
            g = g * post_t
        if not up:
            e, g = e.flip(0), g.flip(1)
        w = e[1:] - e[:-1]
        cum = torch.cumsum(g * w, 1) - g * w
        pi = pe.clamp(float(e[0]), float(e[-1]))
        j = (torch.searchsorted(e, pi.contiguous(), right=True) - 1).clamp(0, self.D - 1)
        G = cum[:, j] + (pi - e[j]) * g[:, j]
        d = G.diff(dim=2)
        return xmode, d * weight if weighted else d

    def to_image(self, y, weighted=False, quirk=False):
        """projection_t; weighted: backprojection (quirk: of the rows scaled as backprojection_t does)."""
        y = y[:, 0].double()
        acc = {True: torch.zeros(len(y), self.H, self.W, device=self.dev, dtype=torch.float64),
               False: torch.zeros(len(y), self.W, self.H, device=self.dev, dtype=torch.float64)}
        for v in range(self.V):
            xmode, d = self._view_image(y, v, weighted, quirk)
            acc[xmode] += d
        return (acc[True] + acc[False].transpose(1, 2).flip(1))[:, None]

    def views(self, y):
        y = y[:, 0].double()
        out = torch.empty(len(y), self.V, self.H, self.W, device=self.dev, dtype=torch.float64)
        for v in range(self.V):
            xmode, d = self._view_image(y, v, True)
            out[:, v] = d if xmode else d.transpose(1, 2).flip(1)
        return out

    def _ramp(self):
        delta = self.mag * self.d_det
        r = torch.arange(self.D, device=self.dev, dtype=torch.float64)
        off = r[:, None] - r[None, :]
        h = torch.where(off.remainder(2) == 1, -1 / (math.pi * off * delta) ** 2, torch.zeros_like(off))
        h.fill_diagonal_(1 / (4 * delta * delta))
        r = r - self.D / 2 + 0.5
        if self.scan == 0:
            pre = self.R / torch.sqrt(self.R ** 2 + (r * delta) ** 2) * delta
        elif self.scan == 1:
            pre = torch.cos(r * self.d_det) * self.R * self.d_det
        else:
            pre = torch.full_like(r, self.d_det)
        return h, pre

    def fbp(self, y):
        h, pre = self._ramp()
        return self.to_image((y.double() * pre) @ h, weighted=True) * (self.d_ang / 2)

    def fbp_t(self, x):
        h, pre = self._ramp()
        return (self.to_sino(x, weighted=True) @ h) * pre * (self.d_ang / 2)

    def apply(self, op, x):
        return {"projection": lambda: self.to_sino(x), "projection_t": lambda: self.to_image(x),
                "backprojection": lambda: self.to_image(x, True), "fbp": lambda: self.fbp(x),
                "backprojection_t": lambda: self.to_sino(x, True, True), "backprojection_sv": lambda: self.views(x)}[op]()

    def adjoint(self, op, g):
        return {"projection": lambda: self.to_image(g), "projection_t": lambda: self.to_sino(g),
                "backprojection": lambda: self.to_sino(g, True), "fbp": lambda: self.fbp_t(g),
                "backprojection_t": lambda: self.to_image(g, True, True)}[op]()


def _exact_laplacian(x, k):
    x = x.double()
    n = len(x)
    dist, cols = [], []
    sq = (x * x).sum(1)
    for part in range(0, n, 2048):
        d = sq[part:part + 2048, None] + sq[None, :] - 2 * x[part:part + 2048] @ x.T
        v, c = torch.topk(d, k, largest=False, sorted=True)
        dist.append(v)
        cols.append(c)
    dist = torch.cat(dist)
    w = torch.exp(-dist / dist.flatten().median())
    return w / w.sum(1, keepdim=True)


def exact(case, seed):
    got, o = _inputs(case, seed)
    op = case["op"]
    if op == "laplacian":
        return {"indices": None, "values": _exact_laplacian(got["points"], case["k"]).reshape(-1)}
    device = torch.device("cuda")
    if op == "hetero":
        ys, grads = [], []
        for x, m, one in zip(got["xs"], got["ms"], o):
            A = _Exact(one, device)
            ys.append(A.to_sino(x))
            grads.append(A.to_image(ys[-1] - m.double()))
        return {"y": ys, "grad": grads}
    A = _Exact(o, device)
    if op in ("residual_step", "least_squares"):
        y = A.to_sino(got["image"])
        r = y - got["sino"].double()
        grad = A.to_image(r)
        return {"y": y, "grad": grad} if op == "residual_step" else {"loss": 0.5 * (r * r).sum(), "grad": grad}
    if op == "unrolled":
        m, a = got["sino"].double(), _step(o)
        x = torch.zeros_like(got["image"], dtype=torch.float64)
        steps = []
        for _ in range(case["iters"]):
            steps.append(A.to_image(A.to_sino(x) - m))
            x = x - a * steps[-1]
        g, grads = x - got["image"].double(), []
        for k in reversed(range(case["iters"])):
            grads.append(-(g * steps[k]).sum())
            if k:
                g = g - a * A.to_image(A.to_sino(g))
        return {"image": x, "alpha_grad": torch.stack(grads[::-1])}
    name, other = ("image", "sino") if op in TO_SINO else ("sino", "image")
    out = A.apply(op, got[name])
    if not case["train"]:
        return {"out": out}
    return {"out": out, "grad": A.adjoint(op, got[other])}
