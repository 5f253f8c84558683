"""What the performance of this framework is measured on: calls of its public
entry points over the sizes it is used at.

listed()            the named cases
draw(rng)           one more case of the same ranges
prepare(case, seed) what a program holds before the call (inputs on the GPU,
                    or on the host where the call takes host data; contexts
                    with their events and plans)
run(state)          one pass through the public entry points, its outputs
work(case)          bytes and operations a pass cannot do without
exact(case, seed)   the outputs in 64 bits from the formulas alone, where
                    that is quick enough (the ellipse test, the kernel and the
                    update of src/2d/strip/reconstruction.h:110-298 and
                    gaussian_kernel.h:45-137)

Lengths are in millimetres except where a case's own pixel size says
otherwise (the command line's defaults are in metres).
"""
import math
import os
import sys

import numpy as np
import torch

_PACKAGE = os.path.join(os.path.dirname(os.path.dirname(
    os.path.abspath(__file__))), "j-pet-mlem-old_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import pystrip  # noqa: E402
from pystrip import hybrid  # noqa: E402

DEVICE = "cuda:0"

# The phantom of a strip case: ellipses (centre z, y, half axes a, b) in units
# of the phantom's half size, and the share of the emissions each gets: a body
# with hot, cold and small regions, as the reconstruction examples have.
REGIONS = [(0.0, 0.0, 1.0, 1.0, 0.60), (-0.33, 0.28, 0.05, 0.05, 0.04),
           (0.28, 0.40, 0.08, 0.08, 0.06), (0.40, 0.0, 0.22, 0.18, 0.08),
           (-0.40, -0.05, 0.20, 0.16, 0.12), (0.0, -0.60, 0.18, 0.15, 0.10)]


def strip(name, kind, n_z, n_y, pixel, events, body_z, body_y, radius, length,
          sigma_z=10.0, sigma_dl=42.0, **more):
    case = {"kind": kind, "n_z": n_z, "n_y": n_y, "pixel": pixel,
            "events": events, "body_z": body_z, "body_y": body_y,
            "radius": radius, "length": length, "sigma_z": sigma_z,
            "sigma_dl": sigma_dl, **more}
    return {"name": name, **case} if name else case


def listed():
    return [
        # a scoring or serving loop: a few events projected through an image
        # that is already on the device, nothing allocated; latency counts
        strip("project-129-events", "project", 256, 160, 2.0, 129, 80, 60,
              350, 500),
        # the smallest whole reconstruction: the command line's own scanner
        # and grid (in metres), a short list, host arrays in and out
        strip("run-100x100-20k", "run", 100, 100, 0.01, 20_011, 0.25, 0.25,
              0.5, 1.0, 0.015, 0.06, blocks=2, iterations=3),
        # an ordinary whole reconstruction: host events to host image,
        # upload, setup and plan included
        strip("run-256x160-1e6", "run", 256, 160, 2.0, 1_000_000, 80, 60, 350,
              500, blocks=2, iterations=5),
        # the reference's legacy --gpu semantics (analytic kernel,
        # sensitivity in the denominator)
        strip("legacy-256x160-1e5", "legacy", 256, 160, 2.0, 100_000, 80, 60,
              350, 500, iterations=2),
        # MLEM iterations of resident events on a grid of odd size, other
        # resolutions than the benchmark's
        strip("mlem-381x203-3e5", "mlem", 381, 203, 1.25, 300_007, 150, 90,
              300, 700, 7.5, 35.0, iterations=4),
        # the benchmark: 2e7 resident events, 1000 x 400 at 1 mm
        strip("mlem-1000x400-2e7", "mlem", 1000, 400, 1.0, 20_000_000, 180,
              140, 400, 1000, iterations=2),
        # ordered subsets on the largest grid, one full iteration
        strip("osem-2000x800-1.6e7", "osem", 2000, 800, 0.5, 16_000_000, 180,
              140, 400, 1000, iterations=1, subsets=16),
        # many independent reconstructions of uneven size iterated together
        {"name": "batch-24", "kind": "batch", "members": 24, "least": 10_000,
         "most": 300_000, "iterations": 10},
        # calibration: log-likelihood and its image and sigma gradients
        strip("loglik-512x256-2e6", "loglik", 512, 256, 1.0, 2_000_000, 120,
              90, 400, 1000, 14.0, 60.0),
        # backward through unrolled iterations
        strip("unrolled-512x256-2e5", "unrolled", 512, 256, 1.0, 200_000, 120,
              90, 400, 1000, 14.0, 60.0, iterations=4),
        # 3D hybrid iterations: the 48-detector test ring ...
        {"name": "hybrid-ring48-5e4", "kind": "hybrid", "detectors": 48,
         "width": 0.02, "pixels": 80, "planes": 80, "fov": 0.2,
         "events": 50_000, "iterations": 2},
        # ... and a ring of the full scanner's radius
        {"name": "hybrid-ring192-1e6", "kind": "hybrid", "detectors": 192,
         "width": 0.014, "pixels": 120, "planes": 80, "fov": 0.3,
         "events": 1_000_000, "iterations": 2},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a kind of call, a grid of any size with pixels of
    0.5-2.5 mm, resolutions around the scanner's, and an event count over the
    range that kind is used at."""
    kind = rng.choice(["project", "run", "legacy", "mlem", "mlem", "osem",
                       "batch", "loglik", "unrolled", "hybrid"])
    if kind == "batch":
        return {"kind": "batch", "members": rng.randint(3, 40),
                "least": _log_uniform(rng, 1_000, 30_000),
                "most": _log_uniform(rng, 30_000, 300_000),
                "iterations": rng.randint(1, 10)}
    if kind == "hybrid":
        detectors = rng.randint(32, 160)
        return {"kind": "hybrid", "detectors": detectors,
                "width": round(2 * math.pi * 0.41 / detectors, 4),
                "pixels": rng.randint(50, 120), "planes": rng.randint(24, 100),
                "fov": 0.25, "events": _log_uniform(rng, 5_000, 1_000_000),
                "iterations": rng.randint(1, 4)}
    pixel = rng.choice([0.5, 0.75, 1.0, 1.25, 1.5, 2.0, 2.5])
    n_z = rng.randint(int(160 / pixel), int(800 / pixel))
    n_y = rng.randint(int(120 / pixel), int(400 / pixel))
    half_z, half_y = n_z * pixel / 2, n_y * pixel / 2
    range_of = {"project": (1, 200_000), "run": (5_000, 2_000_000),
                "legacy": (5_000, 200_000), "mlem": (10_000, 10_000_000),
                "osem": (200_000, 8_000_000), "loglik": (20_000, 3_000_000),
                "unrolled": (20_000, 500_000)}
    # a fine grid has more work per event: fewer of them, so that a drawn
    # case never costs more than the largest listed one
    most = range_of[kind][1] * min(1.0, pixel * pixel)
    more = {"mlem": {"iterations": rng.randint(1, 4)},
            "run": {"blocks": rng.randint(1, 3),
                    "iterations": rng.randint(1, 5)},
            "legacy": {"iterations": rng.randint(1, 3)},
            "osem": {"iterations": 1, "subsets": rng.choice([4, 8, 16])},
            "unrolled": {"iterations": rng.randint(1, 6)}}.get(kind, {})
    return strip(None, kind, n_z, n_y, pixel,
                 _log_uniform(rng, range_of[kind][0], most),
                 round(half_z * rng.uniform(0.25, 0.75), 1),
                 round(half_y * rng.uniform(0.25, 0.75), 1),
                 round(half_y + rng.uniform(50, 250)),
                 round(2 * half_z + rng.uniform(50, 300)),
                 rng.choice([5.0, 7.5, 10.0, 12.0, 14.0]),
                 rng.choice([30.0, 42.0, 60.0]), **more)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _events(case, gen):
    """(n, 3) float32 detected responses z_u, z_d, dl on the GPU: an emission
    in one of the phantom's ellipses, a uniform direction, both ends inside
    the strips, Gaussian errors (src/2d/strip/scanner.h:107-113,196-267)."""
    n, R, half = case["events"], case["radius"], case["length"] / 2
    regions = torch.tensor(REGIONS, dtype=torch.float64, device=DEVICE)
    edges = torch.cumsum(regions[:, 4], 0)
    out = torch.empty((n, 3), dtype=torch.float32, device=DEVICE)
    filled = 0
    while filled < n:
        m = int(min(max(2 * (n - filled), 1024), 1 << 22))
        u = torch.rand((4, m), dtype=torch.float64, device=DEVICE,
                       generator=gen)
        k = torch.bucketize(u[0] * edges[-1], edges).clamp(
            max=len(REGIONS) - 1)
        r = torch.sqrt(u[1])
        angle = 2 * math.pi * u[2]
        z = (regions[k, 0] + regions[k, 2] * r * torch.cos(angle)) \
            * case["body_z"]
        y = (regions[k, 1] + regions[k, 3] * r * torch.sin(angle)) \
            * case["body_y"]
        tan = torch.tan(0.5 * math.pi * (2 * u[3] - 1))
        z_u, z_d = z + (R - y) * tan, z - (R + y) * tan
        dl = -2 * y * torch.sqrt(tan * tan + 1)
        noise = torch.randn((3, m), dtype=torch.float64, device=DEVICE,
                            generator=gen)
        keep = ((z_u.abs() < half) & (z_d.abs() < half)).nonzero()[:, 0]
        keep = keep[:n - filled]
        rows = torch.stack([z_u + case["sigma_z"] * noise[0],
                            z_d + case["sigma_z"] * noise[1],
                            dl + case["sigma_dl"] * noise[2]], 1)[keep]
        out[filled:filled + len(keep)] = rows.to(torch.float32)
        filled += len(keep)
    return out


def _body(case):
    """The phantom's body sampled at the pixel centres: a smooth image."""
    w = case["pixel"]
    z = (torch.arange(case["n_z"], device=DEVICE) + 0.5) * w \
        - case["n_z"] * w / 2
    y = case["n_y"] * w / 2 - (torch.arange(case["n_y"], device=DEVICE)
                               + 0.5) * w
    q = (y[:, None] / case["body_y"]) ** 2 + (z[None] / case["body_z"]) ** 2
    return torch.exp(-0.5 * q)


def _image(case, gen):
    """A positive image like one some iterations in: the body's shape over a
    low background, with noise."""
    body = _body(case)
    noise = torch.rand(body.shape, device=DEVICE, generator=gen)
    return ((body + 0.05) * (0.5 + noise)).to(torch.float32).contiguous()


def _geometry(case):
    return pystrip.Geometry.make(case["radius"], case["length"], case["n_z"],
                                 case["n_y"], case["pixel"], case["sigma_z"],
                                 case["sigma_dl"])


def _members(case):
    """The batch's members: grids and pixel sizes as the batched benchmark
    has them, event counts spread over [least, most]; fixed by the case, so
    that another seed is other events of the same members."""
    rng = np.random.default_rng(case["members"] * 1_000_003 + case["least"])
    out = []
    for _ in range(case["members"]):
        n_z, n_y = [(128, 128), (256, 128), (512, 256), (512, 512)][
            int(rng.integers(4))]
        pixel = 1.0 + 0.25 * float(rng.integers(5))
        n = int(round(math.exp(rng.uniform(math.log(case["least"]),
                                           math.log(case["most"])))))
        half_z, half_y = n_z * pixel / 2, n_y * pixel / 2
        out.append(strip(None, "mlem", n_z, n_y, pixel, n,
                         half_z * 0.8 * rng.uniform(0.6, 1.0),
                         half_y * 0.8 * rng.uniform(0.6, 1.0), half_y + 50,
                         2 * half_z + 100, iterations=case["iterations"]))
    return out


_rings = {}


def _ring(case):
    """A ring's geometry: it does not depend on the events, so a process makes
    it once."""
    key = (case["detectors"], case["width"], case["pixels"], case["planes"],
           case["fov"])
    if key not in _rings:
        _rings.clear()
        _rings[key] = hybrid.ring_geometry(
            case["detectors"], 0.4278 if case["detectors"] > 64 else 0.4,
            case["width"], case["pixels"], 0.005, case["planes"], case["fov"])
    return _rings[key]


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind == "batch":
        state["batch"] = batch = pystrip.Batch(device=0)
        state["start"] = []
        for i, member in enumerate(_members(case)):
            gen = _generator(seed * 1000 + i)
            batch.add(_geometry(member), _events(member, gen).cpu().numpy())
            state["start"].append(_image(member, gen).cpu().numpy())
        batch.iterate(1)
        return state
    if kind == "hybrid":
        geo = _ring(case)
        rec = hybrid.HybridReconstruction(geo)
        rec.prepare_weights(True, 0)
        rec.add_responses(hybrid.hybrid_events(
            geo, case["events"], seed, radius=min(0.25, 0.6 * case["fov"]),
            half_z=0.4 * geo.n_planes * geo.pixel_size))
        rng = np.random.default_rng(seed)
        state["start"] = rng.uniform(0.5, 1.5, geo.shape).astype(np.float32)
        state["rec"] = rec
        rec.iterate(1)
        return state
    gen = _generator(seed)
    events = _events(case, gen)
    image = _image(case, gen)
    state["geometry"] = geometry = _geometry(case)
    if kind == "project":
        state.update(events=events, image=image,
                     out=torch.empty(case["events"], device=DEVICE))
        torch.cuda.synchronize()
        return state
    if kind == "run":
        state.update(events=events.cpu().numpy(), image=image.cpu().numpy())
        return state
    mode = pystrip.MODE_LEGACY_GPU if kind == "legacy" else pystrip.MODE_CPU
    rec = pystrip.Reconstruction(geometry, mode, device=0)
    torch.cuda.synchronize()
    rec.set_events_device(events.data_ptr(), len(events))
    if kind == "osem":
        rec.set_subsets(case["subsets"])
    if kind != "legacy":
        rec.iterate(1)  # builds the plan of the resident events
    state.update(rec=rec, image=image, out=torch.empty_like(image))
    if kind == "unrolled":
        state["target"] = (_body(case) * (case["events"] / image.numel())
                           ).to(torch.float32).contiguous()
    torch.cuda.synchronize()
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "project":
        pystrip.forward_noalloc(
            state["geometry"], state["events"].data_ptr(), case["events"],
            state["image"].data_ptr(), state["out"].data_ptr(),
            stream=torch.cuda.current_stream().cuda_stream)
        return state["out"]
    if kind == "run":
        return pystrip.run(state["geometry"], state["events"], state["image"],
                           case["blocks"], case["iterations"])
    if kind == "batch":
        batch = state["batch"]
        for i, image in enumerate(state["start"]):
            batch.set_rho(i, image)
        batch.iterate(case["iterations"])
        return [batch.rho(i) for i in range(len(state["start"]))]
    rec = state["rec"]
    if kind == "hybrid":
        rec.rho = state["start"]
        rec.iterate(case["iterations"])
        return rec.rho
    if kind == "loglik":
        value, sigma = rec.loglik_gradient_device(state["image"].data_ptr(),
                                                  state["out"].data_ptr())
        return {"value": value, "d_image": state["out"],
                "d_sigma_z": float(sigma[0]), "d_sigma_dl": float(sigma[1])}
    if kind == "unrolled":
        loss, sigma = rec.unrolled_gradient_device(
            state["image"].data_ptr(), case["iterations"],
            state["target"].data_ptr(), state["out"].data_ptr())
        return {"loss": loss, "d_image": state["out"],
                "d_sigma_z": float(sigma[0]), "d_sigma_dl": float(sigma[1])}
    rec.set_rho_device(state["image"].data_ptr())
    rec.iterate(case["iterations"])
    rec.get_rho_device(state["out"].data_ptr())
    return state["out"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _passes(case):
    """Walks over every event's support: a forward and a back-projection of
    each iteration, a forward and a back-projection of each reverse step."""
    return {"project": 1, "loglik": 2}.get(case["kind"]) or \
        2 * case["iterations"] * case.get("blocks", 1) * \
        (2 if case["kind"] == "unrolled" else 1)


def _support(case):
    """Mean pixels of an event's three-sigma ellipse: its area at a mean
    slope, 9 pi / sqrt(det) of the form Q (gaussian_kernel.h:121-123)."""
    area = 9 * math.pi * case["sigma_z"] * case["sigma_dl"] / math.sqrt(8.0)
    return area / case["pixel"] ** 2


def work(case):
    if case["kind"] == "batch":
        parts = [work(m) for m in _members(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    if case["kind"] == "hybrid":
        # a visit: offset, square, exponential, product and sum, twice; the
        # box of an event is about 12 planes by 50 pixels
        n, its = case["events"], case["iterations"]
        voxels = case["pixels"] ** 2 * case["planes"]
        return {"bytes": its * (n * 20.0 + voxels * 8.0),
                "flops": its * n * 600.0 * 15}
    # each pass reads the events (12 bytes) and the image, and writes an image
    # or one number per event; a kernel evaluation is 8 operations
    n, passes = case["events"], _passes(case)
    pixels = case["n_z"] * case["n_y"]
    return {"bytes": passes * (n * 12.0 + pixels * 8.0),
            "flops": passes * n * _support(case) * 8.0}


# ---------------------------------------------------------------------------
# the outputs in 64 bits
# ---------------------------------------------------------------------------

class _Exact:
    """The strip model of one case's events in FP64."""

    CHUNK = 3e7  # box pixels held at once

    def __init__(self, case, events):
        self.n_z, self.n_y = case["n_z"], case["n_y"]
        self.w, self.R = case["pixel"], case["radius"]
        self.iz, self.id = case["sigma_z"] ** -2, case["sigma_dl"] ** -2
        self.norm = self.iz * math.sqrt(self.id) / (2 * math.pi ** 2)
        self.left, self.top = -self.n_z * self.w / 2, self.n_y * self.w / 2
        ev = events.to(torch.float64)
        t = (ev[:, 0] - ev[:, 1]) / (2 * self.R)
        y = -0.5 * ev[:, 2] / torch.sqrt(1 + t * t)
        z = 0.5 * (ev[:, 0] + ev[:, 1] + 2 * y * t)
        A = 4 * (1 + t * t) * self.id + 2 * t * t * self.iz
        B, C = -4 * t * self.iz, 2 * self.iz
        half_y = 3 / torch.sqrt(A - B * B / (4 * C))
        half_z = 3 / torch.sqrt(C - B * B / (4 * A))
        cx = ((z - self.left) / self.w).to(torch.int64)
        cy = ((self.top - y) / self.w).to(torch.int64)
        hw = (half_z / self.w + 0.5).to(torch.int64)
        hh = (half_y / self.w + 0.5).to(torch.int64)
        self.x0 = (cx - hw).clamp(0, self.n_z - 1)
        self.x1 = (cx + hw).clamp(0, self.n_z - 1)
        self.y0 = (cy - hh).clamp(0, self.n_y - 1)
        self.y1 = (cy + hh).clamp(0, self.n_y - 1)
        self.t, self.y, self.z, self.A, self.B, self.C = t, y, z, A, B, C
        self.n = len(ev)
        self.width = int((self.x1 - self.x0).max())
        self.height = int((self.y1 - self.y0).max())
        self.boxes = self.n * float(max(self.width, 1) * max(self.height, 1))

    def kernels(self):
        """(slice, K, pixel index, Qz, Qd, w) of the events, chunk by chunk;
        K is 0 outside the support."""
        if self.width < 1 or self.height < 1:
            return
        step = max(1, int(self.CHUNK / (self.width * self.height)))
        col = torch.arange(self.width, device=DEVICE)
        row = torch.arange(self.height, device=DEVICE)
        for lo in range(0, self.n, step):
            s = slice(lo, min(lo + step, self.n))
            ix = self.x0[s, None] + col
            iy = self.y0[s, None] + row
            dz = (self.left + self.w / 2 + ix * self.w
                  - self.z[s, None])[:, None, :]
            py = self.top - self.w / 2 - iy * self.w
            dy = (py - self.y[s, None])[:, :, None]
            t = self.t[s, None, None]
            sec2 = 1 + t * t
            # the row's prefactor: a . Sigma^-1 . a (gaussian_kernel.h:58-74)
            yp = py[:, :, None]
            across = 2 * self.iz * sec2 * sec2 * (yp * yp + self.R ** 2)
            along = 4 * self.id * sec2 * t * t * yp * yp
            w = across / (across + along)
            Qd = 4 * self.id * sec2 * dy * dy
            shift = dz - t * dy
            Qz = 2 * self.iz * shift * shift
            Q = Qz + Qd
            inside = (Q <= 9) & (ix < self.x1[s, None])[:, None, :] & \
                (iy < self.y1[s, None])[:, :, None]
            K = torch.where(inside, torch.exp(-0.5 * Q) * self.norm
                            / torch.sqrt(across + along), 0.0)
            at = iy.clamp(max=self.n_y - 1)[:, :, None] * self.n_z + \
                ix.clamp(max=self.n_z - 1)[:, None, :]
            yield s, K, at, Qz, Qd, w

    def project(self, image):
        flat = image.reshape(-1)
        out = torch.zeros(self.n, dtype=torch.float64, device=DEVICE)
        for s, K, at, *_ in self.kernels():
            out[s] = (K * flat[at]).sum((1, 2))
        return out

    def moments(self, images):
        """Per image: sum K x, sum K x dlnK/dln sigma_z, ... sigma_dl."""
        out = [torch.zeros((3, self.n), dtype=torch.float64, device=DEVICE)
               for _ in images]
        for s, K, at, Qz, Qd, w in self.kernels():
            for o, image in zip(out, images):
                Kx = K * image.reshape(-1)[at]
                o[0, s] = Kx.sum((1, 2))
                o[1, s] = (Kx * (Qz + w - 2)).sum((1, 2))
                o[2, s] = (Kx * (Qd - w)).sum((1, 2))
        return out

    def back_project(self, weights):
        out = torch.zeros(self.n_y * self.n_z, dtype=torch.float64,
                          device=DEVICE)
        for s, K, at, *_ in self.kernels():
            out.index_add_(0, at.reshape(-1),
                           (K * weights[s, None, None]).reshape(-1))
        return out.reshape(self.n_y, self.n_z)

    @staticmethod
    def inverse(D):
        return torch.where(D > 0, 1 / D, torch.zeros_like(D))


def _exact_mlem(case, events, image, iterations):
    """MLEM (subsets by event index with the count ratio, or all events)."""
    subsets = case.get("subsets", 1)
    bounds = [len(events) * s // subsets for s in range(subsets + 1)]
    models = [_Exact(case, events[a:b])
              for a, b in zip(bounds[:-1], bounds[1:])]
    if sum(m.boxes for m in models) * 2 * iterations > 2e11:
        return None
    rho = image.to(torch.float64)
    for _ in range(iterations):
        for m in models:
            back = m.back_project(m.inverse(m.project(rho)))
            rho = rho * back * (len(events) / m.n)
    return rho


def exact(case, seed):
    kind = case["kind"]
    if kind in ("legacy", "hybrid"):
        return None  # their outputs follow the reference's own quirks
    if kind == "batch":
        out = []
        for i, member in enumerate(_members(case)):
            gen = _generator(seed * 1000 + i)
            events = _events(member, gen)
            out.append(_exact_mlem(member, events, _image(member, gen),
                                   case["iterations"])
                       if case["iterations"] * case["most"] < 1e6 else None)
        return out if any(o is not None for o in out) else None
    gen = _generator(seed)
    events = _events(case, gen)
    image = _image(case, gen).to(torch.float64)
    if kind in ("run", "mlem", "osem"):
        if len(events) > 4e6:
            return None
        return _exact_mlem(case, events, image, case["iterations"]
                           * case.get("blocks", 1))
    m = _Exact(case, events)
    if m.boxes * _passes(case) > 2e11:
        return None
    if kind == "project":
        return m.project(image)
    if kind == "loglik":
        Kx, Zz, Zd = m.moments([image])[0]
        inv = m.inverse(Kx)
        value = torch.log(torch.where(Kx > 0, Kx, torch.ones_like(Kx))).sum() \
            - image.sum()
        return {"value": float(value), "d_image": m.back_project(inv) - 1,
                "d_sigma_z": float((Zz * inv).sum()) / case["sigma_z"],
                "d_sigma_dl": float((Zd * inv).sum()) / case["sigma_dl"]}
    # unrolled: the iterations, then the reverse steps of
    # rho' = rho * sum_e K / D
    rhos, backs = [image], []
    for _ in range(case["iterations"]):
        backs.append(m.back_project(m.inverse(m.project(rhos[-1]))))
        rhos.append(rhos[-1] * backs[-1])
    target = (_body(case) * (case["events"] / image.numel())
              ).to(torch.float32).to(torch.float64)
    diff = rhos[-1] - target
    bar = 2 * diff / diff.numel()
    d_z = d_d = 0.0
    for rho, back in zip(rhos[-2::-1], backs[::-1]):
        (D, z0, d0), (G, z1, d1) = m.moments([rho, bar * rho])
        inv = m.inverse(D)
        d_z += float(((z1 - z0 * G * inv) * inv).sum())
        d_d += float(((d1 - d0 * G * inv) * inv).sum())
        bar = bar * back - m.back_project(G * inv * inv)
    return {"loss": float((diff * diff).mean()), "d_image": bar,
            "d_sigma_z": d_z / case["sigma_z"],
            "d_sigma_dl": d_d / case["sigma_dl"]}
