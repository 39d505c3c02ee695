"""The work that programs have this package do, as cases that can be timed.

Every case goes through the public entry points (``dpt.torch.Projector`` and
``torch.autograd.grad``, ``Projector.adjoint_gather``,
``dpt.serving.PoseFitEngine``, ``dpt.transport.simulate``).  ``listed()`` names
the typical ones, ``draw()`` gives others of the same ranges, ``prepare()``
makes what a program holds before the call, ``run()`` is one call, ``work()``
its unavoidable bytes and operations, ``tolerance()`` how closely two correct
implementations agree, and ``exact()`` the same results from plain torch in 64
bits.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from dpt import phantoms, serving, transport
from dpt.geometry import BatchedGeometry, DetectorGeometry
from dpt.torch import Projector
from dpt.volumes import GridSpec

DEVICE = "cuda:0"


def _project(name, grid, spacing, views, arc, panel, samples, *, precision="fp32", storage="float32",
             integration="midpoint", volume=True, pose=True, gather=False, tilt=0.0, sod=1000.0, sdd=1500.0,
             window=1.0):
    """A projection case: ``grid`` (nz, ny, nx), ``spacing`` (x, y, z) mm, views
    spread over ``arc`` degrees, ``panel`` (rows, columns), cotangent on the
    central ``window`` of the panel, ``tilt`` the grid's rotation about z."""
    case = dict(kind="project", nz=grid[0], ny=grid[1], nx=grid[2], hx=spacing[0], hy=spacing[1], hz=spacing[2],
                views=views, arc=arc, rows=panel[0], cols=panel[1], samples=samples, precision=precision,
                storage=storage, integration=integration, volume=volume, pose=pose, gather=gather, tilt=tilt,
                sod=sod, sdd=sdd, window=window)
    return dict(case, name=name) if name else case


def _fit(name, n, requests, views, panel, samples, iterations, storage="bfloat16"):
    case = dict(kind="fit", nz=n, ny=n, nx=n, requests=requests, views=views, panel=panel, samples=samples,
                iterations=iterations, storage=storage)
    return dict(case, name=name) if name else case


def _transport(name, n, panel, histories, spectrum):
    case = dict(kind="transport", n=n, panel=panel, histories=histories, spectrum=spectrum)
    return dict(case, name=name) if name else case


def listed():
    return [
        # a rendered preview of a coarse volume, no gradients: launches and latency
        _project("preview", (64, 64, 64), (4.0, 4.0, 4.0), 1, 0.0, (64, 64), 128, volume=False, pose=False),
        # one evaluation of a pose search on a coarse pyramid level: image and pose gradient
        _project("search", (128, 128, 128), (2.0, 2.0, 2.0), 1, 0.0, (128, 128), 256, volume=False),
        # one registration request on a chest CT: one view, image, volume and pose gradients
        _project("request", (139, 512, 512), (0.762, 0.762, 2.5), 1, 0.0, (512, 512), 1024, sod=600.0, sdd=1200.0),
        # odd sizes throughout: seven views of an anisotropic tilted grid on a ragged panel
        _project("ragged", (97, 181, 203), (1.1, 0.9, 1.7), 7, 200.0, (257, 301), 517, tilt=17.0),
        # one gradient step of an iterative sparse-view reconstruction (volume only)
        _project("recon", (128, 128, 128), (2.0, 2.0, 2.0), 60, 360.0, (256, 256), 512, pose=False),
        # the full circular scan: joint calibration and reconstruction step
        _project("fullscan", (256, 256, 256), (1.0, 1.0, 1.0), 360, 360.0, (512, 512), 1024),
        # the same step on a volume held in bfloat16
        _project("half", (256, 256, 256), (1.0, 1.0, 1.0), 24, 360.0, (256, 256), 1024, storage="bfloat16"),
        # strict double precision: reference images, gradient checks
        _project("double", (128, 128, 128), (2.0, 2.0, 2.0), 24, 360.0, (256, 256), 512, precision="fp64"),
        # the exact integration rule
        _project("gauss", (128, 128, 128), (2.0, 2.0, 2.0), 24, 360.0, (256, 256), 512, precision="fp64",
                 integration="cell_gauss"),
        # reproducible back-projection of a double residual
        _project("gather", (128, 128, 128), (2.0, 2.0, 2.0), 24, 360.0, (256, 256), 512, precision="fp64",
                 gather=True),
        # Monte Carlo primary and scatter images of a 40-120 keV spectrum
        _transport("transport", 128, 256, 10_000_000, True),
        # pose-fit requests served together on resident volumes
        _fit("fit", 128, 6, 3, 192, 384, 10),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["small", "small", "request", "scan", "scan", "half", "double", "gauss", "gather", "transport",
                       "fit"])
    if kind == "transport":
        return _transport(None, rng.choice([48, 64, 96, 128]), _log(rng, 32, 256), _log(rng, 100_000, 10_000_000),
                          rng.random() < 0.5)
    if kind == "fit":
        return _fit(None, _log(rng, 48, 160), rng.randint(1, 8), rng.randint(2, 5), _log(rng, 64, 256),
                    _log(rng, 128, 640), rng.randint(4, 12), rng.choice(["bfloat16", "float32"]))
    if kind == "small":
        grid = tuple(_log(rng, 24, 128) for _ in range(3))
        views, panel, samples = rng.randint(1, 4), (_log(rng, 24, 192), _log(rng, 24, 192)), _log(rng, 48, 400)
    elif kind == "request":
        grid = (_log(rng, 60, 200), _log(rng, 200, 512), _log(rng, 200, 512))
        views, panel, samples = rng.randint(1, 3), (_log(rng, 200, 600), _log(rng, 200, 600)), _log(rng, 300, 1100)
    else:
        top = 300 if kind in ("scan", "half") else 150
        grid = tuple(_log(rng, 48, top) for _ in range(3))
        views, panel = _log(rng, 8, 180 if kind == "scan" else 40), (_log(rng, 80, 400), _log(rng, 80, 400))
        samples = _log(rng, 128, 1024)
    extent = rng.uniform(180.0, 400.0)
    spacing = tuple(round(extent / n * rng.uniform(0.7, 1.0), 3) for n in reversed(grid))
    volume = rng.random() < 0.7
    pose = rng.random() < 0.7 or (kind != "small" and not volume)
    gather = kind == "gather"
    return _project(None, grid, spacing, views, rng.choice([0.0, 40.0, 200.0, 360.0]) if views > 1 else 0.0, panel,
                    samples, precision="fp64" if kind in ("double", "gauss", "gather") else "fp32",
                    storage=rng.choice(["bfloat16", "float16"]) if kind == "half" else "float32",
                    integration="cell_gauss" if kind == "gauss" else "midpoint", volume=volume, pose=pose,
                    gather=gather, tilt=round(rng.uniform(-30.0, 30.0), 1), sod=round(rng.uniform(600.0, 1100.0), 1),
                    sdd=round(rng.uniform(1200.0, 1700.0), 1), window=rng.choice([1.0, 1.0, 1.0, 0.4]))


# ---------------------------------------------------------------- inputs ----


def _grid(case):
    shape = (case["nz"], case["ny"], case["nx"])
    h = (case.get("hx", 2.0), case.get("hy", 2.0), case.get("hz", 2.0))
    c, s = math.cos(math.radians(case.get("tilt", 0.0))), math.sin(math.radians(case.get("tilt", 0.0)))
    middle = [-(n - 1) * d / 2 for n, d in zip(reversed(shape), h)]
    origin = (c * middle[0] - s * middle[1], s * middle[0] + c * middle[1], middle[2])
    return GridSpec(shape, h, origin, (c, -s, 0.0, s, c, 0.0, 0.0, 0.0, 1.0))


def _panels(grid, angles, shape, sod, sdd):
    """(views, 12) panel records: source, pixel (0, 0), column step, row step;
    a square pitch at which the panel just covers the magnified grid."""
    n = grid.xyz
    diagonal = math.hypot(n[0] * grid.spacing_mm[0], n[1] * grid.spacing_mm[1])
    height = n[2] * grid.spacing_mm[2]
    magnified = sdd / (sod - diagonal / 2)
    pitch = 1.02 * magnified * max(diagonal / shape[1], height / shape[0])
    out = []
    for a in angles:
        c, s = math.cos(a), math.sin(a)
        u, away = np.array([c, s, 0.0]), np.array([-s, c, 0.0])
        v = np.array([0.0, 0.0, 1.0])
        first = (sdd - sod) * away - 0.5 * pitch * ((shape[1] - 1) * u + (shape[0] - 1) * v)
        out.append(np.concatenate([-sod * away, first, pitch * u, pitch * v]))
    return np.asarray(out)


def _geometry(panels, shape):
    views = []
    for p in panels:
        pitch = float(np.linalg.norm(p[6:9]))
        views.append(DetectorGeometry(tuple(map(float, p[:3])), tuple(map(float, p[3:6])),
                                      tuple(map(float, p[6:9] / pitch)), tuple(map(float, p[9:12] / pitch)),
                                      (pitch, pitch), tuple(shape)))
    return BatchedGeometry(tuple(views))


def _angles(case):
    span = case["views"] if case["arc"] >= 360.0 else max(case["views"] - 1, 1)
    return [math.pi + math.radians(case["arc"]) * k / span for k in range(case["views"])]


def _case_panels(case):
    return _panels(_grid(case), _angles(case), (case["rows"], case["cols"]), case["sod"], case["sdd"])


def _phantom(grid, seed):
    """The package's chest ellipsoids with noise, evaluated on the device."""
    g = torch.Generator(DEVICE).manual_seed(seed)
    nx, ny, nz = grid.xyz
    out = torch.zeros(grid.shape, device=DEVICE)
    flat = GridSpec(grid.shape, grid.spacing_mm, tuple(-(n - 1) * h / 2 for n, h in zip(grid.xyz, grid.spacing_mm)))
    axes = [flat.origin_mm[a] + flat.spacing_mm[a] * torch.arange(n, device=DEVICE) for a, n in enumerate(grid.xyz)]
    for e in phantoms.chest_ellipsoids(flat, seed):
        x, y, z = (((axes[a] - e.centre_mm[a]) / e.axes_mm[a]) ** 2 for a in range(3))
        inside = z.view(nz, 1, 1) + y.view(1, ny, 1) + x.view(1, 1, nx) <= 1.0
        out.masked_fill_(inside, e.attenuation_mm_inverse)
    out += 1e-4 * torch.randn(grid.shape, generator=g, device=DEVICE)
    return out.clamp_(min=0.0)


def _tangent(seed, mm=4.0, rad=0.03):
    rng = np.random.default_rng(seed)
    return np.concatenate([rng.uniform(-mm, mm, 3), rng.uniform(-rad, rad, 3)])


def _target(case, seed):
    """A measured image: a smooth pattern of the optical depths a chest shows, with noise."""
    g = torch.Generator(DEVICE).manual_seed(seed + 7)
    coarse = torch.rand((case["views"], 1, 9, 9), generator=g, device=DEVICE)
    shape = (case["rows"], case["cols"])
    smooth = torch.nn.functional.interpolate(coarse, size=shape, mode="bilinear", align_corners=True)[:, 0]
    target = 4.0 * smooth + 0.01 * torch.randn((case["views"], *shape), generator=g, device=DEVICE)
    return target.double() if case["precision"] == "fp64" else target


def _window(case):
    w, (r, c) = case["window"], (case["rows"], case["cols"])
    if w >= 1.0:
        return None
    mask = torch.zeros((1, r, c), dtype=torch.float64 if case["precision"] == "fp64" else torch.float32, device=DEVICE)
    mask[:, int(r * (1 - w) / 2): math.ceil(r * (1 + w) / 2), int(c * (1 - w) / 2): math.ceil(c * (1 + w) / 2)] = 1.0
    return mask


def prepare(case, seed):
    if case["kind"] == "transport":
        spec, physical, labels, absorption, scattering, density, source = transport.chest_transport_scene(
            seed=seed, shape=(case["n"],) * 3, detector=(case["panel"],) * 2, spectrum=case["spectrum"])
        workspace = transport.prepare_transport(spec, material_ids=labels, absorption=absorption,
                                                scattering=scattering, max_histories=case["histories"],
                                                physical=physical)
        return dict(kind="transport", density=density, source=source,
                    batch=transport.HistoryBatch(seed, 0, case["histories"]),
                    workspace=transport.prepare_simulation(workspace))
    if case["kind"] == "fit":
        return _prepare_fit(case, seed)
    grid = _grid(case)
    state = dict(kind="project", volume=case["volume"], pose=case["pose"], gather=case["gather"],
                 module=Projector(grid=grid, geometry=_geometry(_case_panels(case), (case["rows"], case["cols"])),
                                  precision=case["precision"], samples_per_ray=case["samples"],
                                  storage=case["storage"], integration=case["integration"]),
                 target=_target(case, seed), window=_window(case),
                 xi=torch.tensor(_tangent(seed), device=DEVICE, requires_grad=case["pose"] and not case["gather"]))
    if case["gather"]:
        if state["window"] is not None:
            state["target"] = state["target"] * state["window"]
    else:
        state["field"] = _phantom(grid, seed).requires_grad_(case["volume"])
    return state


def _prepare_fit(case, seed):
    shape, count = (case["panel"],) * 2, case["requests"]
    registry = serving.VolumeRegistry(DEVICE)
    grid = _grid(case)
    fields = [_phantom(grid, seed + 100 * i) for i in range(2)]
    for i, field in enumerate(fields):
        registry.add("volume%d" % i, field.cpu().numpy(), grid, storage=case["storage"])
    rng = np.random.default_rng(seed)
    requests = []
    for j in range(count):
        panels = _panels(grid, rng.uniform(0.0, 2 * math.pi, case["views"]), shape, 1000.0, 1500.0)
        packed = _compose(torch.tensor(_tangent(seed + j, 12.0, 0.1), device=DEVICE))
        image = _march(grid, panels, shape, case["samples"], fields[j % 2], packed)["image"].float()
        image += 1e-3 * torch.randn(image.shape, generator=torch.Generator(DEVICE).manual_seed(seed + j), device=DEVICE)
        requests.append(serving.FitRequest("request%03d" % j, "volume%d" % (j % 2), _geometry(panels, shape),
                                           image.cpu().numpy(), case["samples"], case["iterations"]))
    engine = serving.PoseFitEngine(registry, max_requests=16, max_tiles=1 << 16)
    return dict(kind="fit", engine=engine, requests=requests)


# ------------------------------------------------------------------ calls ----


def run(state):
    if state["kind"] == "transport":
        r = transport.simulate(state["density"], source=state["source"], batch=state["batch"],
                               workspace=state["workspace"])
        return {"mean": r.mean, "variance": r.estimated_variance_of_mean, "primary": r.primary_mean,
                "primary_variance": r.primary_variance_of_mean, "scatter": r.scatter_mean,
                "scatter_variance": r.scatter_variance_of_mean, "statuses": list(r.status_histogram.counts)}
    if state["kind"] == "fit":
        results = sorted(state["engine"].run(state["requests"], realtime=False).results, key=lambda r: r.key)
        return {"pose": np.stack([r.pose for r in results]), "loss": np.asarray([r.loss for r in results]),
                "evaluations": np.asarray([r.evaluations for r in results])}
    module = state["module"]
    if state["gather"]:
        return {"volume": module.adjoint_gather(state["target"], state["xi"])}
    if not state["volume"] and not state["pose"]:
        with torch.no_grad():
            return {"image": module(state["field"], state["xi"])}
    image = module(state["field"], state["xi"])
    residual = image.detach() - state["target"]
    if state["window"] is not None:
        residual = residual * state["window"]
    inputs = ([state["field"]] if state["volume"] else []) + ([state["xi"]] if state["pose"] else [])
    gradients = list(torch.autograd.grad(image, inputs, residual))
    out = {"image": image.detach()}
    if state["volume"]:
        out["volume"] = gradients.pop(0)
    if state["pose"]:
        out["pose"] = gradients.pop(0)
    return out


# ------------------------------------------------------- bytes, operations ----


def _hits(grid, panels, shape):
    """Share of the rays that meet the grid's support, and the mean number of
    interpolation planes that such a ray crosses, on a lattice of pixels."""
    ys, xs = np.linspace(0, shape[0] - 1, 24), np.linspace(0, shape[1] - 1, 24)
    picked = panels[:: max(1, len(panels) // 12)]
    end = picked[:, None, None, 3:6] + xs[None, None, :, None] * picked[:, None, None, 6:9] \
        + ys[None, :, None, None] * picked[:, None, None, 9:12]
    matrix = np.asarray(grid.object_to_grid_matrix()).reshape(3, 3)
    o = (picked[:, None, None, :3] - np.asarray(grid.origin_mm)) @ matrix.T
    d = (end - picked[:, None, None, :3]) @ matrix.T
    d = np.where(d == 0.0, 1e-300, d)
    t0, t1 = (-0.5 - o) / d, (np.asarray(grid.xyz) - 0.5 - o) / d
    lower = np.maximum(np.minimum(t0, t1).max(-1), 0.0)
    upper = np.minimum(np.maximum(t0, t1).min(-1), 1.0)
    hit = upper > lower
    crossed = (np.abs(d).sum(-1) * (upper - lower))[hit].mean() if hit.any() else 0.0
    return float(hit.mean()), float(crossed)


def work(case):
    """Operations per sample: 27 place it (position, cell, eight weights), 16
    interpolate, 51 form and sum its slopes, 16 add it to eight voxels."""
    if case["kind"] == "transport":
        # four image pairs; a dozen random draws and 60 further operations per
        # event, about 12 events per history, and its score
        return {"bytes": 6 * 8 * case["panel"] ** 2 + case["n"] ** 3, "flops": 12 * 180.0 * case["histories"]}
    grid = _grid(case)
    voxels = case["nz"] * case["ny"] * case["nx"]
    if case["kind"] == "fit":
        shape = (case["panel"],) * 2
        panels = _panels(grid, [0.3 + 0.7 * k for k in range(case["views"])], shape, 1000.0, 1500.0)
        rays = case["requests"] * case["views"] * shape[0] * shape[1]
        samples = rays * case["samples"] * _hits(grid, panels, shape)[0]
        element = 4 if case["storage"] == "float32" else 2
        return {"bytes": case["iterations"] * (2 * voxels * element + 4 * rays),
                "flops": case["iterations"] * (samples * 94.0 + rays * 90.0)}
    shape = (case["rows"], case["cols"])
    hit, crossed = _hits(grid, _case_panels(case), shape)
    rays = case["views"] * shape[0] * shape[1]
    element = 8 if case["precision"] == "fp64" else 4
    samples = rays * hit * (2 * crossed if case["integration"] == "cell_gauss" else case["samples"])
    seen = samples * min(1.0, case["window"] ** 2 / hit if hit else 1.0)
    if case["gather"]:
        return {"bytes": rays * 8 + voxels * 8, "flops": seen * 43.0}
    flops, moved = samples * 43.0, voxels * 4 + rays * element
    if case["pose"]:
        flops += seen * (27.0 + 16.0 + 51.0)
        moved += voxels * 4
    if case["volume"]:
        flops += seen * (16.0 if case["pose"] else 43.0)
        moved += voxels * 4
    return {"bytes": moved + (rays * element if case["pose"] or case["volume"] else 0), "flops": flops}


def tolerance(case):
    """About four times the distance from ``exact()``: FP32 sampling rounds an
    image to 9e-7, a volume gradient to 3e-5 and a pose gradient, in which the
    residual's signs cancel, to 6e-4; FP64 sampling a volume of FP32-rounded
    additions to 2.4e-8, a pose to 4e-11, an image or an FP64 gather to 1e-14."""
    # counts of histories divided by their number: the same whatever the order
    # in which they are added
    if case["kind"] == "transport":
        return "exact"
    # ten damped steps of FP32 normal equations from FP32 rays
    if case["kind"] == "fit":
        return {"rel": 1e-4, "max": 1e-3}
    if case["gather"]:
        return {"rel": 1e-13}
    if case["precision"] == "fp64":
        return {"rel": 1e-7 if case["volume"] else 2e-10 if case["pose"] else 1e-13}
    return {"rel": 2.5e-3 if case["pose"] else 1e-4 if case["volume"] else 4e-6}


# ------------------------------------------------------------ 64-bit values ----


def _compose(xi):
    """Packed pose exp(hat(xi)): row-major rotation, then translation."""
    zero = xi.new_zeros(())
    hat = torch.stack([zero, -xi[5], xi[4], xi[0], xi[5], zero, -xi[3], xi[1], -xi[4], xi[3], zero, xi[2],
                       zero, zero, zero, zero]).reshape(4, 4)
    e = torch.linalg.matrix_exp(hat)
    return torch.cat([e[:3, :3].reshape(9), e[:3, 3]])


def _rays(grid, panel, pixels, cols, packed):
    """Origins, directions (grid units), lengths and clipped intervals of one view's pixels."""
    p = torch.tensor(panel, dtype=torch.float64, device=packed.device)
    r, c = (pixels // cols).double(), (pixels % cols).double()
    end = p[3:6] + c[:, None] * p[6:9] + r[:, None] * p[9:12]
    matrix = torch.tensor(grid.object_to_grid_matrix(), dtype=torch.float64, device=packed.device).reshape(3, 3)
    rotation, shift = packed[:9].reshape(3, 3), packed[9:]
    origin = torch.tensor(grid.origin_mm, dtype=torch.float64, device=packed.device)
    o = ((p[:3] - shift) @ rotation - origin) @ matrix.T
    d = ((end - p[:3]) @ rotation) @ matrix.T
    n = torch.tensor(grid.xyz, dtype=torch.float64, device=packed.device)
    t0, t1 = (-0.5 - o) / d, (n - 0.5 - o) / d
    lower = torch.minimum(t0, t1).amax(-1).clamp(min=0.0)
    upper = torch.maximum(t0, t1).amin(-1).clamp(max=1.0)
    return o.expand_as(d), d, (end - p[:3]).norm(dim=-1), lower, upper


class _Corners:
    """Cells, weights, values and slopes of a batch of points in grid units."""

    def __init__(self, grid, points, field, values=True, slopes=False):
        n, top = grid.xyz, [m - 1 for m in grid.xyz]
        low, frac = [], []
        for a in range(3):
            q = points[..., a].clamp(0.0, top[a])
            cell = q.floor().clamp(max=max(n[a] - 2, 0))
            low.append(cell.long())
            frac.append(q - cell)
        self.weights, self.index = [], []
        step = (1 if n[0] > 1 else 0, n[0] if n[1] > 1 else 0, n[0] * n[1] if n[2] > 1 else 0)
        base = (low[2] * n[1] + low[1]) * n[0] + low[0]
        parts = [(1.0 - f, f) for f in frac]
        corner = []
        for k in range(8):
            b = (k & 1, k >> 1 & 1, k >> 2)
            self.index.append(base + sum(s * t for s, t in zip(step, b)))
            self.weights.append(parts[0][b[0]] * parts[1][b[1]] * parts[2][b[2]])
            if values:
                corner.append(field[self.index[-1]])
        self.value = sum(w * v for w, v in zip(self.weights, corner)) if values else None
        if slopes:
            out = []
            for a in range(3):
                i, j = [x for x in range(3) if x != a]
                total = 0.0
                for k in range(8):
                    b = (k & 1, k >> 1 & 1, k >> 2)
                    total = total + (1.0 if b[a] else -1.0) * parts[i][b[i]] * parts[j][b[j]] * corner[k]
                live = (points[..., a] >= 0.0) & (points[..., a] < top[a])
                out.append(torch.where(live, total, 0.0))
            self.slopes = torch.stack(out, -1)


def _march(grid, panels, shape, samples, field, packed, *, gauss=False, cotangent=None, want_volume=False,
           want_pose=False, chunk=12_000_000):
    """Optical depths and, with ``cotangent`` (a function of one view's number
    and image), the volume and packed-pose gradients; plain torch, FP64."""
    flat = None if field is None else field.reshape(-1).double()
    views, pixels = len(panels), shape[0] * shape[1]
    image = torch.zeros((views, pixels), dtype=torch.float64, device=DEVICE)
    volume = torch.zeros(math.prod(grid.shape), dtype=torch.float64, device=DEVICE) if want_volume else None
    pose = torch.zeros(12, dtype=torch.float64, device=DEVICE) if want_pose else None
    per = sum(grid.xyz) + 1 if gauss else samples
    rays_at_once = max(1, chunk // (per * (2 if gauss else 1)))

    def nodes(o, d, lower, upper):
        """Positions along the rays and the share of the interval each stands for."""
        if not gauss:
            step = (upper - lower) / samples
            k = torch.arange(samples, dtype=torch.float64, device=DEVICE) + 0.5
            return lower[:, None] + k * step[:, None], step[:, None].expand(-1, samples)
        cuts = [lower[:, None], upper[:, None]]
        for a, n in enumerate(grid.xyz):
            planes = torch.arange(n, dtype=torch.float64, device=DEVICE)
            t = (planes - o[:, a:a + 1]) / d[:, a:a + 1]
            cuts.append(torch.minimum(torch.maximum(t, lower[:, None]), upper[:, None]))
        cuts = torch.cat(cuts, 1).sort(1).values
        radius = (cuts[:, 1:] - cuts[:, :-1]) / 2
        centre = cuts[:, :-1] + radius
        return torch.cat([centre - radius / math.sqrt(3.0), centre + radius / math.sqrt(3.0)], 1), \
            torch.cat([radius, radius], 1)

    for view in range(views):
        every = torch.arange(pixels, device=DEVICE)
        o, d, length, lower, upper = _rays(grid, panels[view], every, shape[1], packed.detach())
        hit = every[upper > lower]
        if field is not None:
            for part in hit.split(rays_at_once):
                at, share = nodes(o[part], d[part], lower[part], upper[part])
                c = _Corners(grid, o[part, None] + at[..., None] * d[part, None], flat)
                image[view, part] = length[part] * (c.value * share).sum(1)
        if cotangent is None:
            continue
        seed = cotangent(view, image[view])
        for part in hit[seed[hit] != 0.0].split(rays_at_once):
            at, share = nodes(o[part], d[part], lower[part], upper[part])
            c = _Corners(grid, o[part, None] + at[..., None] * d[part, None], flat, field is not None, want_pose)
            factor = (seed[part] * length[part])[:, None] * share
            if want_volume:
                for k in range(8):
                    volume.index_add_(0, c.index[k].reshape(-1), (factor * c.weights[k]).reshape(-1))
            if want_pose:
                leaf = packed.detach().clone().requires_grad_(True)
                ro, rd, _, rl, ru = _rays(grid, panels[view], part, shape[1], leaf)
                integral = (c.value * share).sum(1)
                weighted = c.slopes * share[..., None]
                s0, s1 = weighted.sum(1), (weighted * at[..., None]).sum(1)
                linear = (s0 * ro + s1 * rd).sum(-1)
                if gauss:
                    ends = [_Corners(grid, o[part] + t[part, None] * d[part], flat).value for t in (lower, upper)]
                    linear = linear + ends[1] * ru - ends[0] * rl
                else:
                    along = (weighted * d[part, None]).sum(-1)
                    alpha = (torch.arange(samples, dtype=torch.float64, device=DEVICE) + 0.5) / samples
                    mean = integral / (upper[part] - lower[part])
                    linear = linear + rl * (along * (1.0 - alpha)).sum(1) + ru * (along * alpha).sum(1) \
                        + mean * (ru - rl)
                pose += torch.autograd.grad((seed[part] * length[part] * linear).sum(), leaf)[0]
    out = {"image": image.reshape(views, *shape)}
    if want_volume:
        out["volume"] = volume.reshape(grid.shape)
    if want_pose:
        out["pose"] = pose
    return out


def exact(case, seed):
    """``None`` for the Monte Carlo images and the fitted poses (ends of a
    random walk and of a search that stops early: neither is the value of a
    formula) and for calls of more than 3e9 samples."""
    if case["kind"] != "project":
        return None
    per = 2 * (case["nx"] + case["ny"] + case["nz"]) if case["integration"] == "cell_gauss" else case["samples"]
    if case["views"] * case["rows"] * case["cols"] * per > 3_000_000_000:
        return None
    grid, shape, target, window = _grid(case), (case["rows"], case["cols"]), _target(case, seed), _window(case)
    xi = torch.tensor(_tangent(seed), device=DEVICE, requires_grad=True)
    packed = _compose(xi)
    gauss = case["integration"] == "cell_gauss"
    if case["gather"]:
        got = _march(grid, _case_panels(case), shape, case["samples"], None, packed, want_volume=True,
                     cotangent=lambda v, _: (target[v] if window is None else target[v] * window[0]).reshape(-1))
        return {"volume": got["volume"]}
    field = _phantom(grid, seed)
    if case["storage"] != "float32":
        field = field.to(getattr(torch, case["storage"])).float()

    def residual(view, image):
        r = image.reshape(shape) - target[view]
        return (r if window is None else r * window[0]).reshape(-1)

    active = case["volume"] or case["pose"]
    got = _march(grid, _case_panels(case), shape, case["samples"], field, packed, gauss=gauss,
                 cotangent=residual if active else None, want_volume=case["volume"], want_pose=case["pose"])
    if case["pose"]:
        got["pose"] = torch.autograd.grad(packed, xi, got["pose"])[0]
    return got
