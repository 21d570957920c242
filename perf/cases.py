"""Performance cases: the work a user of the engine has it do, through its
public entry points, over the range of sizes it is used at.

``listed()`` gives the named cases, ``draw(rng)`` one more of the same ranges;
``prepare`` builds what a program holds before the call (volumes, poses, plans),
``run`` makes one pass, ``work`` counts what the path cannot do without and
``exact`` evaluates the same images and gradients in 64 bits with plain torch.

The kinds of case:

* ``view``: ``Projector.project`` of one pose, the drop-in call (a host image
  comes back, neglog applied): one CT, a CT with implants (several volumes with
  priorities) or a CT with a tool (a closed mesh that displaces tissue).
* ``plan``: a ``BatchPlan`` replayed, as a data generator does: many poses over
  one CT or over several CTs and detectors, images left on the device.
* ``set``: ``Projector.project_batch`` of a handful of poses with noise, images
  brought to the host.
* ``fit``: forward and backward of ``DifferentiableProjector`` under an MSE loss:
  density and pose, density alone (reconstruction), pose alone (registration).
* ``scatter``: Monte-Carlo photon histories into a CT.

The CTs are seeded synthetic bodies (skin, lungs, spine, rods and texture) of
the shapes a scanner gives; cameras look at them within 30 degrees of anterior
at 1020 mm from source to detector.
"""
from __future__ import annotations

import ctypes as C
import math
import os

import numpy as np
import torch

SDD = 1020.0
STEP = 0.1
AIR_DENSITY = 0.1129  # g/cm^3 per step of the air outside the volumes, as the projector defines it
FIVE = (("air", -900.0), ("lung", -200.0), ("soft tissue", 300.0), ("bone", 3000.0), ("titanium", math.inf))
THREE = (("air", -800.0), ("soft tissue", 350.0), ("bone", math.inf))


# ---- the cases ---------------------------------------------------------------------


def _view(name, shape, spacing, det, pixel, classes=5, march="fast", air=False, implants=0, tool=0):
    return dict(name=name, kind="view", nx=shape[0], ny=shape[1], nz=shape[2], sx=spacing[0], sy=spacing[1],
                sz=spacing[2], width=det[0], height=det[1], pixel=pixel, classes=classes, march=march, air=air,
                implants=implants, tool=tool)


def _fit(name, shape, views, det, pixel, density, pose):
    return dict(name=name, kind="fit", nx=shape[0], ny=shape[1], nz=shape[2], sx=1.0, sy=1.0, sz=1.0, views=views,
                width=det[0], height=det[1], pixel=pixel, density=density, pose=pose)


def listed():
    return [
        # one small CT onto a small detector: the smallest call, for previews and tests
        _view("view_128_256", (128, 128, 128), (1.0, 1.0, 1.0), (256, 256), 0.8, classes=3),
        # the clinical CT onto the C-arm's full detector
        _view("view_clinical_1536", (512, 512, 400), (0.8, 0.8, 1.0), (1536, 1536), 0.194),
        # the bit-exact march, the air outside the volume attenuating, odd sizes
        _view("view_exact_air", (201, 180, 151), (1.0, 1.1, 1.25), (389, 323), 0.75, march="exact", air=True),
        # a CT with two implants: three volumes with priorities
        _view("view_implants_768", (256, 256, 300), (1.0, 1.0, 1.0), (768, 768), 0.388, implants=2),
        # a CT with a tool in it (a mesh), ragged detector
        _view("view_tool_601x500", (256, 256, 300), (1.0, 1.0, 1.0), (601, 500), 0.5, tool=24),
        # training data: 16 poses of the clinical CT on the full detector
        dict(name="plan_clinical_16x1536", kind="plan", nx=512, ny=512, nz=400, sx=0.8, sy=0.8, sz=1.0, cts=1,
             views=16, width=1536, height=1536, pixel=0.194, mixed=False),
        # training data over CTs of uneven size and detectors of three sizes
        dict(name="plan_mixed_48", kind="plan", nx=256, ny=256, nz=300, sx=1.0, sy=1.0, sz=1.0, cts=3, views=48,
             width=765, height=768, pixel=0.388, mixed=True),
        # a few poses at once with photon noise
        dict(name="set_noise_8", kind="set", nx=256, ny=256, nz=300, sx=1.0, sy=1.0, sz=1.0, views=8, width=500,
             height=400, pixel=0.6),
        # reconstruction with pose refinement: 64 views
        _fit("fit_192_64x256", (192, 192, 192), 64, (256, 256), 1.6, True, True),
        # registration of a fixed CT: few views, the latency of an optimiser's step
        _fit("fit_pose_128_4", (128, 128, 128), 4, (200, 160), 1.2, False, True),
        # a small reconstruction, odd sizes
        _fit("fit_density_96_12", (96, 81, 75), 12, (144, 145), 1.3, True, False),
        # scatter of one clinical view
        dict(name="scatter_clinical", kind="scatter", nx=512, ny=512, nz=400, sx=0.8, sy=0.8, sz=1.0, width=256,
             height=256, pixel=1.164, histories=1 << 24),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: the kinds above with sizes spread over their ranges."""
    kind = rng.choice(["view", "view", "view", "plan", "set", "fit", "fit", "scatter"])
    nx, ny, nz = (_log(rng, 64, 320) for _ in range(3))
    sx, sy, sz = (round(rng.uniform(0.7, 1.4), 3) for _ in range(3))
    case = dict(kind=kind, nx=nx, ny=ny, nz=nz, sx=sx, sy=sy, sz=sz)
    extent = max(nx * sx, ny * sy, nz * sz)

    def detector(lo, hi):
        w, h = _log(rng, lo, hi), _log(rng, lo, hi)
        return dict(width=w, height=h, pixel=round(1.4 * extent / max(w, h), 4))

    if kind == "view":
        form = rng.choice(["ct", "ct", "implants", "tool"])
        case.update(detector(96, 1200 if form == "ct" else 600), classes=rng.choice([3, 5]),
                    march=rng.choice(["fast", "fast", "exact"]), air=rng.random() < 0.25,
                    implants=rng.choice([1, 2]) if form == "implants" else 0,
                    tool=_log(rng, 8, 48) if form == "tool" else 0)
    elif kind == "plan":
        case.update(detector(96, 700), cts=rng.choice([1, 2, 3]), views=_log(rng, 4, 48), mixed=rng.random() < 0.5)
    elif kind == "set":
        case.update(detector(96, 500), views=_log(rng, 1, 16))
    elif kind == "fit":
        density = rng.random() < 0.7
        case.update(detector(48, 256), views=_log(rng, 1, 32), density=density, pose=not density or rng.random() < 0.5)
    else:
        case.update(detector(96, 512), histories=_log(rng, 1 << 18, 1 << 23))
    return case


# ---- inputs ------------------------------------------------------------------------


def _hu(shape, seed):
    """A body of int16 HU values [i, j, k] on the GPU: the seed moves the organs
    a little and makes the texture."""
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    nx, ny, nz = shape
    x, y, z = (torch.arange(n, device="cuda", dtype=torch.float32) / n - 0.5 for n in shape)
    x, y, z = x[:, None, None], y[None, :, None], z[None, None, :]
    jig = rng.uniform(-0.01, 0.01, 12)

    def disc(cx, cy, rx, ry):
        return ((x - cx) / rx) ** 2 + ((y - cy) / ry) ** 2 <= 1.0

    hu = torch.randn(shape, generator=gen, device="cuda").mul_(30.0)
    body = disc(jig[0], jig[1], 0.42, 0.30)
    lungs = (disc(-0.17 + jig[2], -0.02 + jig[3], 0.11, 0.16) | disc(0.17 + jig[4], -0.02 + jig[5], 0.11, 0.16)) & (
        z.abs() < 0.35)
    spine = disc(jig[6], 0.18 + jig[7], 0.045, 0.045)
    rods = (disc(-0.03 + jig[8], 0.12, 0.008, 0.008) | disc(0.03 + jig[9], 0.12, 0.008, 0.008)) & (z.abs() < 0.2)
    ribs = ((((x - jig[0]) / 0.40) ** 2 + ((y - jig[1]) / 0.28) ** 2).sqrt() - 0.93).abs() < 0.02
    ribs = ribs & ((((z + 0.5) * nz / 24).floor() % 2) == 0)
    level = torch.full((nx, ny, 1), -1000.0, device="cuda").expand(shape).clone()
    level.masked_fill_(body.expand(shape), 40.0)
    level.masked_fill_(lungs, -800.0)
    level.masked_fill_(spine.expand(shape), 1100.0)
    level.masked_fill_(ribs & body, 900.0)
    level.masked_fill_(rods, 5900.0)
    hu.add_(level).masked_fill_(level == -1000.0, -1000.0)
    return hu.round_().clamp_(-1024, 8000).to(torch.int16)


def _density(hu):
    """Density of HU values: float32 of the two-line law evaluated in 64 bits."""
    h = hu.double()
    return torch.minimum(0.001029 * h + 1.030, 0.0005886 * h + 1.03).clamp_min_(0.0).float()


def _labels(hu, classes):
    """Index into ``classes`` of each voxel."""
    out = torch.full(hu.shape, len(classes) - 1, dtype=torch.uint8, device=hu.device)
    for i in range(len(classes) - 2, -1, -1):
        out.masked_fill_(hu <= classes[i][1], i)
    return out


def _pose(shape, spacing):
    """world_from_ijk of a CT with its centre at the world's origin."""
    m = np.eye(4)
    m[:3, :3] = [[spacing[0], 0, 0], [0, 0, spacing[2]], [0, -spacing[1], 0]]
    m[:3, 3] = -m[:3, :3] @ (np.array(shape, np.float64) / 2)
    return m


def _cameras(case, n, seed, axis_turn=False):
    """(R, source, width, height, pixel) of n cameras: R's rows are the camera's
    x, y and z axes in the world.  Within 30 degrees of anterior about a point
    near the centre, or (``axis_turn``) around the long axis."""
    rng = np.random.default_rng(seed + 17)
    extent = min(case["nx"] * case["sx"], case["ny"] * case["sy"], case["nz"] * case["sz"])
    out = []
    for k in range(n):
        if axis_turn:
            a = 2 * math.pi * k / n + rng.uniform(0, 0.05)
            z, point, frac = np.array([math.sin(a), math.cos(a), 0.0]), np.zeros(3), 0.5
        else:
            c, phi = rng.uniform(math.cos(math.radians(30.0)), 1.0), rng.uniform(0, 2 * math.pi)
            s = math.sqrt(1.0 - c * c)
            z = np.array([s * math.cos(phi), c, s * math.sin(phi)])
            point, frac = rng.uniform(-0.12, 0.12, 3) * extent, rng.uniform(0.5, 0.85)
        x = np.cross(z, [0.0, 0.0, 1.0])
        x /= np.linalg.norm(x)
        scale = (1, 2, 4)[k % 3] if case.get("mixed") else 1
        out.append((np.stack([x, np.cross(z, x), z]), point - frac * SDD * z, max(1, case["width"] // scale),
                    max(1, case["height"] // scale), case["pixel"] * scale))
    return out


def _projection(cam):
    from deepdrr_amd import geo

    R, src, w, h, pixel = cam
    return geo.CameraProjection(geo.CameraIntrinsicTransform.from_sizes((w, h), pixel, SDD),
                                geo.FrameTransform.from_rt(R, -R @ src))


def _blocks(case, seed):
    """Implants: (density [i, j, k], material, world_from_ijk) of uniform blocks
    with grids of their own, turned a little, around the body's middle."""
    rng = np.random.default_rng(seed + 5)
    extent = min(case["nx"] * case["sx"], case["ny"] * case["sy"], case["nz"] * case["sz"])
    out = []
    for k, (material, rho, n) in enumerate((("bone", 1.9, (41, 37, 30)), ("titanium", 4.5, (15, 60, 22)))[:case["implants"]]):
        size = extent * np.array([[0.18, 0.15, 0.12], [0.05, 0.25, 0.08]][k])
        spacing = size / np.array(n)
        a = rng.uniform(-0.3, 0.3)
        turn = np.array([[math.cos(a), -math.sin(a), 0], [math.sin(a), math.cos(a), 0], [0, 0, 1]])
        m = np.eye(4)
        m[:3, :3] = turn @ _pose(n, spacing)[:3, :3]
        m[:3, 3] = rng.uniform(-0.08, 0.08, 3) * extent - m[:3, :3] @ (np.array(n) / 2)
        out.append((np.full(n, rho, np.float32), material, m))
    return out


def _tool(case, seed):
    """A closed convex tool: a long ellipsoid of ``tool`` rings (world vertices,
    outward faces)."""
    rng = np.random.default_rng(seed + 9)
    extent = min(case["nx"] * case["sx"], case["ny"] * case["sy"], case["nz"] * case["sz"])
    rings, around = case["tool"], 2 * case["tool"]
    th = np.pi * np.arange(1, rings) / rings
    ph = 2 * np.pi * np.arange(around) / around
    ring = np.stack([np.outer(np.sin(th), np.cos(ph)), np.outer(np.sin(th), np.sin(ph)),
                     np.repeat(np.cos(th)[:, None], around, 1)], -1).reshape(-1, 3)
    v = np.concatenate([[[0, 0, 1.0]], ring, [[0, 0, -1.0]]])
    f = []
    at = lambda i, j: 1 + i * around + j % around  # noqa: E731
    for j in range(around):
        f.append((0, at(0, j), at(0, j + 1)))
        f.append((len(v) - 1, at(rings - 2, j + 1), at(rings - 2, j)))
        for i in range(rings - 2):
            f.append((at(i, j), at(i + 1, j), at(i + 1, j + 1)))
            f.append((at(i, j), at(i + 1, j + 1), at(i, j + 1)))
    d = rng.normal(size=3)
    d /= np.linalg.norm(d)
    e = np.cross(d, [0.0, 1.0, 0.2])
    e /= np.linalg.norm(e)
    axes = np.stack([e, np.cross(d, e), d], 1) * (extent * np.array([0.03, 0.03, 0.2]))
    return v @ axes.T + rng.uniform(-0.05, 0.05, 3) * extent, np.array(f)


def _shape(case):
    return (case["nx"], case["ny"], case["nz"]), (case["sx"], case["sy"], case["sz"])


def _cts(case, seed):
    """(shape, spacing, seed) of a plan's CTs: the case's own, then smaller ones."""
    shape, spacing = _shape(case)
    out = []
    for k in range(case.get("cts", 1)):
        n = tuple(max(16, s // (1, 2, 3)[k]) for s in shape)
        out.append((n, tuple(sp * s / m for sp, s, m in zip(spacing, shape, n)) if k else spacing, seed + 1000 * k))
    return out


def _target(case, cams, seed):
    """Measured images of a fit: a body of two ellipsoids seen by the cameras
    (kilo-electronvolts per photon), in closed form."""
    rng = np.random.default_rng(seed + 23)
    size = np.array([case["nx"] * case["sx"], case["nz"] * case["sz"], case["ny"] * case["sy"]])
    bodies = [(np.zeros(3), size * np.array([0.42, 0.5, 0.3]), 0.02),
              (rng.uniform(-0.1, 0.1, 3) * size, size * 0.08, 0.06)]
    out = []
    for R, src, w, h, pixel in cams:
        u = (torch.arange(w, device="cuda", dtype=torch.float64) + 0.5 - w / 2) * pixel
        v = (torch.arange(h, device="cuda", dtype=torch.float64) + 0.5 - h / 2) * pixel
        d = (u[None, :, None] * torch.tensor(R[0], device="cuda") + v[:, None, None] * torch.tensor(R[1], device="cuda")
             + SDD * torch.tensor(R[2], device="cuda"))
        d = d / d.norm(dim=-1, keepdim=True)
        path = torch.zeros((h, w), dtype=torch.float64, device="cuda")
        for c, semi, mu in bodies:
            inv = torch.tensor(1.0 / semi, device="cuda")
            o = torch.tensor((src - c) / semi, device="cuda")
            q = d * inv
            a, b = (q * q).sum(-1), (q * o).sum(-1)
            path += mu * 2.0 * (b * b - a * ((o * o).sum() - 1.0)).clamp_min(0.0).sqrt() / a
        out.append(55.0 * torch.exp(-path))
    return torch.stack(out).float()


# ---- what a program holds before the call --------------------------------------------


class _Engine:
    """An engine context with CTs ingested on the GPU, and what was built on it."""

    def __init__(self, cts):
        from deepdrr_amd import _abi
        from deepdrr_amd._abi_types import MARCH_FAST, Scene
        from deepdrr_amd.material import attenuation_table
        from deepdrr_amd.spectral_data import spectrum_tables, synthetic_120kv

        self.abi, self.plan, self.volumes = _abi, None, []
        self.materials = sorted(name for name, _ in FIVE)
        self.ctx = C.c_void_p()
        _abi.call("drr_ctx_create", 0, C.byref(self.ctx))
        scene = Scene(step=STEP, n_materials=len(self.materials), attenuate_outside=0, air_index=0, march=MARCH_FAST)
        _abi.call("drr_ctx_set_scene", self.ctx, C.byref(scene))
        energies, pdf = spectrum_tables(synthetic_120kv())
        mu = attenuation_table(self.materials, energies)
        _abi.call("drr_ctx_set_spectrum", self.ctx, len(energies), energies.ctypes.data, pdf.ctypes.data,
                  mu.ctypes.data)
        upper = np.array([1.0e9 if math.isinf(u) else u for _, u in FIVE], np.float32)
        label = np.array([self.materials.index(name) for name, _ in FIVE], np.uint8)
        for shape, _, seed in cts:
            hu = _hu(shape, seed).permute(2, 1, 0).contiguous()
            handle = C.c_void_p()
            _abi.call("drr_volume_create_from_hu", self.ctx, _abi.ptr(hu), *shape, 1, len(upper), upper.ctypes.data,
                      label.ctypes.data, C.byref(handle))
            self.volumes.append(handle)

    def __del__(self):
        if self.plan is not None:
            self.plan.close()
        for v in self.volumes:
            self.abi.lib().drr_volume_destroy(v)
        self.abi.lib().drr_ctx_destroy(self.ctx)


class _Fit:
    """A differentiable projector with its tensors."""

    def __init__(self, case, seed):
        from deepdrr_amd.autograd import DifferentiableProjector
        from deepdrr_amd.spectral_data import synthetic_120kv

        shape, spacing = _shape(case)
        hu = _hu(shape, seed)
        cams = _cameras(case, case["views"], seed, axis_turn=True)
        self.projections = [_projection(c) for c in cams]
        self.target = _target(case, cams, seed)
        self.density = _density(hu).requires_grad_(case["density"])
        self.theta = torch.zeros(6, device="cuda", requires_grad=case["pose"])
        self.projector = DifferentiableProjector(_labels(hu, THREE).cpu().numpy(), [name for name, _ in THREE],
                                                 _pose(shape, spacing), step=STEP, spectrum=synthetic_120kv())

    def __del__(self):
        if hasattr(self, "projector"):
            self.projector.close()


def _projector(case, seed, **options):
    """An initialised Projector over the case's CT, implants and tool."""
    from deepdrr_amd import Projector, Volume, geo
    from deepdrr_amd.mesh import DRRMaterial, Mesh, TriangleMesh
    from deepdrr_amd.spectral_data import synthetic_120kv

    shape, spacing = _shape(case)
    hu = _hu(shape, seed).cpu().numpy()
    if case.get("classes", 5) == 3:
        hu = hu.astype(np.float32)
    things = [Volume.from_hu(hu, origin=_pose(shape, spacing)[:3, 3], spacing=spacing,
                             anatomical_coordinate_system="LPS",
                             material_classes=THREE if case.get("classes", 5) == 3 else FIVE)]
    for rho, material, m in _blocks(case, seed) if case.get("implants") else []:
        things.append(Volume(rho, {material: np.ones(rho.shape, bool)}, anatomical_from_IJK=geo.FrameTransform(m)))
    if case.get("tool"):
        v, f = _tool(case, seed)
        steel = DRRMaterial("titanium", density=4.51, additive=True, subtractive=True, drrMatName="titanium")
        things.append(Mesh(mesh=TriangleMesh.from_arrays(v, f, steel)))
    cams = _cameras(case, case.get("views", 1), seed)
    intrinsics = _projection(cams[0]).intrinsic
    p = Projector(things, camera_intrinsics=intrinsics, source_to_detector_distance=SDD, step=STEP,
                  spectrum=synthetic_120kv(), march=case.get("march", "fast"),
                  attenuate_outside_volume=case.get("air", False), **options)
    p.initialize()
    return p, [_projection(c) for c in cams]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "view":
        return kind, _projector(case, seed)
    if kind == "set":
        p, projections = _projector(case, seed, add_noise=True, photon_count=20000)
        p.noise_seed = int(seed)
        return kind, (p, projections)
    if kind == "fit":
        return kind, _Fit(case, seed)
    from deepdrr_amd import mc
    from deepdrr_amd.batch import BatchPlan
    from deepdrr_amd.projector import build_view
    from deepdrr_amd.spectral_data import synthetic_120kv
    from deepdrr_amd.volume import VolumePose

    cts = _cts(case, seed)
    engine = _Engine(cts)
    if kind == "plan":
        poses = [VolumePose(_pose(shape, spacing), shape) for shape, spacing, _ in cts]
        which = [k % len(cts) for k in range(case["views"])]
        views = [build_view([poses[i]], [0], _projection(c), 4 * SDD)
                 for i, c in zip(which, _cameras(case, case["views"], seed))]
        engine.plan = BatchPlan(engine.ctx, engine.volumes, views, which, neglog=True)
        return kind, engine
    shape, spacing, _ = cts[0]
    params = mc.make_params(engine.materials, synthetic_120kv(), _projection(_cameras(case, 1, seed)[0]), SDD,
                            _pose(shape, spacing))
    return kind, (engine, params, case["histories"], int(seed))


def run(state):
    kind, s = state
    if kind == "view":
        p, projections = s
        return p.project(projections[0])
    if kind == "set":
        p, projections = s
        return p.project_batch(*projections)
    if kind == "plan":
        s.plan.launch()
        return {"images": s.plan.images, "intensity": s.plan.intensity, "photon_prob": s.plan.photon_prob}
    if kind == "fit":
        images = s.projector(s.density, s.theta, s.projections)
        loss = ((images - s.target) ** 2).mean()
        wanted = {k: t for k, t in (("density", s.density), ("pose", s.theta)) if t.requires_grad}
        grads = torch.autograd.grad(loss, list(wanted.values()))
        return {"images": images.detach(), "loss": loss.detach(), **dict(zip(wanted, grads))}
    from deepdrr_amd import mc

    engine, params, histories, seed = s
    m = mc.MonteCarlo(engine.ctx, engine.volumes[0], params)
    m.run(histories, seed=seed)
    return {"energy": m.img, "energy_squared": m.img2, "steps": m.steps}


# ---- what the path cannot do without ---------------------------------------------------


def _samples(case, cts, cams, which):
    """Samples inside the CTs, from 32 x 32 rays of each camera."""
    total = 0.0
    for cam, k in zip(cams, which):
        shape, spacing, _ = cts[k]
        R, src, w, h, pixel = cam
        u = (np.linspace(0, w, 33)[:-1] + w / 64 - w / 2) * pixel
        v = (np.linspace(0, h, 33)[:-1] + h / 64 - h / 2) * pixel
        d = u[None, :, None] * R[0] + v[:, None, None] * R[1] + SDD * R[2]
        d /= np.linalg.norm(d, axis=-1, keepdims=True)
        # the volume's axes i, j, k lie along world x, -z and y
        half = 0.5 * np.array([shape[0] * spacing[0], shape[2] * spacing[2], shape[1] * spacing[1]])
        with np.errstate(divide="ignore", invalid="ignore"):
            a0, a1 = (-half - src) / d, (half - src) / d
        near, far = np.minimum(a0, a1).max(-1), np.maximum(a0, a1).min(-1)
        total += np.maximum(0.0, far - np.maximum(near, 0.0)).mean() / STEP * w * h
    return total


def work(case):
    """One pass: each CT read once (float32 density and one byte of label a
    voxel), each output written once; about 24 operations a sample (position 6,
    trilinear filter 14, fractions and sums 4), three times that for a backward
    pass with it, and 200 a photon history."""
    kind = case["kind"]
    cts = _cts(case, 0)
    voxels = sum(s[0] * s[1] * s[2] for s, _, _ in cts)
    n = case.get("views", 1)
    cams = _cameras(case, n, 0, axis_turn=kind == "fit")
    pixels = sum(c[2] * c[3] for c in cams)
    if kind == "scatter":
        return {"bytes": 5.0 * voxels + 8.0 * 4 * pixels, "flops": 200.0 * case["histories"]}
    samples = _samples(case, cts, cams, [k % len(cts) for k in range(n)])
    if kind == "fit":
        gradient = 4.0 * voxels if case["density"] else 0.0
        return {"bytes": 5.0 * voxels + gradient + 8.0 * pixels, "flops": 72.0 * samples}
    return {"bytes": 5.0 * voxels + {"plan": 12.0, "set": 4.0, "view": 4.0}[kind] * pixels, "flops": 24.0 * samples}


# ---- the same in 64 bits ------------------------------------------------------------
#
# The sample lattice (ray directions, slab interval, number of steps and the
# float32 sequence alpha += step) is part of what the projector computes, so it
# is followed in float32; every quantity along it is evaluated in 64 bits.


def _tables(materials):
    """Energies (keV), spectrum and mass attenuation [bins, materials]."""
    import deepdrr_amd

    e = 20.0 + 5.0 * np.arange(20, dtype=np.float64)
    w = e * (120.0 - e) ** 2 * np.exp(-e / 40.0)
    folder = os.path.join(os.path.dirname(deepdrr_amd.__file__), "data", "materials")
    files = {"soft tissue": "tissue_soft", "titanium": "22_Ti_Titanium"}
    mu = []
    for name in materials:
        rows = []
        for line in open(os.path.join(folder, files.get(name, name))):
            if line.strip() and not line.startswith(("_", "Energy")):
                rows.append([float(x) for x in line.split()])
        x, y = np.array(rows)[:, 0], np.array(rows)[:, 1]
        for j in range(1, len(x)):  # an absorption edge repeats its energy
            if x[j] == x[j - 1]:
                x[j - 1] *= 1 - 1e-9
        mu.append(10.0 ** np.interp(np.log10(e / 1000.0), np.log10(x), np.log10(y)))
    dev = dict(device="cuda", dtype=torch.float64)
    return torch.tensor(e, **dev), torch.tensor(w / w.sum(), **dev), torch.tensor(np.stack(mu, 1), **dev)


class _Grid:
    """A volume on the GPU: density, labels (of the scene's materials) and pose."""

    def __init__(self, density, labels, world_from_ijk, priority):
        self.n = density.shape
        self.density = density.permute(2, 1, 0).contiguous().reshape(-1)
        self.labels = labels.permute(2, 1, 0).contiguous().reshape(-1)
        self.ijk_from_world = np.linalg.inv(world_from_ijk)
        self.priority = priority


class _Rays:
    """All rays of some cameras against some grids, on the float32 lattice."""

    def __init__(self, cams, grids, max_ray_length, keep=None):
        rx, ry, rz, src, length = [], [], [], [], []
        for R, s, w, h, pixel in cams:
            k = np.array([[SDD / pixel, 0, w / 2], [0, SDD / pixel, h / 2], [0, 0, 1.0]])
            W = torch.tensor((R.T @ np.linalg.inv(k)).astype(np.float32), device="cuda")
            u = (torch.arange(w, device="cuda", dtype=torch.float32) + 0.5)[None, :].expand(h, w).reshape(-1)
            v = (torch.arange(h, device="cuda", dtype=torch.float32) + 0.5)[:, None].expand(h, w).reshape(-1)
            d = [(u * W[a, 0] + v * W[a, 1]) + W[a, 2] for a in range(3)]
            L = ((d[0] * d[0] + d[1] * d[1]) + d[2] * d[2]).sqrt()
            inv = 1.0 / L
            rx.append(d[0] * inv)
            ry.append(d[1] * inv)
            rz.append(d[2] * inv)
            length.append(L)
            src.append(torch.tensor(s, device="cuda").expand(w * h, 3))
        self.r = torch.stack([torch.cat(rx), torch.cat(ry), torch.cat(rz)])  # [3, rays] float32
        self.length = torch.cat(length)
        self.source = torch.cat(src).t().contiguous()  # [3, rays] float64
        self.step = torch.tensor(STEP, dtype=torch.float32, device="cuda")
        self.grids, self.local = grids, []
        n = self.length.numel()
        lo_all, hi_all = self.length.clone(), torch.zeros(n, device="cuda")
        for g in grids:
            A = torch.tensor(g.ijk_from_world.astype(np.float32), device="cuda")
            ri = torch.stack([(A[a, 0] * self.r[0] + A[a, 1] * self.r[1]) + A[a, 2] * self.r[2] for a in range(3)])
            M = torch.tensor(g.ijk_from_world, device="cuda")
            s = (M[:3, :3] @ self.source + M[:3, 3:]).float()
            lo = torch.zeros(n, device="cuda")
            hi = torch.full((n,), max_ray_length if max_ray_length > 0 else math.inf, device="cuda")
            ok = torch.ones(n, dtype=torch.bool, device="cuda")
            for a in range(3):
                moving = ri[a] != 0
                rec = 1.0 / torch.where(moving, ri[a], torch.ones_like(ri[a]))
                a0, a1 = (-0.5 - s[a]) * rec, (g.n[a] - 0.5 - s[a]) * rec
                lo = torch.where(moving, torch.maximum(lo, torch.minimum(a0, a1)), lo)
                hi = torch.where(moving, torch.minimum(hi, torch.maximum(a0, a1)), hi)
                ok &= moving | ((s[a] >= -0.5) & (s[a] <= g.n[a] - 0.5))
            self.local.append((s.double(), ri.double(), lo, hi, ok))
            lo_all = torch.where(ok, torch.minimum(lo_all, lo), lo_all)
            hi_all = torch.where(ok, torch.maximum(hi_all, hi), hi_all)
        self.lo, self.hi = lo_all, hi_all
        self.count = ((hi_all - lo_all) / self.step).ceil().clamp_min(0.0).long()

    def steps(self):
        """(alpha, t < count, weight of an end sample) of the steps at which some
        ray is near a grid, and the number of steps left out before them."""
        alpha = self.lo.clone()
        most = int(self.count.max())
        near = torch.full_like(self.lo, math.inf)
        far = torch.full_like(self.lo, -math.inf)
        for _, _, lo, hi, ok in self.local:
            near = torch.where(ok & (hi >= lo), torch.minimum(near, lo), near)
            far = torch.where(ok & (hi >= lo), torch.maximum(far, hi), far)
        margin = 4.0  # mm: more than a voxel, so that a cell is entered before the grid is
        t = 0
        while t < most:
            k = min(32, most - t)
            inside = (alpha + 1.01 * k * STEP + margin >= near) & (alpha <= far + margin) & (t < self.count)
            if not bool(inside.any()):
                for _ in range(k):
                    alpha = alpha + self.step
                t += k
                continue
            for _ in range(k):
                end = torch.where((t == 0) | (self.count - 1 == t), 0.5, 1.0)
                yield alpha, t < self.count, end
                alpha = alpha + self.step
                t += 1

    def cell(self, g, alpha):
        """Of grid g at alpha: base [3, rays], weights [8, rays], their x, y and z
        factors, and the corners' voxels."""
        s, ri = self.local[g][:2]
        n = self.grids[g].n
        p = s + alpha.double() * ri - 1.0
        b = p.floor()
        f = p - b
        e = torch.stack([1.0 - f, f])  # [2, 3, rays]
        wx, wy, wz = e[:, 0], e[:, 1], e[:, 2]
        w = (wz[:, None, None] * wy[None, :, None] * wx[None, None, :]).reshape(8, -1)
        i = b.long()
        at = [torch.stack([i[a].clamp(0, n[a] - 1), (i[a] + 1).clamp(0, n[a] - 1)]) for a in range(3)]
        v = ((at[2][:, None, None] * n[1] + at[1][None, :, None]) * n[0] + at[0][None, None, :]).reshape(8, -1)
        return b, w, (wx, wy, wz), v


def _area_densities(rays, n_materials, air=None, hidden=None):
    """Area densities [materials, rays] in g/cm^2 before any mesh's."""
    n = rays.length.numel()
    ad = torch.zeros((n_materials, n), dtype=torch.float64, device="cuda")
    sampled = torch.zeros(n, dtype=torch.int64, device="cuda")
    several = len(rays.grids) > 1
    labels = torch.zeros((8, n), dtype=torch.int64, device="cuda")
    base = torch.full((3, n), math.inf, dtype=torch.float64, device="cuda")
    for alpha, live, end in rays.steps():
        cells, best = [], torch.full((n,), 1 << 20, device="cuda")
        for g, grid in enumerate(rays.grids):
            b, w, _, v = rays.cell(g, alpha)
            own = grid.labels[v].long()
            if several:  # a cell's labels are read again only where its base is another one than the last
                same = (b == base).all(0)
                labels = torch.where(same, labels, own)
                base = b
                own = labels
            lo, hi, ok = rays.local[g][2:]
            inside = live & ok & (alpha >= lo) & (alpha <= hi)
            cells.append((inside, w, v, own))
            best = torch.where(inside, best.clamp_max(grid.priority), best)
        count = sum((c[0] & (best == g.priority)).long() for c, g in zip(cells, rays.grids))
        shown = count > 0
        sampled += shown.long()
        if hidden is not None:
            blocked = (alpha > hidden[0]) & (alpha <= hidden[1])
            sampled += (blocked & live & ~shown).long()
            shown = shown & ~blocked
        for (inside, w, v, own), grid in zip(cells, rays.grids):
            rho = (w * grid.density[v].double()).sum(0)
            # every grid of the chosen priority that the ray meets counts, as the projector has it
            use = shown & (best == grid.priority) & rays.local[rays.grids.index(grid)][4]
            share = torch.where(use, rho * end / count.clamp_min(1), torch.zeros_like(rho))
            ad.scatter_add_(0, own, share * w)
    if air is not None:
        missed = rays.count - sampled
        ad[air] += AIR_DENSITY * ((rays.lo.double() + rays.length.double() - rays.hi.double()) / STEP + missed)
    return ad * float(np.float32(STEP)) / 10.0


def _intensity(ad, tables):
    e, pdf, mu = tables
    out = torch.zeros_like(ad[0])
    for b in range(len(e)):
        out += e[b] * pdf[b] * torch.exp(-(mu[b][:, None] * ad).sum(0))
    return out


def _neglog(x):
    x = x + (x.amin((-2, -1), keepdim=True) + 0.01)
    y = -x.log()
    lo, hi = y.amin((-2, -1), keepdim=True), y.amax((-2, -1), keepdim=True)
    return (y - lo) / (hi - lo)


def _chord(rays, vertices, faces):
    """(entry, exit) of each ray through a closed convex mesh (inf, inf where it
    misses)."""
    v = torch.tensor(vertices.astype(np.float32), device="cuda").double()
    lo = torch.full((rays.length.numel(),), math.inf, dtype=torch.float64, device="cuda")
    hi = torch.full_like(lo, -math.inf)
    d, o = rays.r.double(), rays.source.float().double()
    for f in faces:
        v0, e1, e2 = v[f[0]], v[f[1]] - v[f[0]], v[f[2]] - v[f[0]]
        p = torch.linalg.cross(d, e2[:, None].expand_as(d), dim=0)
        det = (e1[:, None] * p).sum(0)
        tv = o - v0[:, None]
        u = (tv * p).sum(0) / det
        q = torch.linalg.cross(tv, e1[:, None].expand_as(tv), dim=0)
        w = (d * q).sum(0) / det
        t = (e2[:, None] * q).sum(0) / det
        hit = (u >= 0) & (w >= 0) & (u + w <= 1) & (t > 0) & (det != 0)
        lo = torch.where(hit, torch.minimum(lo, t), lo)
        hi = torch.where(hit, torch.maximum(hi, t), hi)
    lo = torch.where(hi > lo, lo, torch.full_like(lo, math.inf))
    return lo, torch.where(torch.isinf(lo), lo, hi)


def _ct_grid(hu, classes, materials, world_from_ijk, priority=0):
    remap = torch.tensor([materials.index(name) for name, _ in classes], dtype=torch.uint8, device="cuda")
    return _Grid(_density(hu), remap[_labels(hu, classes).long()], world_from_ijk, priority)


def _exact_view(case, seed):
    shape, spacing = _shape(case)
    classes = THREE if case["classes"] == 3 else FIVE
    blocks = _blocks(case, seed) if case["implants"] else []
    materials = sorted({name for name, _ in classes} | {m for _, m, _ in blocks} | ({"titanium"} if case["tool"] else set())
                       | ({"air"} if case["air"] else set()))
    grids = [_ct_grid(_hu(shape, seed), classes, materials, _pose(shape, spacing), len(blocks))]
    for k, (rho, material, m) in enumerate(blocks):
        d = torch.tensor(rho, device="cuda")
        grids.append(_Grid(d, torch.full_like(d, materials.index(material), dtype=torch.uint8), m, len(blocks) - 1 - k))
    cam = _cameras(case, 1, seed)[0]
    rays = _Rays([cam], grids, 4 * SDD)
    chord = _chord(rays, *_tool(case, seed)) if case["tool"] else None
    ad = _area_densities(rays, len(materials), materials.index("air") if case["air"] else None, chord)
    if chord is not None:
        length = torch.where(torch.isinf(chord[0]), torch.zeros_like(chord[0]), chord[1] - chord[0])
        ad[materials.index("titanium")] += 4.51 * length / 10.0
    return _neglog(_intensity(ad, _tables(materials)).reshape(cam[3], cam[2]))


def _exact_plan(case, seed):
    materials = sorted(name for name, _ in FIVE)
    tables = _tables(materials)
    cts = _cts(case, seed)
    grids = [_ct_grid(_hu(shape, s), FIVE, materials, _pose(shape, spacing)) for shape, spacing, s in cts]
    images, intensity, prob = [], [], []
    for k, cam in enumerate(_cameras(case, case["views"], seed)):
        ad = _area_densities(_Rays([cam], [grids[k % len(cts)]], 4 * SDD), len(materials))
        i = _intensity(ad, tables)
        images.append(_neglog(i.reshape(cam[3], cam[2])).reshape(-1))
        intensity.append(i)
        prob.append(_intensity(ad, (torch.ones_like(tables[0]), *tables[1:])))
    return {"images": torch.cat(images), "intensity": torch.cat(intensity), "photon_prob": torch.cat(prob)}


def _exact_fit(case, seed):
    shape, spacing = _shape(case)
    names = [name for name, _ in THREE]
    grid = _ct_grid(_hu(shape, seed), THREE, names, _pose(shape, spacing))
    cams = _cameras(case, case["views"], seed, axis_turn=True)
    rays = _Rays(cams, [grid], -1.0)
    e, pdf, mu = _tables(names)
    ad = _area_densities(rays, len(names))
    images = _intensity(ad, (e, pdf, mu))
    off = images - _target(case, cams, seed).double().reshape(-1)
    out = {"images": images.reshape(len(cams), case["height"], case["width"]), "loss": (off ** 2).mean()}
    slope = torch.zeros_like(ad)  # dL/d(area density before the step's scale)
    for b in range(len(e)):
        slope -= mu[b][:, None] * (e[b] * pdf[b] * torch.exp(-(mu[b][:, None] * ad).sum(0)))
    slope *= 2.0 * off / off.numel() * float(np.float32(STEP)) / 10.0
    density = torch.zeros(grid.density.numel(), dtype=torch.float64, device="cuda")
    shift = torch.zeros(3, dtype=torch.float64, device="cuda")
    turn = torch.zeros(3, dtype=torch.float64, device="cuda")
    A = torch.tensor(grid.ijk_from_world[:3, :3], device="cuda")
    _, _, lo, hi, ok = rays.local[0]
    sign = torch.tensor([-1.0, 1.0], dtype=torch.float64, device="cuda")[:, None]
    for alpha, live, end in rays.steps():
        _, w, (wx, wy, wz), v = rays.cell(0, alpha)
        use = torch.where(live & ok & (alpha >= lo) & (alpha <= hi), end, 0.0).double()
        h = slope.gather(0, grid.labels[v].long())
        g = (w * h).sum(0) * use
        if case["density"]:
            density.scatter_add_(0, v.reshape(-1), (g * w).reshape(-1))
        if case["pose"]:
            d = grid.density[v].double()
            rho = (w * d).sum(0) * use
            both = (g * d + rho * h).reshape(2, 2, 2, -1)
            one = torch.ones_like(wx) * sign
            dp = torch.stack([(both * (wz[:, None, None] * wy[None, :, None] * one[None, None, :])).sum((0, 1, 2)),
                              (both * (wz[:, None, None] * one[None, :, None] * wx[None, None, :])).sum((0, 1, 2)),
                              (both * (one[:, None, None] * wy[None, :, None] * wx[None, None, :])).sum((0, 1, 2))])
            dw = A.t() @ dp
            x = rays.source + alpha.double() * rays.r.double()  # the pose turns about the world's origin
            shift -= dw.sum(1)
            turn += torch.linalg.cross(dw, x, dim=0).sum(1)
    if case["density"]:
        out["density"] = density.reshape(shape[2], shape[1], shape[0]).permute(2, 1, 0)
    if case["pose"]:
        out["pose"] = torch.cat([shift, turn])
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("scatter", "set"):
        return None  # random draws: no value of their own in 64 bits
    pixels = sum(c[2] * c[3] for c in _cameras(case, case.get("views", 1), 0))
    length = math.sqrt((case["nx"] * case["sx"]) ** 2 + (case["ny"] * case["sy"]) ** 2 + (case["nz"] * case["sz"]) ** 2)
    cost = pixels * length / STEP * (3.0 if kind == "fit" else 1.0 + case.get("implants", 0))
    if cost > 2.0e10:
        return None
    return {"view": _exact_view, "plan": _exact_plan, "fit": _exact_fit}[kind](case, seed)
