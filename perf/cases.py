"""The projector's measured cases: what a user has it do, through its public
entry points, over the sizes, storage types and options it is used with.

Four kinds of pass:
  forward  Projector.forward over a range of views of a resident phantom
  step     one gradient step of the differentiable projector (autograd.project,
           weighted least squares on log projections, backward)
  host     the whole drop-in call on host data: a label volume uploaded, every
           view projected, the projections back in host memory
  batch    several uneven scans through Batch.run

Phantoms are seeded ellipsoid bodies made on the GPU (water with inserts of
the other materials), scanners are the circular cone beam at SOD 1000 mm and
SDD 1500 mm, spectra and attenuation are the package's synthetic tables.
`exact` evaluates the same method (zero-padded trilinear samples every dx
along each ray, Beer-Lambert per energy bin) with plain torch in FP64.
"""
import math
import random

import numpy as np
import torch

import ct_forward_projection_amd as P
from ct_forward_projection_amd import autograd as A
from ct_forward_projection_amd import synthetic as S

DEVICE = torch.device("cuda", 0)
MATERIALS = (S.WATER, S.BONE, S.IODINE, S.ALUMINIUM, S.CAESIUM, S.IODINE)
# densities (g/cm^3) of the inserts of each material
INSERT = ((0.2, 0.9), (1.2, 1.9), (0.002, 0.020), (0.3, 1.0), (0.002, 0.010), (0.005, 0.030))
DTYPES = {"f32": P.CTFP_F32, "f16": P.CTFP_F16, "bf16": P.CTFP_BF16}
GRID = dict(strip_width=36, interspace_width=214, height_mm=2.14, focal_mm=1500.0, strip_density=11.35)

DEFAULTS = dict(kind="forward", nx=128, ny=128, nz=128, px=1.0, py=1.0, pz=1.0, nu=256, nv=256, pitch=0.8,
                views=90, first=0, count=90, mats=1, dtype="f32", kvp=120.0, grid=True, jitter=0.0, focal=0.0,
                rot=1, weighting=False, keep=True, items=0, largest=0)


def _case(**kw):
    return dict(DEFAULTS, **kw)


def listed():
    return [
        # one view of a small single-material scan (the interactive call: one
        # angle at a time), where launches and latency count
        _case(name="view_128", kvp=80.0, grid=False, weighting=True, first=11, count=1),
        # the whole small scan: 128^3, one material, 90 views, FP32
        _case(name="scan_128", kvp=80.0, grid=False, weighting=True),
        # a subset of views of the 3 x 512^3 scan in FP32 (one subset of an
        # ordered-subsets reconstruction)
        _case(name="subset_512_f32", nx=512, ny=512, nz=512, px=0.5, py=0.5, pz=0.5, nu=1024, nv=768, pitch=0.4,
              views=360, first=40, count=12, mats=3),
        # the headline scan: 3 x 512^3 in FP16, every one of its 360 views
        _case(name="scan_512_f16", nx=512, ny=512, nz=512, px=0.5, py=0.5, pz=0.5, nu=1024, nv=768, pitch=0.4,
              views=360, count=360, mats=3, dtype="f16"),
        # two materials in BF16, a scintillator that varies from pixel to
        # pixel (a weight per bin and pixel), no grid
        _case(name="jitter_320_bf16", nx=320, ny=320, nz=320, px=0.6, py=0.6, pz=0.6, nu=640, nv=480, pitch=0.6,
              views=120, count=48, mats=2, dtype="bf16", kvp=100.0, grid=False, jitter=0.05),
        # odd extents, unequal voxel sides, a detector of odd size, the other
        # sense of rotation and a focal spot drawn per view, FP16
        _case(name="odd_focal_f16", nx=201, ny=167, nz=119, px=0.9, py=1.1, pz=1.3, nu=333, nv=217, pitch=0.9,
              views=37, count=37, mats=3, dtype="f16", kvp=110.0, focal=0.4, rot=-1),
        # six materials: two groups of channels, then a spectrum pass
        _case(name="six_materials", nx=160, ny=160, nz=160, px=1.0, py=1.0, pz=1.0, nu=320, nv=240, pitch=1.1,
              views=60, count=45, mats=6),
        # one gradient step on a small subset (a few views at a time)
        _case(name="step_97", kind="step", nx=97, ny=97, nz=80, px=1.5, py=1.5, pz=1.5, nu=161, nv=128, pitch=2.0,
              views=72, first=24, count=12, mats=2),
        # a gradient step that marches again instead of keeping the line
        # integrals, densities stored in FP16
        _case(name="step_160_remarch", kind="step", nx=160, ny=160, nz=128, px=1.25, py=1.25, pz=1.25, nu=256,
              nv=192, pitch=1.6, views=120, count=40, mats=3, dtype="f16", keep=False),
        # the full differentiable workload: 3 x 256^3, 512 x 512, 180 views
        _case(name="step_256", kind="step", nx=256, ny=256, nz=256, nu=512, nv=512, views=180, count=180, mats=3),
        # the drop-in call on host data: labels in, projections out
        _case(name="host_192", kind="host", nx=192, ny=192, nz=192, nu=384, nv=288, pitch=1.1, views=60, count=60,
              mats=3),
        # five uneven scans in one graph-captured launch, FP16
        _case(name="batch_5", kind="batch", items=5, largest=256, dtype="f16", first=2024),
    ]


def _samples(case):
    """Lattice samples of the rays inside the phantom's bounding box."""
    if case["kind"] == "batch":
        return sum(_samples(c) for c in _batch_cases(case))
    s = _scalars(case)
    u = (np.arange(16) + 0.5) / 16 * case["nu"] - 0.5
    v = (np.arange(16) + 0.5) / 16 * case["nv"] - 0.5
    vv, uu = np.meshgrid(v, u, indexing="ij")
    total = 0.0
    for view in np.linspace(0, case["count"] - 1, 12).astype(int):
        src, d = _rays(case, s, torch.from_numpy(uu.reshape(-1)), torch.from_numpy(vv.reshape(-1)),
                       case["first"] + int(view), None)
        lo, hi = np.full(256, s["t0"]), np.full(256, s["t0"] + (s["K"] - 1) * s["dx"])
        for a, n in enumerate((case["nx"], case["ny"], case["nz"])):
            da = d[a].numpy()
            da = np.where(np.abs(da) < 1e-12, 1e-12, da)
            k1, k2 = (-1 - src[a]) / da, (n - src[a]) / da
            lo, hi = np.maximum(lo, np.minimum(k1, k2)), np.minimum(hi, np.maximum(k1, k2))
        total += float(np.maximum(hi - lo, 0).mean()) / s["dx"]
    return total / 12 * case["count"] * case["nu"] * case["nv"]


def draw(rng):
    """One more case of the listed ranges: phantoms of 64 to 512 voxels a
    side, detectors of 96 to 1024 columns, one view to a whole scan."""
    while True:
        kind = rng.choice(["forward"] * 5 + ["step"] * 3 + ["host", "batch"])
        if kind == "batch":
            return _case(kind="batch", items=rng.randint(2, 8), largest=rng.choice([160, 192, 256, 320]),
                         dtype=rng.choice(["f32", "f16", "f16", "bf16"]), first=rng.randrange(1 << 20))
        top = {"forward": 512, "step": 256, "host": 256}[kind]
        size = lambda lo, hi: int(round(lo * (hi / lo) ** rng.random()))
        n = size(64, top)
        c = _case(kind=kind, nx=n, ny=n, nz=n)
        if rng.random() < 0.6:
            c["ny"], c["nz"] = max(33, int(n * rng.uniform(0.6, 1.0))), max(33, int(n * rng.uniform(0.4, 1.0)))
        c["px"] = round(256.0 / n * rng.uniform(0.7, 1.0), 3)
        c["py"] = c["px"] if rng.random() < 0.7 else round(c["px"] * rng.uniform(0.8, 1.3), 3)
        c["pz"] = c["px"] if rng.random() < 0.7 else round(c["px"] * rng.uniform(0.8, 1.5), 3)
        c["nu"] = size(96, 1024 if kind == "forward" else 512)
        c["nv"] = max(64, int(c["nu"] * rng.uniform(0.5, 1.0)))
        span = math.hypot(c["nx"] * c["px"], c["ny"] * c["py"])
        c["pitch"] = round(1.5 * span / c["nu"] * rng.uniform(0.8, 1.05), 3)
        c["views"] = size(24, 360)
        c["count"] = c["views"] if kind == "host" else size(1, c["views"])
        c["first"] = 0 if kind == "host" else rng.randint(0, c["views"] - c["count"])
        c["mats"] = rng.choice([1, 2, 3, 3, 3, 4, 6] if kind == "forward" else [1, 2, 3, 3])
        c["dtype"] = rng.choice(["f32", "f16", "bf16"] if kind == "forward" else ["f32", "f32", "f16"])
        c["kvp"] = float(rng.choice([80, 90, 100, 110, 120, 130, 140]))
        c["grid"] = rng.random() < 0.6
        c["jitter"] = 0.05 if rng.random() < 0.25 and c["nu"] * c["nv"] <= 320 * 240 else 0.0
        c["focal"] = 0.4 if rng.random() < 0.25 else 0.0
        c["rot"] = rng.choice([1, 1, -1])
        c["keep"] = rng.random() < 0.7
        most = {"forward": 2.0e11, "step": 1.4e10, "host": 1.5e10}[kind]
        if _samples(c) * (1 if c["mats"] <= 4 else 3) <= most and c["count"] * c["nu"] * c["nv"] <= 3e8:
            return c


# ------------------------------------------------------------------ inputs

def _batch_cases(case):
    """The scans of a batch: uneven phantoms, detectors, views and spectra."""
    rng = random.Random(case["first"])
    sizes = [n for n in (96, 128, 160, 192, 256, 320) if n <= case["largest"]]
    out = []
    for _ in range(case["items"]):
        n = rng.choice(sizes)
        nu, nv = rng.choice([(192, 192), (256, 192), (384, 288), (333, 251)])
        views = rng.randint(24, 90)
        out.append(_case(nx=n, ny=n, nz=n, px=0.5, py=0.5, pz=0.5, nu=nu, nv=nv,
                         pitch=round(n * 0.5 * 1.45 * 1.5 / min(nu, nv), 4), views=views, count=views,
                         mats=rng.randint(1, 3), dtype=case["dtype"], kvp=float(rng.choice([80, 100, 120, 140])),
                         grid=rng.random() < 0.5))
    return out


def _setup(case):
    s = S.config2()
    s.n_vox = (case["nx"], case["ny"], case["nz"])
    s.length_mm = (case["nx"] * case["px"], case["ny"] * case["py"], case["nz"] * case["pz"])
    s.det, s.d_size, s.views, s.rot = (case["nu"], case["nv"]), case["pitch"], case["views"], case["rot"]
    s.kvp, s.materials = case["kvp"], MATERIALS[:case["mats"]]
    s.grid = dict(GRID) if case["grid"] else None
    s.scint_thickness_err, s.energy_weighting = case["jitter"], case["weighting"]
    return s


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _inserts(case, seed):
    """Ellipsoids (material, centre, semi-axes, rotation, density): an elliptic
    water cylinder first, then six to eight inserts of every material."""
    rng = np.random.default_rng([seed, case["nx"], case["nz"], case["mats"]])
    n = np.array([case["nz"], case["ny"], case["nx"]], dtype=np.float64)
    out = []
    for m in range(case["mats"]):
        lo, hi = (0.05, 0.12) if m != 2 else (0.03, 0.07)
        for _ in range(int(rng.integers(6, 9))):
            q = rng.normal(size=(3, 3))
            rot = np.linalg.qr(q)[0]
            centre = n / 2 - 0.5 + rng.uniform(-0.25, 0.25, 3) * n
            out.append((m, centre, rng.uniform(lo, hi, 3) * n.min(), rot, rng.uniform(*INSERT[m])))
    return rng.uniform(0.95, 1.05), out


def _volumes(case, seed, noise=0.0):
    """Density channels [mats][nz][ny][nx] (g/cm^3) on the GPU."""
    water, inserts = _inserts(case, seed)
    nz, ny, nx = case["nz"], case["ny"], case["nx"]
    vol = torch.zeros((case["mats"], nz, ny, nx), dtype=torch.float32, device=DEVICE)
    y = (torch.arange(ny, device=DEVICE) - (ny - 1) / 2)[:, None] / (0.35 * ny)
    x = (torch.arange(nx, device=DEVICE) - (nx - 1) / 2)[None, :] / (0.45 * nx)
    z0, z1 = int(round(0.07 * nz)), int(round(0.93 * nz))
    vol[0, z0:z1] = (y * y + x * x <= 1).float() * water
    for m, centre, semi, rot, rho in inserts:
        lo = [max(0, int(c - semi.max() - 1)) for c in centre]
        hi = [min(s, int(c + semi.max() + 2)) for c, s in zip(centre, (nz, ny, nx))]
        if any(a >= b for a, b in zip(lo, hi)):
            continue
        p = torch.meshgrid(*[torch.arange(a, b, device=DEVICE, dtype=torch.float32) - float(c)
                             for a, b, c in zip(lo, hi, centre)], indexing="ij")
        q = sum((sum(float(rot[i, j]) * p[i] for i in range(3)) / float(semi[j])) ** 2 for j in range(3))
        box = vol[:, lo[0]:hi[0], lo[1]:hi[1], lo[2]:hi[2]]
        keep = (q > 1).float()
        if INSERT[m][1] > 0.1:      # dense inserts displace what was there
            box *= keep
        box[m] += (1 - keep) * rho
    if noise:
        vol *= 1 - noise + 2 * noise * torch.rand(vol.shape, device=DEVICE, generator=_generator(seed + 17))
    return vol


def _labels(case, seed):
    """uint8 label volume [nz][ny][nx] (host) and the density of each label."""
    vol = _volumes(case, seed)
    lab = (vol[0] > 0).to(torch.uint8)
    for m in range(1, case["mats"]):
        lab[vol[m] > 0] = m + 1
    return lab.cpu().numpy(), [m.density for m in MATERIALS[:case["mats"]]]


def _focal(case):
    return P.focal_spot_offsets(case["views"], case["focal"]) if case["focal"] else None


def _spectral(case):
    s = _setup(case)
    return P.spectral_inputs(s, *s.det)


def _projector(case, volumes=None, kw=None):
    s = _setup(case)
    proj = P.Projector(P.scan_params(**s.scan_kwargs()), device=0)
    if volumes is not None:
        proj.set_volumes(list(volumes), storage_dtype=DTYPES[case["dtype"]])
    proj.set_spectral(**(kw or _spectral(case)))
    if case["focal"]:
        proj.set_focal_spot(_focal(case))
    return proj


def _measured(case, seed):
    """A measured scan to fit: counts and log projections [count][nv][nu] of a
    water ellipsoid in place of the phantom, with counting noise (FP64)."""
    s = _scalars(case)
    g = _generator(seed + 29)
    semi = (0.45 * case["nx"] * case["px"], 0.35 * case["ny"] * case["py"], 0.45 * case["nz"] * case["pz"])
    u = torch.arange(case["nu"], device=DEVICE, dtype=torch.float64).repeat(case["nv"])
    v = torch.arange(case["nv"], device=DEVICE, dtype=torch.float64).repeat_interleave(case["nu"])
    scale = (case["px"], case["py"], case["pz"])
    half = (case["nx"], case["ny"], case["nz"])
    p = torch.empty((case["count"], case["nv"], case["nu"]), dtype=torch.float64, device=DEVICE)
    for i in range(case["count"]):
        src, d = _rays(case, s, u, v, case["first"] + i, None)
        o = [(src[a] - half[a] / 2) * scale[a] / semi[a] for a in range(3)]
        e = [d[a] * scale[a] / semi[a] for a in range(3)]
        aa = sum(x * x for x in e)
        bb = sum(x * y for x, y in zip(o, e))
        cc = sum(x * x for x in o) - 1
        chord = 2 * torch.sqrt(torch.clamp(bb * bb - aa * cc, min=0)) / aa
        p[i] = (0.019 * chord).reshape(case["nv"], case["nu"])
    counts = 1e5 * torch.exp(-p)
    noise = torch.randn(p.shape, device=DEVICE, dtype=torch.float64, generator=g)
    counts = torch.clamp(torch.round(counts + torch.sqrt(counts) * noise), min=1)
    return counts, math.log(1e5) - torch.log(counts)


def prepare(case, seed):
    c = dict(DEFAULTS, **case)
    if c["kind"] == "batch":
        items, projs = [], []
        for k, b in enumerate(_batch_cases(c)):
            pr = _projector(b, _volumes(b, seed + 101 * k))
            I = torch.empty((b["count"], b["nv"], b["nu"]), device=DEVICE)
            items.append((pr, 0, b["count"], I, torch.empty_like(I)))
            projs.append(pr)
        return dict(case=c, projs=projs, batch=P.Batch(items), out=[t for it in items for t in it[3:]])
    if c["kind"] == "host":
        labels, density = _labels(c, seed)
        return dict(case=c, proj=_projector(c), labels=labels, density=density)
    if c["kind"] == "step":
        proj = _projector(c)
        counts, target = _measured(c, seed)
        rho = _volumes(c, seed, noise=0.1).requires_grad_(True)
        return dict(case=c, proj=proj, rho=rho, I0=proj.flat_field().double(), counts=counts, target=target)
    return dict(case=c, proj=_projector(c, _volumes(c, seed)))


def run(state):
    c = state["case"]
    if c["kind"] == "batch":
        state["batch"].run()
        return state["out"]
    proj = state["proj"]
    if c["kind"] == "host":
        proj.set_labels(state["labels"], state["density"], False, storage_dtype=DTYPES[c["dtype"]])
        return proj.forward_host()
    if c["kind"] == "step":
        rho = state["rho"]
        rho.grad = None
        I, IA = A.project(rho, proj, c["first"], c["count"], DTYPES[c["dtype"]], keep_line_integrals=c["keep"])
        loss = A.wls_loss(A.log_projection(I.double(), state["I0"]), state["target"], state["counts"])
        loss.backward()
        return [I.detach(), IA.detach(), rho.grad, loss.detach()]
    return proj.forward(c["first"], c["count"])


def work(case):
    """Samples inside the phantom's box at eight multiply-adds a material,
    every ray's energy sums (M multiply-adds, an exponential and two weighted
    sums per bin), both twice for a gradient step; every input and output
    moved once."""
    c = dict(DEFAULTS, **case)
    if c["kind"] == "batch":
        each = [work(b) for b in _batch_cases(c)]
        return {k: sum(e[k] for e in each) for k in ("bytes", "flops")}
    rays, nvox = c["count"] * c["nu"] * c["nv"], c["nx"] * c["ny"] * c["nz"]
    bins = int(c["kvp"]) - 19
    flops = 16.0 * c["mats"] * _samples(c) + rays * bins * (2.0 * c["mats"] + 5)
    table = 4.0 * bins * c["nu"] * (c["nv"] if c["jitter"] else 1)
    if c["kind"] == "step":
        return {"bytes": 8.0 * c["mats"] * nvox + rays * (8.0 + 16.0) + table, "flops": 2 * flops}
    if c["kind"] == "host":
        return {"bytes": nvox + 8.0 * rays + table, "flops": flops}
    store = 4.0 if c["dtype"] == "f32" else 2.0
    return {"bytes": store * c["mats"] * nvox + 8.0 * rays + table, "flops": flops}


# ----------------------------------------------------- the method in 64 bits

def _scalars(case):
    """The scan's derived scalars, in FP32 as the method defines them."""
    f = np.float32
    half_u, half_v = f(case["nu"]) * f(case["pitch"]) / f(2), f(case["nv"]) * f(case["pitch"]) / f(2)
    sod, sdd = f(1000.0), f(1500.0)
    fov = sod * half_u / np.sqrt(half_u * half_u + sdd * sdd)
    length = [f(case[n] * case[p]) for n, p in (("nx", "px"), ("ny", "py"), ("nz", "pz"))]
    size = [l / f(case[n]) for l, n in zip(length, ("nx", "ny", "nz"))]
    dx = f(0.5 * float(size[0]))
    step = f(360) / f(case["views"])
    ratio = f(2) * fov / dx
    return dict(half_u=float(half_u), half_v=float(half_v), pitch=float(f(case["pitch"])), sod=1000.0, sdd=1500.0,
                size=[float(x) for x in size], half=[float(l / f(2)) for l in length], dx=float(dx),
                K=int(math.floor(float(ratio) + 0.5)), t0=1000.0 - float(fov) + float(dx) / 2, step=step)


def _rays(case, s, u, v, view, offset):
    """Source (index space) and direction per mm of rays (u, v) of a view:
    the lattice samples are source + t direction, t = t0 + k dx."""
    f = np.float32
    ang = float(f(case["rot"] * view) * s["step"] / f(180) * np.arccos(f(-1.0)))
    c, n = math.cos(ang), math.sin(ang)
    du = s["half_u"] - s["pitch"] / 2 - u * s["pitch"]
    dv = s["half_v"] - s["pitch"] / 2 - v * s["pitch"]
    r = torch.sqrt(s["sdd"] ** 2 + du * du + dv * dv)
    cg, sg = torch.sqrt(s["sdd"] ** 2 + du * du) / r, dv / r
    cb, sb = torch.sqrt(s["sdd"] ** 2 + dv * dv) / r, du / r
    X, Y, Z = cg * cb, cg * sb, sg
    fu, fv = (0.0, 0.0) if offset is None else (float(offset[0]), float(offset[1]))
    if offset is not None:
        qx, qy, qz = torch.full_like(X, s["sdd"]), s["sdd"] * Y / X - fu, s["sdd"] * Z / X - fv
        q = torch.sqrt(qx * qx + qy * qy + qz * qz)
        X, Y, Z = qx / q, qy / q, qz / q
    px, py, pz = s["size"]
    hx, hy, hz = s["half"]
    src = ((hx - s["sod"] * c - fu * n) / px, (hy + s["sod"] * n - fu * c) / py, (hz - fv) / pz)
    return src, ((X * c - Y * n) / px, -(X * n + Y * c) / py, -Z / pz)


def _exact_lines(case, vol, offsets, backproject=None):
    """Line integrals [count][mats][nv][nu] in FP64; with `backproject`
    [count][mats][nv][nu], their adjoint instead."""
    s = _scalars(case)
    nu, nv = case["nu"], case["nv"]
    u = torch.arange(nu, device=DEVICE, dtype=torch.float64).repeat(nv)
    v = torch.arange(nv, device=DEVICE, dtype=torch.float64).repeat_interleave(nu)
    dims = (case["nx"], case["ny"], case["nz"])
    # samples of the lattice that can lie in the volume's bounding sphere
    reach = math.sqrt(sum(((n + 2) * p) ** 2 for n, p in zip(dims, s["size"]))) / 2 + 2
    k0 = max(0, int((s["sod"] - reach - s["t0"]) / s["dx"]))
    k1 = min(s["K"], int((s["sod"] + reach - s["t0"]) / s["dx"]) + 2)
    t = s["t0"] + torch.arange(k0, k1, device=DEVICE, dtype=torch.float64) * s["dx"]
    leaf = vol[None].double()
    if backproject is not None:
        leaf = torch.zeros_like(leaf).requires_grad_(True)
        total = torch.zeros_like(leaf)
    out = torch.zeros((case["count"], case["mats"], nv * nu), dtype=torch.float64, device=DEVICE)
    per = max(1, (1 << 24) // max(1, k1 - k0))
    for i in range(case["count"]):
        view = case["first"] + i
        src, d = _rays(case, s, u, v, view, None if offsets is None else offsets[view])
        for r in range(0, nu * nv, per):
            axes = [((src[a] + d[a][r:r + per, None] * t) * 2 / (dims[a] - 1) - 1) for a in range(3)]
            grid = torch.stack(axes, dim=-1)[None, None]
            got = torch.nn.functional.grid_sample(leaf, grid, mode="bilinear", padding_mode="zeros",
                                                  align_corners=True)[0, :, 0].sum(-1) * s["dx"]
            if backproject is None:
                out[i, :, r:r + per] = got
            else:
                w = backproject[i].reshape(case["mats"], -1)[:, r:r + per]
                total += torch.autograd.grad((got * w).sum(), leaf)[0]
    return out.reshape(case["count"], case["mats"], nv, nu) if backproject is None else total[0].detach()


def _exact_weights(case):
    """W [bins][nv][nu] and attenuation [bins][mats] of the non-zero bins."""
    kw = _spectral(case)
    as64 = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEVICE).double()
    spec, atten = as64(kw["spectrum"]), as64(kw["atten"])
    if kw["energy_weighting"]:
        spec = spec * torch.arange(1, spec.numel() + 1, device=DEVICE, dtype=torch.float64)
    on = (spec != 0).nonzero()[:, 0]
    thick = as64(kw["scint_thickness"]).reshape(1, case["nv"], case["nu"])
    W = kw["i0_val"] * spec[on][:, None, None] * kw["det_factor"] * -torch.expm1(
        -as64(kw["scint_mu"])[on][:, None, None] * thick)
    if "grid" in kw:
        W = W * as64(kw["grid"])[on][:, None, :]
    return W, atten[on]


def _exact_intensity(case, L):
    W, atten = _exact_weights(case)
    I, IA = torch.zeros_like(L[:, 0]), torch.zeros_like(L[:, 0])
    for e in range(W.shape[0]):
        tau = sum(atten[e, m] * L[:, m] for m in range(case["mats"]))
        I += W[e] * torch.exp(-tau)
        IA -= W[e] * torch.expm1(-tau)
    return I, IA, W, atten


def exact(case, seed):
    c = dict(DEFAULTS, **case)
    if c["kind"] == "batch":
        cases = _batch_cases(c)
        if sum(_samples(b) for b in cases) > 1.2e10:
            return None
        out = []
        for k, b in enumerate(cases):
            out += _exact_intensity(b, _exact_lines(b, _volumes(b, seed + 101 * k), None))[:2]
        return out
    if _samples(c) * (4 if c["kind"] == "step" else 1) * (c["mats"] + 2) / 5 > 1.2e10:
        return None
    if c["kind"] == "host":
        labels, density = _labels(c, seed)
        lab = torch.from_numpy(labels).to(DEVICE)
        vol = torch.stack([(lab == m + 1).double() * float(np.float32(density[m])) for m in range(c["mats"])])
        I, IA, W, _ = _exact_intensity(c, _exact_lines(c, vol, None if not c["focal"] else _focal(c)))
        return [I.cpu().numpy(), IA.cpu().numpy(), W.sum(0).expand(c["nv"], c["nu"]).cpu().numpy()]
    vol = _volumes(c, seed, noise=0.1 if c["kind"] == "step" else 0.0)
    offsets = _focal(c)
    L = _exact_lines(c, vol, offsets)
    I, IA, W, atten = _exact_intensity(c, L)
    if c["kind"] == "forward":
        return [I, IA]
    counts, target = _measured(c, seed)
    I0 = W.sum(0)
    p = torch.log(I0) - torch.log(torch.clamp(I, min=1e-12))
    gI = -counts * (p - target) / I
    gL = torch.zeros_like(L)
    for e in range(W.shape[0]):
        we = W[e] * torch.exp(-sum(atten[e, m] * L[:, m] for m in range(c["mats"])))
        for m in range(c["mats"]):
            gL[:, m] -= gI * atten[e, m] * we
    return [I, IA, _exact_lines(c, vol, offsets, gL), 0.5 * (counts * (p - target) ** 2).sum()]
