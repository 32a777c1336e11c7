"""The workloads whose speed is measured, each one pass through the public entry points.

A case is a dict of plain values: ``kind`` (the call), the scanner and image
sizes, and the options of that kind. Sizes are those of the 8-ring, RPT, 24-ring
and mMR-size configurations of ``stir_amd.geometry``; ``draw`` takes others from
the ranges they stand for. Kinds:

* ``forward`` / ``back``: one projection of a device image / of device data
  (also time of flight, where ``tof`` gives the number of timing bins);
* ``osem``: ``steps`` OSMAPOSL subiterations of a device image;
* ``gradient``: Poisson log-likelihood + quadratic prior, forward and backward,
  of a batch of images (values and gradient images);
* ``hessian``: the exact Hessian product of the log-likelihood, all subsets;
* ``map``: one-step-late OSMAPOSL with the relative difference prior, host
  image in and out;
* ``batch``: several uneven reconstructions advanced together, host images in
  and out.

``exact`` restates each of them in float64 from the scanner's geometry alone.
"""
import math

import numpy as np
import torch

from stir_amd.autograd import PoissonLogLikelihoodLoss, QuadraticPriorLoss, UnrolledOSEM, back_project, forward_project
from stir_amd.batch import BatchedOSMAPOSL
from stir_amd.geometry import ProjDataInfoCylindrical, RayTracingMatrixParameters, Scanner, VoxelsOnCartesianGrid
from stir_amd.projectors import (OSMAPOSLReconstruction, PoissonLogLikelihoodWithLinearModelForMeanAndProjData,
                                 ProjectorByBinPairMI355X, ProjMatrixByBinUsingRayTracing, RelativeDifferencePrior)

BACKGROUND = 0.05  # constant additive term, counts per bin
PRIOR_BETA = 0.01  # quadratic prior of the gradient
MAP_BETA, MAP_GAMMA, MAP_EPSILON = 0.1, 2.0, 1e-3
MM_PER_PS = 0.149896229  # half the speed of light
FWHM_PS = 400.0
EXACT_LIMIT = 1.5e11  # elements visited in float64 above which exact() would take longer than about 20 seconds

_EIGHT = dict(rings=8, crystals=192, radius=300.0, spacing=4.0, span=1, mrd=3, views=96, tang=128, xy=128, vox=2.0,
              bin=4.908739, arc=False, lors=1, tilt=0.0, sym90=True, tof=0, tof_ps=0.0)
_RPT = dict(rings=16, crystals=384, radius=380.0, spacing=6.75, span=1, mrd=3, views=96, tang=128, xy=60,
            vox=float(np.float32(3.1088) / np.float32(0.7)), bin=3.1088, arc=True, lors=2,
            tilt=math.radians(-0.46875), sym90=True, tof=0, tof_ps=0.0)
_RING24 = dict(rings=24, crystals=288, radius=350.0, spacing=4.0, span=3, mrd=23, views=144, tang=143, xy=191, vox=2.0,
               bin=3.817908, arc=False, lors=1, tilt=0.0, sym90=True, tof=0, tof_ps=0.0)
_MMR = dict(rings=64, crystals=504, radius=328.0, spacing=4.0625, span=11, mrd=60, views=252, tang=344, xy=344,
            vox=2.08626, bin=2.08626, arc=False, lors=1, tilt=0.0, sym90=True, tof=0, tof_ps=0.0)
_MMR_TOF = dict(_MMR, tof=11, tof_ps=594.0)


def listed():
    return [
        # a small research or animal scanner: launches and layout conversions count
        dict(_EIGHT, name="forward_8ring", kind="forward", subsets=1),
        dict(_EIGHT, name="back_8ring", kind="back", subsets=1),
        # one full OSEM iteration of it, 16 short kernels and the image conversions between them
        dict(_EIGHT, name="osem_8ring", kind="osem", subsets=8, steps=8),
        # the reference's RPT recipe (arc-corrected data, two tangential LORs, zoomed 60 x 60 image) with a prior
        dict(_RPT, name="map_rpt", kind="map", subsets=4, steps=4),
        # a mid-size scanner with axial compression: odd sizes, one and two planes per axial position mixed
        dict(_RING24, name="hessian_24ring", kind="hessian", subsets=9),
        # several uneven small studies reconstructed together (gated or dynamic frames, animal studies)
        dict(name="batch_6", kind="batch", problems=6, draw_seed=4, subsets=8, steps=8),
        # whole-scanner projections at mMR size: simulation, sensitivities, data consistency
        dict(_MMR, name="forward_mmr", kind="forward", subsets=21),
        dict(_MMR, name="back_mmr", kind="back", subsets=21),
        # the clinical reconstruction: one iteration of 21 subsets
        dict(_MMR, name="osem_mmr", kind="osem", subsets=21, steps=21),
        # a training or optimisation step: gradient of the penalised objective for a batch of two images
        dict(_MMR, name="gradient_mmr", kind="gradient", subsets=21, images=2),
        # time of flight with 11 timing bins, both directions
        dict(_MMR_TOF, name="tof_forward_mmr", kind="forward", subsets=21),
        dict(_MMR_TOF, name="tof_back_mmr", kind="back", subsets=21),
    ]


def draw(rng):
    """One more case: any kind, 6 to 64 rings, non-TOF or 5 to 13 timing bins."""
    while True:
        kind = rng.choice(["forward", "back", "osem", "gradient", "hessian", "map", "batch", "tof_forward", "tof_back"])
        if kind == "batch":
            return dict(kind="batch", problems=rng.randint(2, 8), draw_seed=rng.randint(10, 10**6),
                        subsets=rng.choice([4, 8]), steps=rng.randint(4, 8))
        rings = int(round(math.exp(rng.uniform(math.log(6), math.log(64)))))
        crystals = 8 * rng.randint(20, 63)
        spans = [1, 3] if rings < 20 else [3, 5, 7] if rings < 40 else [7, 9, 11]
        span = rng.choice(spans)
        mrd = rng.randint(max((span - 1) // 2, rings // 3), rings - 1)
        radius = rng.choice([300.0, 328.0, 350.0, 400.0])
        tang = crystals // 2 + rng.choice([0, 0, -1, -3, crystals // 8])
        xy = int(round(math.exp(rng.uniform(math.log(60), math.log(344)))))
        vox = rng.uniform(0.8, 1.3) * radius / xy
        views = crystals // 2
        subsets = rng.choice([n for n in range(2, 25) if views % n == 0 and n <= views // 8])
        case = dict(kind=kind.replace("tof_", ""), rings=rings, crystals=crystals, radius=radius,
                    spacing=rng.choice([4.0, 4.0625, 5.0]), span=span, mrd=mrd, views=views, tang=tang, xy=xy,
                    vox=float(np.float32(vox)), bin=math.pi * radius / crystals, arc=rng.random() < 0.2,
                    lors=2 if rng.random() < 0.15 else 1, tilt=0.0, sym90=rng.random() < 0.8, tof=0, tof_ps=0.0,
                    subsets=subsets)
        if kind.startswith("tof_"):
            case.update(tof=rng.choice([5, 7, 8, 9, 11, 13]), arc=False, lors=1)
            case["tof_ps"] = float(round(1.1 * radius * 2 / case["tof"] / MM_PER_PS, 1))
        if case["kind"] in ("osem", "map"):
            case["steps"] = rng.randint(2, subsets)
        if case["kind"] == "gradient":
            case["images"] = rng.randint(1, 2)
        w = work(case)
        if w["flops"] <= (1.0 if case["tof"] else 0.8) * work(listed()[6])["flops"] and w["bytes"] <= 2e9:
            return case


# ---- geometry -------------------------------------------------------------
def _batch_problems(case):
    """Uneven small problems as ``stir_amd.geometry.config4_problems`` chooses
    them: 8 to 32 rings, 96 to 256 voxels across."""
    r = np.random.default_rng(case["draw_seed"])
    out = []
    for _ in range(case["problems"]):
        rings = int(r.choice([8, 16, 24, 32]))
        crystals = int(r.choice([192, 288, 384]))
        xy = int(r.choice([96, 128, 192, 256]))
        out.append(dict(rings=rings, crystals=crystals, radius=350.0, spacing=4.0, span=1 if rings <= 16 else 3,
                        mrd=rings - 1, views=crystals // 2, tang=crystals // 2, xy=xy, vox=2.0,
                        bin=math.pi * 350.0 / crystals, arc=False, lors=1, tilt=0.0, sym90=crystals != 288, tof=0,
                        tof_ps=0.0, subsets=case["subsets"], steps=case["steps"]))
    return out


def _setup(c):
    sc = Scanner("scanner", c["rings"], c["crystals"], c["radius"], 0.0, c["spacing"], float(np.float32(c["bin"])),
                 c["tilt"], c["tang"], c["tang"], FWHM_PS if c["tof"] else 0.0, c["tof_ps"], c["tof"])
    pdi = ProjDataInfoCylindrical.construct(sc, c["span"], c["mrd"], c["views"], c["tang"], c["arc"])
    if c["tof"]:
        pdi = pdi.with_tof(1)
    img = VoxelsOnCartesianGrid(2 * c["rings"] - 1, c["xy"], c["xy"], c["spacing"] / 2, float(np.float32(c["vox"])),
                                float(np.float32(c["vox"])))
    pm = RayTracingMatrixParameters(num_tangential_LORs=c["lors"], do_symmetry_90degrees_min_phi=c["sym90"])
    return pdi, img, pm


def _segments(c):
    """(segment, mean ring difference, axial positions, axial sampling) in storage order 0, +1, -1, ..."""
    span, mrd, nr = c["span"], c["mrd"], c["rings"]
    lo = [-((span - 1) // 2)]
    hi = [lo[0] + span - 1]
    while hi[-1] < mrd:
        lo.append(hi[-1] + 1)
        hi.append(lo[-1] + span - 1)
    hi[-1] = min(hi[-1], mrd)
    out = []
    for i, (a, b) in enumerate(zip(lo, hi)):
        nax = (nr if i == 0 else nr - i) if span == 1 else (2 * nr - 1 if i == 0 else 2 * nr - 1 - 2 * a)
        samp = c["spacing"] / (2 if a != b else 1)
        out.append((i, (a + b) / 2.0, nax, samp))
        if i:
            out.append((-i, -(a + b) / 2.0, nax, samp))
    return out


def _num_bins(c):
    return sum(s[2] for s in _segments(c)) * c["views"] * c["tang"] * max(1, c["tof"])


def _s_of(c, t):
    if c["arc"]:
        return t * c["bin"]
    return c["radius"] * np.sin(t * math.pi / c["crystals"])


def _fov(c):
    return (c["xy"] // 2 - (1 - c["xy"] % 2)) * c["vox"]


def _nnz(c):
    """Matrix elements of all bins, from the mean number of voxels a chord meets."""
    t = np.arange(c["tang"]) - c["tang"] // 2
    chord = 2 * np.sqrt(np.maximum(_fov(c) ** 2 - _s_of(c, t) ** 2, 0))
    total = 0.0
    for _, delta, nax, samp in _segments(c):
        lors = max(1, round(samp / (c["spacing"] / 2)))
        copies = lors if delta else (3 if lors == 2 else 1)
        along = chord * (4 / math.pi / c["vox"] + abs(delta) * c["spacing"] / (2 * c["radius"]) / (c["spacing"] / 2))
        total += nax * c["views"] * copies * c["lors"] * along.sum()
    return total


def work(case):
    """Two operations per matrix element and projection; data, images and
    sensitivities read or written once."""
    if case["kind"] == "batch":
        parts = [work(dict(p, kind="osem")) for p in _batch_problems(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    nnz, image, data = _nnz(case), 4 * (2 * case["rings"] - 1) * case["xy"] ** 2, 4 * _num_bins(case)
    live = 4 if case["tof"] else 1  # timing bins an element reaches
    kind = case["kind"]
    if kind in ("forward", "back"):
        return {"bytes": image + data, "flops": 2 * nnz * live}
    if kind in ("osem", "map"):
        part = case["steps"] / case["subsets"]
        return {"bytes": (2 + case["steps"]) * image + data * part, "flops": 4 * nnz * part}
    if kind == "gradient":
        return {"bytes": 2 * case["images"] * image + data, "flops": 4 * nnz * case["images"]}
    return {"bytes": 3 * image + data, "flops": 6 * nnz}  # hessian: two forward, one back


# ---- inputs, from the seed alone --------------------------------------------
def _device():
    return torch.device("cuda:0" if torch.cuda.is_available() else "cpu")


def _image(c, seed, noise=0.1):
    """Ellipsoidal body of activity 1 with eight hot spheres, times log-normal noise (an early iterate)."""
    dev = _device()
    nz, n = 2 * c["rings"] - 1, c["xy"]
    r = np.random.default_rng(seed)
    g = torch.Generator(device=dev).manual_seed(seed)
    z = (torch.arange(nz, device=dev, dtype=torch.float32) - (nz - 1) / 2).view(-1, 1, 1) * (c["spacing"] / 2)
    y = ((torch.arange(n, device=dev, dtype=torch.float32) - n // 2) * c["vox"]).view(1, -1, 1)
    x = ((torch.arange(n, device=dev, dtype=torch.float32) - n // 2) * c["vox"]).view(1, 1, -1)
    R = _fov(c)
    out = ((x / (0.7 * R)) ** 2 + (y / (0.5 * R)) ** 2 <= 1).float().expand(nz, -1, -1) + 0.02
    for _ in range(8):
        rad, val = r.uniform(0.03, 0.1) * R, r.uniform(3, 8)
        cx, cy, cz = r.uniform(-0.5, 0.5) * R, r.uniform(-0.35, 0.35) * R, r.uniform(-0.4, 0.4) * nz * c["spacing"] / 2
        out = torch.where((x - cx) ** 2 + (y - cy) ** 2 + (z - cz) ** 2 <= rad ** 2, float(val), out)
    return out * torch.exp(noise * torch.randn(out.shape, generator=g, device=dev))


def _ratios(c, seed):
    """Projection data as the quotient of measured and estimated counts: around 1, all positive."""
    dev = _device()
    g = torch.Generator(device=dev).manual_seed(seed)
    return torch.randn(_num_bins(c), generator=g, device=dev).mul_(0.3).exp_()


def _counts(c, seed):
    """Poisson counts of a uniform cylinder (mean about 2 per bin through its centre) plus the background."""
    dev = _device()
    g = torch.Generator(device=dev).manual_seed(seed)
    t = np.arange(c["tang"]) - c["tang"] // 2
    profile = torch.from_numpy(np.sqrt(np.maximum(1 - (_s_of(c, t) / (0.7 * _fov(c))) ** 2, 0))).to(dev).float()
    mean = (2 * profile + BACKGROUND).expand(_num_bins(c) // c["tang"], c["tang"])
    return torch.poisson(mean.contiguous(), generator=g).reshape(-1)


# ---- state and pass ---------------------------------------------------------
def _pair(c):
    pdi, img, pm = _setup(c)
    pair = ProjectorByBinPairMI355X(ProjMatrixByBinUsingRayTracing(pm))
    pair.set_up(pdi, img, num_subsets=c["subsets"])
    return pair


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        problems = _batch_problems(case)
        batch = BatchedOSMAPOSL([_setup(p) for p in problems], case["subsets"])
        for i, p in enumerate(problems):
            batch.set_data(i, _counts(p, seed + i).cpu().numpy(), BACKGROUND)
        start = [_image(p, seed + i).cpu().numpy() for i, p in enumerate(problems)]
        return dict(kind=kind, batch=batch, start=start, steps=case["steps"])
    state = dict(kind=kind, pair=_pair(case))
    if kind == "forward":
        state["x"] = _image(case, seed)
        return state
    if kind == "back":
        state["p"] = _ratios(case, seed)
        return state
    obj = PoissonLogLikelihoodWithLinearModelForMeanAndProjData(state["pair"])
    # the Hessian product and the gradient need no sensitivities
    obj.set_up(_counts(case, seed).cpu().numpy(), BACKGROUND, compute_sensitivities=kind in ("osem", "map"))
    state["obj"] = obj
    if kind == "osem":
        state["x"] = _image(case, seed)
        state["recon"] = UnrolledOSEM(obj, case["steps"])
    elif kind == "map":
        obj.set_prior(RelativeDifferencePrior(MAP_BETA, gamma=MAP_GAMMA, epsilon=MAP_EPSILON))
        state["x"] = _image(case, seed).cpu().numpy()
        state["recon"] = OSMAPOSLReconstruction(obj, num_subiterations=case["steps"])
        state["subsets"] = case["subsets"]
        state["steps"] = case["steps"]
    elif kind == "gradient":
        state["x"] = torch.stack([_image(case, seed + i) for i in range(case["images"])])
        state["nll"] = PoissonLogLikelihoodLoss(obj)
        state["prior"] = QuadraticPriorLoss(state["pair"], PRIOR_BETA)
    else:
        state["x"] = _image(case, seed)
        state["v"] = _image(case, seed + 1)
    return state


def run(state):
    kind = state["kind"]
    if kind == "forward":
        return forward_project(state["x"], state["pair"])
    if kind == "back":
        return back_project(state["p"], state["pair"])
    if kind == "osem":
        with torch.no_grad():
            return state["recon"](state["x"])
    if kind == "gradient":
        x = state["x"].detach().requires_grad_(True)
        values = state["nll"](x) + state["prior"](x)
        values.sum().backward()
        return values.detach(), x.grad
    if kind == "hessian":
        out = torch.zeros_like(state["v"])
        return state["obj"].accumulate_Hessian_times_input_without_penalty(out, state["x"], state["v"])
    if kind == "map":
        state["obj"].set_estimate(state["x"], enforce_positivity=True)
        for k in range(1, state["steps"] + 1):
            state["recon"].update_estimate((k - 1) % state["subsets"], k)
        return state["obj"].get_estimate()
    batch = state["batch"]
    for i, x in enumerate(state["start"]):
        batch.set_estimate(i, x)
    batch.run(state["steps"])
    batch.synchronize()
    return [batch.get_estimate(i) for i in range(len(batch))]


# ---- the same in float64, from the geometry ---------------------------------
class _Matrix64:
    """Ray-tracing matrix in float64: chunks of rays traced through the voxel
    grid, applied to all axial positions of their (segment, view, tangential
    position) by shifting z."""

    def __init__(self, c):
        self.c, self.dev = c, _device()
        self.nz, self.n = 2 * c["rings"] - 1, c["xy"]
        self.vz, self.vx = c["spacing"] / 2, float(np.float32(c["vox"]))
        self.segs, off = [], 0
        for seg, delta, nax, samp in _segments(c):
            self.segs.append((seg, delta, nax, samp, off))
            off += nax * c["views"] * c["tang"]
        self.block, self.ntof = off, max(1, c["tof"])
        t = np.arange(c["tang"]) - c["tang"] // 2
        self.s = _s_of(c, t)
        self.ds = np.full(len(t), c["bin"]) if c["arc"] else np.abs(_s_of(c, t + 1) - _s_of(c, t - 1)) / 2
        self.phi0 = c["tilt"]
        if 2 * c["views"] != c["crystals"] and c["crystals"] % (2 * c["views"]) == 0:
            self.phi0 += math.pi / c["crystals"] * (c["crystals"] / 2 / c["views"] - 1)
        straight = abs(self.phi0) < 1e-4 and not c["tof"]
        self.sym90 = straight and c["sym90"] and c["views"] % 4 == 0
        self.sym180 = straight and c["views"] % 2 == 0

    def subset_of(self, view):
        nv = self.c["views"]
        if self.sym90:
            if view >= 3 * (nv // 4):
                view = nv - view
            elif view >= nv // 2:
                view -= nv // 2
            elif view > nv // 4:
                view = nv // 2 - view
        elif self.sym180 and view > nv // 2:
            view = nv - view
        return view % self.c["subsets"]

    def _rays(self, delta, samp, nax, views):
        """Voxel column, plane and weight of every element of the rays of axial
        position 0 (views x tangential positions x tangential LORs), and the
        axial copies (plane offset, weight)."""
        c, dev, vz, vx = self.c, self.dev, self.vz, self.vx
        f = dict(dtype=torch.float64, device=dev)
        nt = c["lors"]
        s0 = torch.tensor(self.s, **f).view(1, -1)
        k = (torch.arange(nt, **f) - (nt - 1) / 2).view(-1, 1)
        s = (s0 + k * torch.tensor(self.ds, **f).view(1, -1) / nt)  # [nt, tang]
        tan = delta * c["spacing"] / (2 * torch.sqrt(c["radius"] ** 2 - s0 ** 2))  # of the bin, [1, tang]
        phi = torch.tensor([self.phi0 + v * math.pi / c["views"] for v in views], **f).view(-1, 1, 1)
        s, tan = s.unsqueeze(0), tan.unsqueeze(0)
        fov = _fov(dict(c, vox=vx))
        a = torch.sqrt(torch.clamp(fov ** 2 - s ** 2, min=0))
        inside = (s.abs() <= fov)
        lors = max(1, math.ceil(samp / vz - 1e-3))
        m = -(nax - 1) * samp / 2
        off = -samp / (2 * lors) * (lors - 1) + (self.nz - 1) / 2 * vz
        if delta == 0 and abs(((m + off) / vz) % 1.0 - 0.5) < 1e-3:
            off -= 0.1 * vz

        def at(sign):
            return torch.stack([(s * torch.cos(phi) + sign * a * torch.sin(phi)) / vx,
                                (s * torch.sin(phi) - sign * a * torch.cos(phi)) / vx,
                                ((m + off - sign * a * tan) / vz).expand(len(views), -1, -1)], -1).reshape(-1, 3)

        st, sp = at(1), at(-1)
        inside = inside.expand(len(views), -1, -1).reshape(-1)
        d = sp - st
        moving = d.abs() > 1e-4
        dd = torch.where(moving, d, torch.ones_like(d))
        sg = torch.where(d >= 0, 1.0, -1.0).double()
        rnd = lambda v: torch.where(v >= 0, torch.floor(v + 0.5), -torch.floor(-v + 0.5))
        first = torch.where(moving, (rnd(st) - 0.5 * sg - st) / dd, torch.full_like(d, -math.inf)).amax(1)
        last = torch.where(moving, (rnd(sp) + 0.5 * sg - st) / dd, torch.full_like(d, math.inf)).amin(1)
        planes = []
        for ax, count in ((0, self.n + 1), (1, self.n + 1), (2, int(d[:, 2].abs().max().item()) + 3)):
            j = torch.arange(count, **f).view(1, -1)
            p = j - self.n // 2 - 0.5 if ax < 2 else rnd(st[:, 2:3]) + sg[:, 2:3] * (j - 0.5)
            al = (p - st[:, ax:ax + 1]) / dd[:, ax:ax + 1]
            planes.append(torch.where(moving[:, ax:ax + 1], al, first.view(-1, 1)))
        al = torch.cat(planes, 1)
        al = torch.minimum(torch.maximum(al, first.view(-1, 1)), last.view(-1, 1)).sort(1).values
        mid = (al[:, 1:] + al[:, :-1]) / 2
        length = torch.sqrt((d[:, 0] * vx) ** 2 + (d[:, 1] * vx) ** 2 + (d[:, 2] * vz) ** 2)
        w = (al[:, 1:] - al[:, :-1]) * (length / vx / lors / nt * inside).view(-1, 1)
        x, y, z = (rnd(st[:, i:i + 1] + mid * d[:, i:i + 1]).long() for i in range(3))
        ok = (x >= -(self.n // 2)) & (x < self.n - self.n // 2) & (y >= -(self.n // 2)) & (y < self.n - self.n // 2)
        w = torch.where(ok & (w > 1e-12), w, torch.zeros_like(w))
        col = torch.where(ok, (y + self.n // 2) * self.n + x + self.n // 2, torch.zeros_like(x))
        if delta == 0:
            z0 = math.floor((m + off) / vz + 0.5)
            zf, right = z0 - (self.nz - 1) / 2 - (m - samp / 2) / vz, samp / vz
            copies = [(i, min(right, zf + i + 0.5) - max(0.0, zf + i - 0.5)) for i in range(-1, 6)]
            copies = [(i, o) for i, o in copies if o > 1e-4]
        else:
            copies = [(i, 1.0) for i in range(lors)]
        # the tangential LORs of a bin follow each other: [views, nt, tang, E] -> [views * tang, nt * E]
        shape = (len(views), nt, c["tang"], -1)
        col, z, w = (v.reshape(shape).permute(0, 2, 1, 3).reshape(len(views) * c["tang"], -1) for v in (col, z, w))
        tofw = None
        if c["tof"]:
            cos_theta = 1 / torch.sqrt(1 + tan ** 2)  # direction of the LOR (z, y, x), from its first to its second end
            u = [(tan * cos_theta).expand(len(views), 1, -1), torch.cos(phi) * cos_theta, -torch.sin(phi) * cos_theta]
            mid3 = [torch.full_like(u[0], m), s * torch.sin(phi), s * torch.cos(phi)]
            u, mid3 = ([v.reshape(-1, 1) for v in q] for q in (u, mid3))
            py = ((col // self.n) - self.n // 2) * vx
            px = ((col % self.n) - self.n // 2) * vx
            inc, r = c["tof_ps"] * MM_PER_PS, 2.355 / (FWHM_PS * MM_PER_PS * math.sqrt(2.0))

            def tofw(k, dz):
                pz = (z + dz) * vz - (c["rings"] - 1) / 2 * c["spacing"]
                dist = -((pz - mid3[0]) * u[0] + (py - mid3[1]) * u[1] + (px - mid3[2]) * u[2])
                centre = (k - c["tof"] // 2) * inc + (inc / 2 if c["tof"] % 2 == 0 else 0.0)
                lo, hi = (centre - inc / 2 - dist) * r, (centre + inc / 2 - dist) * r
                v = 0.5 * (torch.erf(hi) - torch.erf(lo))
                return torch.where(((lo >= 4) & (hi >= 4)) | ((lo <= -4) & (hi <= -4)), torch.zeros_like(v), v)
        return col, z, w, copies, tofw

    def _apply(self, subset, step):
        """step(data slice, column * (nz + 2), z, weight, plane offset, timing bin) over all elements."""
        c = self.c
        views = [v for v in range(c["views"]) if subset is None or self.subset_of(v) == subset]
        for seg, delta, nax, samp, off in self.segs:
            ppa = round(samp / self.vz)
            per = max(1, int(4e6 / (c["tang"] * c["lors"] * (2 * self.n + 40))))
            for i in range(0, len(views), per):
                vs = views[i:i + per]
                col, z, w, copies, tofw = self._rays(delta, samp, nax, vs)
                tang = torch.arange(c["tang"], device=self.dev)
                base = torch.tensor(vs, device=self.dev).view(-1, 1) * c["tang"] + tang
                keep = (w > 0).any(0).nonzero().view(-1)  # elements that some ray of the chunk has
                if not len(keep):
                    continue
                col, z, w = col[:, keep] * (self.nz + 2), z[:, keep], w[:, keep]
                for k in range(self.ntof):
                    for dz, overlap in copies:
                        wk = w * overlap if tofw is None else w * overlap * tofw(k, dz)[:, keep]
                        if tofw is not None and not (wk > 0).any():
                            continue
                        for ax in range(nax):
                            at = k * self.block + off + ax * c["views"] * c["tang"] + base.reshape(-1)
                            step(at, col + (z + dz + ppa * ax).clamp(-1, self.nz) + 1, wk)

    def forward(self, x, subset=None):
        img = torch.zeros(self.n * self.n, self.nz + 2, dtype=torch.float64, device=self.dev)
        img[:, 1:-1] = x.double().reshape(self.nz, -1).t()
        img, out = img.reshape(-1), torch.zeros(self.block * self.ntof, dtype=torch.float64, device=self.dev)

        def step(at, idx, w):
            out[at] += (img[idx] * w).sum(1)

        self._apply(subset, step)
        return out

    def back(self, p, subset=None):
        p, out = p.double(), torch.zeros(self.n * self.n * (self.nz + 2), dtype=torch.float64, device=self.dev)

        def step(at, idx, w):
            m = w > 0
            out.index_add_(0, idx[m], (p[at].view(-1, 1) * w)[m])

        self._apply(subset, step)
        return out.view(-1, self.nz + 2)[:, 1:-1].t().reshape(self.nz, self.n, self.n)


def _neighbours(x, vz, vx):
    """(weight vox_x / distance, neighbour's value, 1 where it lies inside the image) of the 3 x 3 x 3 neighbourhood."""
    xp = torch.nn.functional.pad(x, (1,) * 6)
    inside = torch.nn.functional.pad(torch.ones_like(x), (1,) * 6)
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                if dz or dy or dx:
                    cut = tuple(slice(1 + o, 1 + o + n) for o, n in zip((dz, dy, dx), x.shape))
                    yield vx / math.sqrt((dz * vz) ** 2 + (dy * vx) ** 2 + (dx * vx) ** 2), xp[cut], inside[cut]


def _osem64(c, A, y, x, map_prior):
    """OSMAPOSL subiterations; the data hold no value that the quotient's thresholds would change."""
    sens = {}
    for k in range(c["steps"]):
        s = k % c["subsets"]
        if s not in sens:
            sens[s] = A.back(torch.ones_like(y), s)
        u, den = A.back(y / (A.forward(x, s) + BACKGROUND), s), sens[s]
        small = 0.0
        if map_prior:
            g = torch.zeros_like(x)
            for w, xn, ins in _neighbours(x, A.vz, A.vx):
                ad = (x - xn).abs()
                den10 = x + xn + MAP_GAMMA * ad + MAP_EPSILON
                g += w * ins * (x - xn) * (MAP_GAMMA * ad + x + 3 * xn + 2 * MAP_EPSILON) / den10 ** 2
            den = torch.minimum(torch.maximum(MAP_BETA * g / c["subsets"] + sens[s], sens[s] / 10), sens[s] * 10)
            small = u.max() * 1e-6
        x = x * torch.where((den.abs() <= small) & (u.abs() <= small), torch.zeros_like(u), u / den)
    return x


def exact(case, seed):
    if case["kind"] == "batch":
        problems = _batch_problems(case)
        if sum(_cost64(dict(p, kind="osem")) for p in problems) > EXACT_LIMIT:
            return None
        return [_osem64(p, _Matrix64(p), _counts(p, seed + i).double(), _image(p, seed + i).double(), False)
                .cpu().numpy() for i, p in enumerate(problems)]
    if _cost64(case) > EXACT_LIMIT:
        return None
    A, kind = _Matrix64(case), case["kind"]
    if kind == "forward":
        return A.forward(_image(case, seed))
    if kind == "back":
        return A.back(_ratios(case, seed))
    y = _counts(case, seed).double()
    if kind in ("osem", "map"):
        x = _osem64(case, A, y, _image(case, seed).double(), kind == "map")
        return x.cpu().numpy() if kind == "map" else x
    if kind == "hessian":
        x, v = _image(case, seed).double(), _image(case, seed + 1)
        return -A.back(y * A.forward(v) / (A.forward(x) + BACKGROUND) ** 2)
    values, grads = [], []
    for i in range(case["images"]):
        x = _image(case, seed + i).double()
        ybar = A.forward(x) + BACKGROUND
        value, grad = (ybar - y * torch.log(ybar)).sum(), -A.back(y / ybar - 1)
        for w, xn, ins in _neighbours(x, A.vz, A.vx):
            value = value + PRIOR_BETA * (w * ins * (x - xn) ** 2 / 4).sum()
            grad = grad + PRIOR_BETA * w * ins * (x - xn)
        values.append(value)
        grads.append(grad)
    return torch.stack(values), torch.stack(grads)


def _cost64(c):
    """Elements that the float64 passes of a case visit, those of weight 0 included."""
    steps, sub = c.get("steps", 1), c["subsets"]
    passes = {"forward": 1, "back": 1, "gradient": 2 * c.get("images", 1), "hessian": 3}.get(
        c["kind"], (2 * steps + min(steps, sub)) / sub)
    rows = sum(nax * (1 if delta else 3) * (1 + (c["span"] == 1 and delta != 0)) for _, delta, nax, _ in _segments(c))
    return rows * c["views"] * c["tang"] * (2 * c["xy"] + 40) * c["lors"] * max(1, c["tof"]) * passes
