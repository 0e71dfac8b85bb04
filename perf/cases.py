"""What a user of the engine has it do, as timed cases.

Kinds of case, each through the package's public entry points:

* transport  one beam into a built world from empty scores, then the dose
             (World / AAVoxelGrid / Transport / doseScored);
* batch      many small worlds in one launch (TransportBatch), doses read;
* infer      the denoiser on one host feature volume (Denoiser.infer);
* apply      the denoiser on a world's own low-history dose (Denoiser.apply);
* train      one training step on a batch of patches, gradients read
             (Denoiser.train_step, Denoiser.grads);
* segment    CT numbers to material and density, on resident device buffers
             (segment_device) or host arrays (CTSegmentationPipeline);
* organs     the organ dose table, resident or from host arrays.

Host arrays go in and come out where the entry point takes host arrays; the
resident variants keep their volumes in device memory, as the caller's program
does.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import opendxmc_amd as dx
from opendxmc_amd import batch_workload, denoise, phantoms, pipelines
from opendxmc_amd.bowtie import DEFAULT_CT_BOWTIE, read_filters

SPACING = (0.1, 0.1, 0.1)      # of the organ dose tables (cm)
ORGAN_ROW = ("n_voxels", "volume_cm3", "mass_g", "dose")


def listed():
    return [
        # A quick look: a 60 keV pencil beam into a small water cube at 1e6 histories.
        # The smallest transport call: launch, drain and read-back latency count.
        _transport("pencil-water-64", "water", (64, 64, 64), 0.1, "pencil", 1, 1e6),
        # A projection X-ray of a small object with binding and fluorescence on
        # (correction level 2), odd grid, output calibrated to a dose-area product.
        _transport("dx-object-level2", "ellipsoid", (97, 161, 79), 0.12, "dx", 2, 5e6),
        # The everyday CT dose run: spiral scan of a body, bowtie, 1e8 histories.
        _transport("ct-spiral-256", "body", (256, 256, 200), 0.15, "spiral", 1, 1e8),
        # Dual-source CT at diagnostic resolution, a short range: most of the grid
        # is tallied once or not at all, and the dose volume is as large as the run.
        _transport("ct-dual-512-slab", "body", (512, 512, 64), 0.08, "dual", 1, 3e7),
        # A study over many small objects: uneven worlds in one launch.
        {"name": "batch-16-uneven", "kind": "batch", "instances": 16, "scale": 0.5, "low": 2.5e5, "high": 5e6},
        # The denoiser on one patch (the smallest call) and on a whole CT volume.
        {"name": "infer-64", "kind": "infer", "nz": 64, "ny": 64, "nx": 64},
        {"name": "infer-128x256x256", "kind": "infer", "nz": 128, "ny": 256, "nx": 256},
        # The denoiser after a low-history run of a body at its training resolution.
        {"name": "apply-body-448", "kind": "apply", "nx": 448, "ny": 448, "nz": 96, "per_voxel": 1.5},
        # One optimiser step of the denoiser's own training recipe: four 64^3 patches.
        {"name": "train-4x64", "kind": "train", "batch": 4, "nz": 64, "ny": 64, "nx": 64},
        # Segmentation of a CT volume that already sits on the device (largest size).
        {"name": "segment-resident-268M", "kind": "segment", "nx": 1024, "ny": 512, "nz": 512, "resident": True},
        # A CT series as it comes from the reader: host arrays in, host arrays out.
        {"name": "segment-host-series", "kind": "segment", "nx": 512, "ny": 512, "nz": 61, "resident": False},
        # Organ doses of a dose volume on the device.
        {"name": "organs-resident-268M", "kind": "organs", "nx": 1024, "ny": 512, "nz": 512, "resident": True, "speckle": False},
    ]


def _transport(name, phantom, dims, spacing, beam, level, histories):
    return {"name": name, "kind": "transport", "phantom": phantom, "nx": dims[0], "ny": dims[1], "nz": dims[2],
            "spacing": spacing, "beam": beam, "level": level, "histories": histories}


def _log(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def _edge(rng, low, high):
    return int(round(_log(rng, low, high)))


def draw(rng):
    kind = rng.choice(["transport"] * 4 + ["batch", "infer", "infer", "apply", "train", "segment", "segment", "organs", "organs"])
    if kind == "transport":
        phantom = rng.choice(["water", "ellipsoid", "body"])
        beam = {"water": ["pencil"], "ellipsoid": ["dx", "sequential", "cbct"], "body": ["spiral", "dual", "sequential"]}[phantom]
        top = 128 if phantom != "body" else 300
        dims = [_edge(rng, 24 if phantom != "body" else 90, top) for _ in range(3)]
        dims[2] = min(dims[2], 128)
        return {"kind": "transport", "phantom": phantom, "nx": dims[0], "ny": dims[1], "nz": dims[2],
                "spacing": round((36.0 if phantom == "body" else 12.0) / max(dims), 4), "beam": rng.choice(beam),
                "level": rng.choice([0, 1, 1, 2]), "histories": round(_log(rng, 2e5, 5e7))}
    if kind == "batch":
        low = _log(rng, 5e4, 5e5)
        return {"kind": "batch", "instances": rng.randint(2, 14), "scale": rng.choice([0.25, 0.37, 0.5]),
                "low": round(low), "high": round(8 * low)}
    if kind == "infer":
        return {"kind": "infer", "nz": _edge(rng, 3, 128), "ny": _edge(rng, 5, 256), "nx": 64 * rng.randint(1, 4)}
    if kind == "apply":
        return {"kind": "apply", "nx": _edge(rng, 64, 448), "ny": _edge(rng, 64, 448), "nz": _edge(rng, 8, 90),
                "per_voxel": round(_log(rng, 0.5, 8.0), 3)}
    if kind == "train":
        return {"kind": "train", "batch": rng.randint(1, 4), "nz": _edge(rng, 8, 64), "ny": 4 * rng.randint(2, 16), "nx": 64}
    resident = rng.random() < 0.5
    n = [_edge(rng, 32, 512) for _ in range(2)] + [_edge(rng, 1, 400 if resident else 60)]
    case = {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "resident": resident}
    return case if kind == "segment" else {**case, "speckle": rng.random() < 0.3}


# ---------------------------------------------------------------- inputs

def _phantom(case, seed):
    dims, spacing = (case["nx"], case["ny"], case["nz"]), (case["spacing"],) * 3
    if case["phantom"] == "water":
        n = dims[0] * dims[1] * dims[2]
        return phantoms.Phantom(dims, spacing, np.ones(n), np.ones(n, dtype=np.uint8), [phantoms.AIR, phantoms.WATER],
                                ["air", "water"])
    return (phantoms.ct_body if case["phantom"] == "body" else phantoms.ellipsoid)(dims, spacing, seed=seed)


def _beam(name, half_z, histories, seed):
    turn = float(seed % 360)
    if name == "pencil":
        beam = dx.PencilBeam((0.05, 0.05, -2 * half_z - 1.0), (0.0, 0.0, 1.0), 60.0)
    elif name == "dx":
        beam = dx.DXBeam({13: 2.0, 29: 0.1})
        beam.tube.voltage = 80.0
        beam.setCollimation((20.0, 20.0))
        beam.setDAPvalue(100.0)
    elif name == "sequential":
        beam = dx.CTSequentialBeam((0.0, 0.0, 0.0))
        beam.setNumberOfSlices(2)
        beam.setSliceSpacing(3.84)
        beam.setStartAngleDeg(turn)
    elif name == "cbct":
        beam = dx.CBCTBeam()
    else:
        bow = read_filters()[DEFAULT_CT_BOWTIE]
        ends = ((0.0, 0.0, -half_z), (0.0, 0.0, half_z), {13: 6.0})
        if name == "dual":
            beam = dx.CTSpiralDualEnergyBeam(*ends)
            beam.setTubeAVoltage(120.0)
            beam.setTubeBVoltage(120.0)
            beam.setBowtieFilterA(bow)
            beam.setBowtieFilterB(bow)
            beam.setPitch(3.2)
        else:
            beam = dx.CTSpiralBeam(*ends)
            beam.setTubeVoltage(120.0)
            beam.setBowtieFilter(bow)
            beam.setPitch(1.0)
        beam.setCollimation(4.0)
        beam.setStepAngleDeg(5.0)
        beam.setStartAngleDeg(turn)
        beam.setSourceDetectorDistance(119.0)
    beam.setNumberOfParticlesPerExposure(max(1, round(histories / beam.numberOfExposures())))
    return beam


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _smooth(g, shape):
    """A random field of mean 0 that varies over about eight voxels."""
    small = torch.randn((1, 1) + tuple(s // 8 + 2 for s in shape), generator=g, device="cuda")
    return torch.nn.functional.interpolate(small, size=shape, mode="trilinear")[0, 0]


def _features(shape, seed):
    """(nz, ny, nx, 4) features of a low-history body dose and its noiseless
    relative dose and body mask."""
    g = _generator(seed)
    tissue = _smooth(g, shape)
    body = _smooth(g, shape) > -0.8
    density = torch.where(tissue > 1.0, 1.92, torch.where(tissue > -1.0, 1.03, 0.26))
    density = torch.where(body, density, 0.001205)
    clean = torch.exp(0.25 * _smooth(g, shape))
    rel = (0.1 + 0.6 * torch.rand(shape, generator=g, device="cuda")).clamp(max=1.0)
    noisy = (clean * (1.0 + 0.3 * torch.randn(shape, generator=g, device="cuda"))).clamp(min=0.0)
    embed = torch.where(density > 1.5, 1.55, torch.where(body, 1.0, 0.96))
    return torch.stack([noisy, density, embed, rel], dim=-1).float(), clean.float(), body.float()


def _ct_numbers(n, seed):
    """CT numbers of a scan: tissues in runs of 32 voxels, with image noise."""
    g = _generator(seed)
    peak = torch.tensor([-1000.0, -1000.0, -90.0, 40.0, 55.0, 700.0], dtype=torch.float64, device="cuda")
    runs = peak[torch.randint(0, 6, ((n + 31) // 32,), generator=g, device="cuda")]
    return runs.repeat_interleave(32)[:n] + 25.0 * torch.randn(n, generator=g, device="cuda", dtype=torch.float64)


def _organ_volume(n, seed, speckle):
    g = _generator(seed)
    if speckle:
        organ = torch.randint(0, 60, (n,), generator=g, device="cuda", dtype=torch.uint8)
    else:   # 60 organs in runs of 1 to 400 voxels
        runs = torch.randint(1, 401, (n // 100 + 2,), generator=g, device="cuda")
        index = (torch.arange(runs.numel(), device="cuda") % 60).to(torch.uint8)
        organ = torch.repeat_interleave(index, runs)
        organ = organ.repeat(-(-n // organ.numel()))[:n].contiguous()
    dose = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    density = 2.0 * torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    return organ, dose, density


def _voxels(case):
    return case["nx"] * case["ny"] * case["nz"]


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case, "seed": seed}
    if kind == "transport":
        ph = _phantom(case, seed)
        state["world"], state["grid"] = batch_workload.make_world(ph, case["level"])
        state["beam"] = _beam(case["beam"], 0.5 * case["nz"] * case["spacing"], case["histories"], seed)
        state["transport"] = dx.Transport(seed=seed)
    elif kind == "batch":
        inst = batch_workload.instances(case["instances"], seed % 100000, case["scale"], (case["low"], case["high"]))
        state["batch"] = dx.TransportBatch()
        state["grids"] = []
        for ph, beam, s in inst:
            world, grid = batch_workload.make_world(ph)
            state["batch"].add(world, beam, s)
            state["grids"].append(grid)
    elif kind == "infer":
        state["net"] = denoise.Denoiser.pretrained()
        state["features"] = _features((case["nz"], case["ny"], case["nx"]), seed)[0].cpu().numpy()
    elif kind == "apply":
        ph = phantoms.ct_body((case["nx"], case["ny"], case["nz"]), (0.08,) * 3, seed=seed)
        world, grid = batch_workload.make_world(ph)
        beam = _beam("dual", 0.04 * case["nz"], case["per_voxel"] * ph.size, seed)
        dx.Transport(seed=seed)(world, beam, None, True)
        state.update(world=world, grid=grid, net=denoise.Denoiser.pretrained())
    elif kind == "train":
        shape = (case["nz"], case["ny"], case["nx"])
        parts = [_features(shape, 16 * seed + k) for k in range(case["batch"])]
        state["net"] = denoise.Denoiser.pretrained()
        for k, name in enumerate(("features", "target", "mask")):
            state[name] = torch.stack([p[k] for p in parts]).cpu().numpy()
    elif kind == "segment":
        n = _voxels(case)
        hu = _ct_numbers(n, seed)
        state["pipeline"] = pipelines.CTSegmentationPipeline()
        state["tables"] = state["pipeline"].tables()
        if case["resident"]:
            state.update(hu=hu, material=torch.empty(n, dtype=torch.uint8, device="cuda"),
                         density=torch.empty(n, dtype=torch.float64, device="cuda"))
        else:
            state["hu"] = hu.cpu().numpy().reshape(case["nz"], case["ny"], case["nx"])
    elif kind == "organs":
        volume = _organ_volume(_voxels(case), seed, case["speckle"])
        state["volume"] = volume if case["resident"] else tuple(v.cpu().numpy() for v in volume)
    else:
        raise ValueError(f"unknown kind {kind!r}")
    return state


# ---------------------------------------------------------------- one pass

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "transport":
        state["grid"].clearScores()
        state["transport"](state["world"], state["beam"], None, True)
        return state["grid"].doseScored()
    if kind == "batch":
        for grid in state["grids"]:
            grid.clearScores()
        state["batch"].run()
        return [grid.doseScored() for grid in state["grids"]]
    if kind == "infer":
        return state["net"].infer(state["features"])
    if kind == "apply":
        return state["net"].apply(state["grid"])
    if kind == "train":
        loss = state["net"].train_step(state["features"], state["target"], state["mask"], lr=1e-4)
        return {"loss": loss, "grads": state["net"].grads()}
    if kind == "segment":
        if case["resident"]:
            pipelines.segment_device(state["tables"], state["hu"].data_ptr(), state["hu"].numel(),
                                     state["material"].data_ptr(), state["density"].data_ptr())
            return state["material"], state["density"]
        seg = state["pipeline"].updateImageData(state["hu"])
        return seg.material, seg.density
    organ, dose, density = state["volume"]
    if case["resident"]:
        table = pipelines.organ_dose_table_device(organ.data_ptr(), dose.data_ptr(), density.data_ptr(), organ.numel(), SPACING)
    else:
        table = pipelines.organ_dose_table(organ, dose, density, SPACING)
    return {k: table[k] for k in ORGAN_ROW}


# ------------------------------------------------------- what a pass cannot do without

def work(case):
    kind = case["kind"]
    if kind == "transport":
        # per history: a few 5-byte voxel reads and about one 24-byte score;
        # then the dose, its variance and the event count per voxel, and one
        # read of the scores for them
        steps = 0 if case["phantom"] == "water" else 6
        return {"bytes": case["histories"] * (5 * steps + 24 * 1.15) + 48 * _voxels(case), "flops": 600 * case["histories"]}
    if kind == "batch":
        voxels = sum(batch_workload.SHAPES[i % 4][0] * batch_workload.SHAPES[i % 4][1] * batch_workload.SHAPES[i % 4][2]
                     for i in range(case["instances"])) * case["scale"] ** 3
        histories = case["instances"] * (case["high"] - case["low"]) / math.log(case["high"] / case["low"])
        return {"bytes": histories * (5 * 6 + 24 * 1.15) + 48 * voxels, "flops": 600 * histories}
    if kind in ("infer", "apply", "train"):
        n = _voxels(case) * case.get("batch", 1)
        live = 27 * (4 * 32 + 16 * 32 * 32 + 32 * 1)      # multiply-adds per voxel of a forward pass
        if kind == "infer":
            return {"bytes": n * 20, "flops": 2 * live * n}
        if kind == "apply":   # about a third of the grid is body
            return {"bytes": n * (4 + 16 + 8), "flops": 2 * live * n / 3}
        return {"bytes": n * 24, "flops": 3 * 2 * live * n}
    return {"bytes": 17 * _voxels(case), "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind in ("transport", "batch"):
        # Every history has its own random stream and the tally is FP64, so a
        # schedule changes nothing but the order of the sums (3e-16).  Another
        # rounding of the FP32 logarithms, reciprocals and roots sends a few
        # histories elsewhere: 4e-3 of the dose of the largest case and 2e-4 of
        # its event counts were seen to differ, single voxels wholly.
        return {"rel": 1.5e-2, "max": 0.99, "differ": 1e-3}
    if kind in ("infer", "apply"):
        # BF16 activations through 18 layers; the first layer summed in another
        # order: rel 8e-4, max 1e-2 (the network is 4e-3 from FP64)
        return {"rel": 3.5e-3, "max": 5e-2}
    if kind == "train":
        # the same for the gradients, which are 5e-2 from FP64: rel 1.1e-4 and
        # max 3e-3 for the first layer alone, of 18 and their backward passes
        return {"rel": 4e-3, "max": 0.1}
    if kind == "organs":
        return {"rel": 2e-14, "max": 1e-12, "differ": 0.0}      # FP64 sums, 5e-15 from another order
    return "exact"


# ------------------------------------------------------- the same in 64 bits

def _shifted(x, tap):
    """x (n, z, y, x, c) read at the tap's offset, zero outside the volume."""
    d = (tap // 9 - 1, tap // 3 % 3 - 1, tap % 3 - 1)
    out = torch.zeros_like(x)
    dst, src = [], []
    for axis, o in enumerate(d):
        size = x.shape[axis + 1]
        dst.append(slice(max(0, -o), size - max(0, o)))
        src.append(slice(max(0, o), size - max(0, -o)))
    out[(slice(None), *dst)] = x[(slice(None), *src)]
    return out


def _conv(x, w, bias):
    """w: (27, c_in, c_out)."""
    y = bias.expand(*x.shape[:-1], w.shape[2]).clone()
    for tap in range(27):
        y += _shifted(x, tap) @ w[tap]
    return y


def _conv_back(x, w, g, need_x=True):
    dw = torch.stack([_shifted(x, tap).reshape(-1, x.shape[-1]).t() @ g.reshape(-1, g.shape[-1]) for tap in range(27)])
    db = g.reshape(-1, g.shape[-1]).sum(0)
    dx_ = sum(_shifted(g, 26 - tap) @ w[tap].t() for tap in range(27)) if need_x else None
    return dx_, dw, db


def _layers(params):
    """[(weights (27, c_in, c_out), biases)] of the 18 layers from the flat
    parameters ([c_out][tap][c_in] then 32 biases per layer)."""
    out = []
    for p in torch.from_numpy(params).double().cuda().reshape(18, -1):
        out.append((p[:27 * 1024].reshape(32, 27, 32).permute(1, 2, 0).contiguous(), p[27 * 1024:]))
    return out


def _network(layers, f, keep):
    x0 = torch.nn.functional.pad(f, (0, 28))
    a = _conv(x0, *layers[0]).relu_()
    saved = [x0, a]
    for k in range(8):
        h = _conv(a, *layers[2 * k + 1]).relu_()
        a = (_conv(h, *layers[2 * k + 2]) + a).relu_()
        if keep:
            saved += [h, a]
    correction = _conv(a, *layers[17])[..., 0]
    return f[..., 0] + correction, saved


def exact(case, seed):
    kind = case["kind"]
    if kind in ("transport", "batch", "apply"):
        return None      # random histories: there is no value but the engine's own
    state = prepare(case, seed)
    if kind == "infer":
        f = torch.from_numpy(state["features"]).double().cuda()[None]
        return _network(_layers(state["net"].params()), f, False)[0][0].cpu().numpy()
    if kind == "train":
        layers = _layers(state["net"].params())
        f, target, mask = (torch.from_numpy(state[k]).double().cuda() for k in ("features", "target", "mask"))
        pred, saved = _network(layers, f, True)
        count = mask.sum()
        diff = pred - target
        loss = float((mask * diff * diff).sum() / count)
        g = torch.zeros_like(saved[1])
        g[..., 0] = 2.0 * mask * diff / count
        grads = [None] * 18
        acts = saved[1:]      # a0, h0, a1, h1, ..., a8
        g, *grads[17] = _conv_back(acts[16], layers[17][0], g)
        g = g * (acts[16] > 0)
        for k in range(7, -1, -1):
            h, a = acts[2 * k + 1], acts[2 * k]
            gh, *grads[2 * k + 2] = _conv_back(h, layers[2 * k + 2][0], g)
            gh = gh * (h > 0)
            ga, *grads[2 * k + 1] = _conv_back(a, layers[2 * k + 1][0], gh)
            g = (g + ga) * (a > 0)
        _, *grads[0] = _conv_back(saved[0], layers[0][0], g, need_x=False)
        flat = [torch.cat([dw.permute(2, 0, 1).reshape(-1), db]) for dw, db in grads]
        return {"loss": loss, "grads": torch.cat(flat).cpu().numpy()}
    if kind == "segment":
        t = state["tables"]
        hu = torch.as_tensor(state["hu"]).cuda()
        sep = torch.tensor(list(t.separators[:t.n_materials - 1]), dtype=torch.float64, device="cuda")
        att = torch.tensor(list(t.attenuation[:t.n_materials]), dtype=torch.float64, device="cuda")
        material = torch.bucketize(hu, sep, right=True)
        density = ((t.slope * hu / 1000.0 + t.offset) / att[material]).clamp(min=0.0)
        return material.to(torch.uint8).cpu(), density.cpu()
    organ, dose, density = (torch.as_tensor(v).cuda() for v in state["volume"])
    voxel = SPACING[0] * SPACING[1] * SPACING[2]
    index = organ.long()
    count = torch.bincount(index, minlength=256)
    mass = voxel * torch.bincount(index, weights=density, minlength=256)
    energy = torch.bincount(index, weights=dose * (voxel * density), minlength=256)
    table = {"n_voxels": count, "volume_cm3": count.double() * voxel, "mass_g": mass,
             "dose": torch.where(count > 0, energy / mass, torch.zeros_like(mass))}
    return {k: v.cpu().numpy() for k, v in table.items()}
