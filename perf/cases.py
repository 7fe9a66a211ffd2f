"""What is timed: the work a trainer and a viewer have this library do, through its public entry points.

A training loop calls, for every step, the ray sampler (kind "sample"), its network, and the compositing with loss and gradients
followed by the roll-over that fills the batch up (kind "composite"); every sixteen steps it draws grid samples, evaluates its
network's density on them and updates the grid and the bitfield (kind "grid").  A viewer renders frames (kind "frame").  The
network itself is the caller's: its outputs are random tensors here, and a table stands in for it while a frame is rendered.

The scenes are the repository's own workloads: one camera outside a 64^3 grid ("single", workload 1), cameras on a hemisphere
round an object in a 128^3 grid ("object", workload 2), a ring of cameras inside a five-cascade 512 x 256 x 256 grid
("unbounded", workloads 3 to 5), and the same with the outermost cascade occupied nearly throughout ("dense"), which is how a
grid looks while training has not yet carved the empty space out.
"""
import math

import torch

from sphericalrf_amd import api, scene

_WORKLOAD = {"single": 1, "object": 2, "unbounded": 3, "dense": 3}
# on average: samples a training ray makes, the share of rays that make any, composited samples a frame's pixel takes
_MARCHED = {"single": 5.5, "object": 0.3, "unbounded": 15.0, "dense": 1050.0}
_KEPT_RAYS = {"single": 0.65, "object": 0.2, "unbounded": 0.75, "dense": 1.0}
_FRAME = {"single": 4.0, "object": 0.45, "unbounded": 11.5}
_CONSUMED = 0.87      # share of a batch's samples that come before their rays' early termination


def listed():
    return [
        # the first steps of a training: 4096 rays (the reference's initial batch) through a grid that is still full, a
        # thousand samples a ray, Coordinate records for the network
        {"name": "sample_first_steps", "kind": "sample", "scene": "dense", "n_rays": 4096, "target_batch": 1 << 20, "records": True, "masked": False},
        # a step later on: the number of rays has adapted to some fifteen samples a ray and a batch of 2^20 samples
        {"name": "sample_step", "kind": "sample", "scene": "unbounded", "n_rays": 79872, "target_batch": 1 << 20, "records": True, "masked": False},
        # the benchmark's batch: 2^20 rays over 200 cameras, side arrays only
        {"name": "sample_million", "kind": "sample", "scene": "unbounded", "n_rays": 1 << 20, "target_batch": 1 << 20, "records": False, "masked": False},
        # what follows in a training step, half in and half out with the activations of a real network, the records compacted and the
        # batch filled up: an object that few rays hit (the smallest call), the first steps, a step later on ...
        {"name": "composite_object", "kind": "composite", "scene": "object", "n_rays": 50176, "target_batch": 1 << 18, "records": True,
         "half_in": True, "half_out": True, "activations": True, "loss": "SmoothL1"},
        {"name": "composite_first_steps", "kind": "composite", "scene": "dense", "n_rays": 4096, "target_batch": 1 << 20, "records": True,
         "half_in": True, "half_out": True, "activations": True, "loss": "L2"},
        {"name": "composite_step", "kind": "composite", "scene": "unbounded", "n_rays": 79872, "target_batch": 1 << 20, "records": True,
         "half_in": True, "half_out": True, "activations": True, "loss": "L2"},
        # ... and the benchmark's: half in, float gradients out, no activation, room for every sample
        {"name": "composite_million", "kind": "composite", "scene": "unbounded", "n_rays": 1 << 20, "target_batch": 1 << 24, "records": False,
         "half_in": True, "half_out": False, "activations": False, "loss": "L2"},
        # grid maintenance: the smallest grid in its first steps (every point uniform), and the full five-cascade grid in the steady
        # state (a quarter of the cells uniform, a quarter above the threshold)
        {"name": "grid_small_first", "kind": "grid", "size": 64, "cascades": 1, "uniform": 64 ** 3, "nonuniform": 0, "cell_order": False, "half": True},
        {"name": "grid_full_steady", "kind": "grid", "size": 256, "cascades": 5, "uniform": 41943040, "nonuniform": 41943040, "cell_order": False, "half": True},
        # frames: a small preview through the one-launch renderer; an object through the loop with the caller's network in half, then
        # accumulated and tone-mapped for display; a full-size frame
        {"name": "frame_preview", "kind": "frame", "scene": "single", "width": 256, "height": 256, "path": "fused", "half": False, "mode": api.RENDER_SHADE, "display": False},
        {"name": "frame_object_loop", "kind": "frame", "scene": "object", "width": 800, "height": 800, "path": "loop", "half": True, "mode": api.RENDER_SHADE, "display": True},
        {"name": "frame_full", "kind": "frame", "scene": "unbounded", "width": 1920, "height": 1080, "path": "fused", "half": False, "mode": api.RENDER_SHADE, "display": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sample", "composite", "grid", "frame"])
    if kind in ("sample", "composite"):
        where = rng.choice(["single", "object", "unbounded", "dense"])
        # a full grid makes a thousand samples a ray, so a training does not go beyond its first 4096 rays there
        case = {"kind": kind, "scene": where, "n_rays": _log_int(rng, 500, 4096) if where == "dense" else _log_int(rng, 1000, 1 << 20),
                "target_batch": rng.choice([1 << 18, 1 << 20]), "records": rng.random() < 0.6}
        if kind == "sample":
            case["masked"] = rng.random() < 0.3
        else:
            case.update(half_in=rng.random() < 0.8, half_out=rng.random() < 0.5, activations=rng.random() < 0.6, loss=rng.choice(["L2", "SmoothL1", "RelativeL2", "L1"]))
        return case
    if kind == "grid":
        size, cascades = rng.choice([(64, 1), (64, 3), (128, 1), (128, 5), (256, 1), (256, 2), (256, 5)])
        cells = _cells(size) * cascades
        # any number of points from a sixteenth to a quarter of the cells each way, or one a cell in the first steps
        if rng.random() < 0.3 and cells <= 1 << 26:
            uniform, nonuniform = cells - rng.randrange(64), 0
        else:
            uniform, nonuniform = _log_int(rng, cells / 16, cells / 4), _log_int(rng, cells / 16, cells / 4)
        return {"kind": kind, "size": size, "cascades": cascades, "uniform": uniform, "nonuniform": nonuniform, "cell_order": rng.random() < 0.3, "half": rng.random() < 0.8}
    width = _log_int(rng, 64, 1920)
    return {"kind": "frame", "scene": rng.choice(["single", "object", "unbounded"]), "width": width, "height": max(36, int(width * rng.choice([0.5625, 0.75, 1.0]) * (1080 / 1920 if width > 1080 else 1))),
            "path": rng.choice(["fused", "loop", "paced"]), "half": rng.random() < 0.5, "mode": rng.choice([api.RENDER_SHADE, api.RENDER_SHADE, api.RENDER_DEPTH]), "display": rng.random() < 0.5}


# ---- what a program has in hand before it calls -------------------------------------------------
def _cells(size):
    return size ** 3 * (2 if size == 256 else 1)      # the 256 grid is 512 cells round, as in workloads 3 to 5


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _sampler(where, seed):
    """the scene's sampler with its grid and bitfield, blobs placed by the seed; cameras and image size as the workload has them"""
    w = scene.workload(_WORKLOAD[where])
    if where == "dense":
        w = dict(w, shell=(0.05, 1.0, 1.0))
    centres, sigmas = scene.blob_set(**dict(w["blobs"], seed=seed))
    size = w["sampler"]["grid_size"]
    size = (size,) * 3 if isinstance(size, int) else size
    grid = scene.density_grid_from_blobs(size, w["sampler"]["num_cascades"], centres, sigmas, w["occupancy"], w["shell"], seed, device="cuda")
    s = api.OccupancySampler(w["sampler"])
    s.set_density_grid(grid)
    s.update_grid_bitfield()
    torch.cuda.synchronize()      # the caller's grid goes away here
    return s, w


def _prepare_rays(case, seed):
    """everything kind "sample" calls with; kind "composite" starts from what that call leaves"""
    s, w = _sampler(case["scene"], seed)
    g = _generator(seed)
    n, cap = case["n_rays"], min(16 * case["target_batch"], 1 << 24)
    width, height = w["resolution"]
    n_images = len(w["cameras"])
    images = torch.empty((n_images, height, width, 4), dtype=torch.float16, device="cuda").uniform_(generator=g)
    images[..., 3] = 1.0
    probability = None
    if case.get("masked"):
        # the object fills the middle of every picture; most of the border is masked out
        y, x = torch.meshgrid(torch.linspace(-1, 1, height, device="cuda"), torch.linspace(-1, 1, width, device="cuda"), indexing="ij")
        near = (x * x + y * y < 0.5).half()
        probability = torch.maximum(near.expand(n_images, height, width), (torch.rand((n_images, height, width), generator=g, device="cuda") < 0.2).half()).contiguous()
    st = {"case": case, "sampler": s, "cap": cap, "shift": 0, "rng": api.Pcg32(seed)}
    st["dataset"] = api.Dataset(torch.from_numpy(w["cameras"]).cuda(), w["resolution"], w["focal"], (0.5, 0.5), images=images, sampling_probability=probability)
    st["rays"] = torch.zeros((n, 6), device="cuda")
    st["rgba"] = torch.zeros((n, 4), device="cuda")
    st["index"] = torch.zeros((n, 2), dtype=torch.int32, device="cuda")
    st["n_rays"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    st["n_coords"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    st["coords"] = torch.zeros((cap, 7), device="cuda") if case["records"] else None
    for name, kind in (("t", torch.float32), ("dt", torch.float32), ("cell", torch.int32)):
        st[name] = None if case["records"] else torch.zeros(cap, dtype=kind, device="cuda")
    return st, g


def _sample(st):
    n = st["case"]["n_rays"]
    st["n_rays"].zero_()
    st["n_coords"].zero_()
    st["sampler"].sample_coords_from_dataset(n, st["shift"], st["cap"], st["dataset"], st["rays"], st["rgba"], st["n_rays"], st["index"], st["coords"], st["n_coords"],
                                             st["rng"], st["t"], st["dt"], st["cell"])
    st["shift"] += n
    st["rng"].advance()


def _prepare_composite(case, seed):
    rays, g = _prepare_rays(case, seed)
    _sample(rays)
    n, cap, batch = case["n_rays"], rays["cap"], case["target_batch"]
    st = {"case": case, "batch": batch, "rng": rays["rng"], "targets": rays["rgba"], "n_rays": rays["n_rays"], "index_in": rays["index"], "coords": rays["coords"],
          "mean": rays["sampler"].density_grid_mean.clone(), "index": torch.zeros_like(rays["index"])}
    st["dt"] = rays["coords"].view(-1)[3:] if case["records"] else rays["dt"]
    net = torch.randn((cap, 4), generator=g, device="cuda")
    if case["activations"]:
        net[:, 3] = net[:, 3] * 2.0 + 1.0          # the logarithm of a density: a ray through something solid ends after a few samples
    else:
        net[:, :3].uniform_(generator=g)
        net[:, 3] = torch.nn.functional.softplus(net[:, 3])
    st["net"] = net.half() if case["half_in"] else net
    st["gradient"] = torch.zeros((batch, 4), dtype=torch.float16 if case["half_out"] else torch.float32, device="cuda")
    st["compacted"] = torch.zeros((batch, 7), device="cuda") if case["records"] else None
    st["loss"] = torch.zeros(n, device="cuda")
    st["colour"] = torch.zeros((n, 3), device="cuda")
    st["n_compacted"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    st["marcher"] = api.RayMarcher({"train_with_random_bg_color": case["activations"], "train_in_linear_color": not case["activations"], "transmittance_threshold": 1e-4})
    torch.cuda.synchronize()
    return st


def _composite(st):
    case, batch = st["case"], st["batch"]
    st["index"].copy_(st["index_in"])              # the call turns the sampler's records into those of the compacted samples
    st["n_compacted"].zero_()
    st["marcher"].volume_rendering_with_loss_and_gradient(
        case["n_rays"], batch, st["targets"], st["n_rays"], st["index"], st["dt"], st["net"], st["gradient"], st["n_compacted"],
        rgb_activation=api.ACT_LOGISTIC if case["activations"] else api.ACT_NONE, density_activation=api.ACT_EXPONENTIAL if case["activations"] else api.ACT_NONE,
        loss_output=st["loss"], loss_type=case["loss"], loss_scale=128.0, density_grid_mean=st["mean"], use_grid=True, rng=st["rng"],
        coords=st["coords"], compacted_coords=st["compacted"], dt_stride=7 if case["records"] else 1, rgb_ray_out=st["colour"])
    if case["records"]:
        # a network trains on whole batches: what is there is repeated until the batch is full
        api.fill_rollover_and_rescale(batch, 4, st["n_compacted"], st["gradient"])
        api.fill_rollover(batch, st["n_compacted"], st["compacted"])


def _prepare_grid(case, seed):
    size = case["size"]
    s = api.OccupancySampler({"warping_type": "ERP", "aabb_scale": 64, "use_grid": True, "init_grid_with_mask": False, "grid_distribution_type": "WarpedSpace_Exp",
                              "grid_size": (2 * size, size, size) if size == 256 else size, "num_cascades": case["cascades"], "sampling_type": "Disparity",
                              "maximum_marching_steps": 2048 if case["cascades"] > 1 else 1024, "near_distance": 0.05, "far_distance": 100.0})
    s.init(1, (800, 800), (1000.0, 1000.0), (0.5, 0.5), None, None, api.Pcg32(seed))
    s.set_grid_sample_order(case["cell_order"])
    g = _generator(seed)
    n = case["uniform"] + case["nonuniform"]
    cells = _cells(size) * case["cascades"]
    if case["nonuniform"]:
        # a trained grid: most cells well below the threshold of 0.01, a few per cent of them, in clusters of 64, above it
        grid = torch.rand(cells, generator=g, device="cuda") * 0.004
        above = torch.rand(cells // 64, generator=g, device="cuda") < 0.05
        grid.view(-1, 64)[above] += 0.05
        s.set_density_grid(grid)
        s.update_grid_bitfield()
        torch.cuda.synchronize()
    # logarithms of densities as a network gives them: mostly empty space once it is trained, all alike when it is not
    raw = torch.randn(n, generator=g, device="cuda") * (3.0 if case["nonuniform"] else 0.5)
    raw -= 3.0 if case["nonuniform"] else 0.0
    st = {"case": case, "sampler": s, "density": raw.half() if case["half"] else raw, "positions": torch.zeros((n, 3), device="cuda"), "indices": torch.zeros(n, dtype=torch.int32, device="cuda")}
    st["out"] = {k: getattr(s, k) for k in ("density_grid", "density_grid_current", "density_grid_mean", "density_grid_bitfield")}
    torch.cuda.synchronize()
    return st


def _prepare_frame(case, seed):
    s, w = _sampler(case["scene"], seed)
    res = (case["width"], case["height"])
    focal = w["focal"][0] * case["width"] / w["resolution"][0]
    cameras = w["cameras"]
    st = {"case": case, "sampler": s, "resolution": res, "focal": (focal, focal), "camera": [float(v) for v in cameras[seed % len(cameras)]], "spp": 0}
    st["marcher"] = api.RayMarcher({"train_in_linear_color": True, "transmittance_threshold": 1e-4})
    st["field"] = api.Field(torch.from_numpy(scene.field_table(1 << 16, seed % (1 << 31))).cuda(), seed % (1 << 31))
    st["frame"] = torch.zeros((res[1], res[0], 4), device="cuda")
    st["accumulated"] = torch.zeros_like(st["frame"])
    st["shown"] = torch.zeros_like(st["frame"])
    st["samples"] = torch.zeros(res[0] * res[1], dtype=torch.int32, device="cuda") if case["path"] == "fused" else None
    torch.cuda.synchronize()
    return st


def prepare(case, seed):
    kind = case["kind"]
    if kind == "sample":
        st, _ = _prepare_rays(case, seed)
        torch.cuda.synchronize()
        return st
    return {"composite": _prepare_composite, "grid": _prepare_grid, "frame": _prepare_frame}[kind](case, seed)


# ---- one pass -----------------------------------------------------------------------------------
def _present(st, names):
    return {k: st[k] for k in names if st[k] is not None}


def run(state):
    st, case = state, state["case"]
    if case["kind"] == "sample":
        _sample(st)
        return _present(st, ("rays", "rgba", "index", "n_rays", "n_coords", "coords", "t", "dt", "cell"))
    if case["kind"] == "composite":
        _composite(st)
        return _present(st, ("index", "gradient", "compacted", "loss", "colour", "n_compacted"))
    s = st["sampler"]
    if case["kind"] == "grid":
        s.sample_positions_from_grid(case["uniform"], case["nonuniform"], st["positions"], st["indices"])
        s.update_grid(case["uniform"] + case["nonuniform"], 1, st["density"], st["indices"], api.ACT_EXPONENTIAL)
        s.update_grid_bitfield()
        return dict(st["out"], positions=st["positions"], indices=st["indices"])
    args = (st["resolution"], st["focal"], (0.5, 0.5), st["camera"], st["frame"])
    out = {"frame": st["frame"]}
    if case["path"] == "fused":
        s.render_frame_fused(st["marcher"], st["field"], *args, n_samples=st["samples"], spp=st["spp"])
        out["samples"] = st["samples"]
    else:
        out["rounds"] = s.render_frame(st["marcher"], st["field"], *args, spp=st["spp"], render_mode=case["mode"], density_activation=api.ACT_NONE, rgb_activation=api.ACT_NONE,
                                       network_output_dtype=api.DTYPE_F16 if case["half"] else api.DTYPE_F32, paced=case["path"] == "paced")
    if case["display"]:
        api.frame_accumulate(st["resolution"], st["frame"], st["accumulated"], st["spp"])
        api.frame_tonemap(st["resolution"], 0.0, (1.0, 1.0, 1.0, 1.0), st["accumulated"], st["shown"], tonemap_curve=api.TONEMAP_ACES)
        out.update(accumulated=st["accumulated"], shown=st["shown"])
    st["spp"] += 1
    return out


def work(case):
    """bytes every input and output takes once; a sample's warp and the exponentials are some tens of operations each"""
    kind = case["kind"]
    if kind in ("sample", "composite"):
        n, cap = case["n_rays"], min(16 * case["target_batch"], 1 << 24)
        marched = min(cap, _MARCHED[case["scene"]] * n)
        kept = n * _KEPT_RAYS[case["scene"]]
        if kind == "sample":
            # ray, target, (count, offset) out and the target's pixel in; a Coordinate or (t, dt, cell) a sample
            return {"bytes": kept * (24 + 16 + 8 + 8) + marched * (28 if case["records"] else 12), "flops": 100.0 * marched}
        # every consumed sample is read (each ray's colour and count come out whatever there is room for), those with room get gradients
        consumed, batch = _CONSUMED * marched, case["target_batch"]
        written = min(consumed, batch)
        per_in, per_out = (8 if case["half_in"] else 16) + 4, 8 if case["half_out"] else 16
        total = kept * (8 + 16 + 8 + 4 + 12) + consumed * per_in + written * per_out
        if case["records"]:
            # the records of the kept samples, and the rest of the batch filled by repeating gradients and records
            total += written * 24 + batch * 28 + (batch - written) * per_out
        return {"bytes": total, "flops": 60.0 * consumed}
    if kind == "grid":
        n = case["uniform"] + case["nonuniform"]
        cells = _cells(case["size"]) * case["cascades"]
        # positions and indices written, indices and densities read; the grid read and written, the samples' maximum written, a bit a cell
        return {"bytes": n * (12 + 4 + 4 + (2 if case["half"] else 4)) + cells * 12.125, "flops": 60.0 * n}
    pixels = case["width"] * case["height"]
    samples = _FRAME[case["scene"]] * pixels
    total = pixels * (16 + (4 if case["path"] == "fused" else 0) + (64 if case["display"] else 0)) + 16 * samples
    return {"bytes": total, "flops": 150.0 * samples}


def tolerance(case):
    if case["kind"] == "composite" and case["half_out"]:
        return {"rel": 1e-3, "differ": 0.0}
    return {"rel": 1e-5, "differ": 0.0}      # counts, offsets, cells and bits are whole numbers and stay as they are
