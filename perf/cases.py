"""Performance cases: the work a user of plenoxels_amd has it do, through its public entry points.

Five kinds of call:
  step     one fused render + loss-gradient + backward pass over a batch of camera rays
           (train_step, the zero-fill or corner-block reduce it needs, and the loss value)
  trainer  one Trainer.step of the whole training loop (pooling, rays, render, loss, TV, Adam)
  view     one forward-only image (render_camera)
  rays     render_rays forward and backward through autograd, explicit rays
  dropin   the reference's own function-by-function chain on the drop-ins, forward and backward

listed() holds fixed sizes (the benchmark workloads, the reference CLI's defaults, the 512^3
training configuration, and ragged ones); draw() gives further sizes of the same ranges.
"""
import math

import numpy as np
import torch
import torch.nn.functional as F

from plenoxels_amd import (CameraRays, CornerBlockPair, LossMean, MarchConfig, fill_, fill_reachable_,
                           occupancy_dilate, pack_occupancy, render_rays, train_step)
from plenoxels_amd.grid_functions import generate_grid, get_nearest_voxels
from plenoxels_amd.optim import tv_loss
from plenoxels_amd.ray_sampling import (compute_alpha_weighted_pixels, normalize_samples_for_indecies,
                                        sample_camera_rays_batched)
from plenoxels_amd.render import render_camera
from plenoxels_amd.train import Trainer

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
THETA = 800 / 1111  # focal 1111 px on 800 px wide images
ADAM_STEPS = 300    # a Trainer state in the middle of a run: steps its moments have seen


# --------------------------------------------------------------------------- the cases

def _step(name, dims, rays, samples, interp, dtype, scene, cams, res, t_stop):
    return {"name": name, "kind": "step", "X": dims[0], "Y": dims[1], "Z": dims[2], "rays": rays, "samples": samples,
            "interp": interp, "dtype": dtype, "scene": scene, "cams": cams, "res": res, "t_stop": t_stop}


def _trainer(name, dims, rays_per_cam, total_rays, samples, interp, dtype, cams, res, step, lr, tv, beta, near, pd,
             delta, t_stop):
    return {"name": name, "kind": "trainer", "X": dims[0], "Y": dims[1], "Z": dims[2], "rays_per_cam": rays_per_cam,
            "total_rays": total_rays, "samples": samples, "interp": interp, "dtype": dtype, "cams": cams, "res": res,
            "step": step, "lr": lr, "tv": tv, "beta": beta, "near": near, "pd": pd, "delta": delta, "t_stop": t_stop}


def listed():
    return [
        # the smallest call: a few hundred rays through a coarse grid inside a user's own autograd
        # loop, where launches and host work are what is paid for
        {"name": "rays_small", "kind": "rays", "X": 64, "Y": 64, "Z": 64, "rays": 512, "samples": 100,
         "interp": "nearest", "scene": "dense", "t_stop": 0.0},
        # autograd through the fused render at an ordinary size: odd ray count, non-cubic grid
        {"name": "rays_trilinear", "kind": "rays", "X": 160, "Y": 128, "Z": 145, "rays": 65537, "samples": 192,
         "interp": "trilinear", "scene": "dense", "t_stop": 0.0},
        # 64^3 blob field, 8 views' worth of rays: an early, coarse, dense grid
        _step("step_blobs64", (64, 64, 64), 32768, 128, "trilinear", "f32", "dense", 8, 64, 0.0),
        # 256^3, ~5% occupied, 2^18 random rays of 100 views: the benchmark's own step
        _step("step_sparse256_trilinear", (256, 256, 256), 1 << 18, 256, "trilinear", "f32", "sparse", 100, 800, 1e-4),
        # the same batch with the reference's own lookup
        _step("step_sparse256_nearest", (256, 256, 256), 1 << 18, 256, "nearest", "f32", "sparse", 100, 800, 1e-4),
        # ragged: non-cubic grid, odd ray count, sample count between chunk sizes, half storage
        _step("step_ragged_bf16", (201, 173, 190), 100003, 300, "trilinear", "bf16", "sparse", 37, 500, 1e-4),
        # every pixel of one 800x800 view against a dense grid: neighbouring rays share cells
        _step("step_view800_nearest", (128, 128, 128), 640000, 256, "nearest", "f32", "dense", 1, 800, 0.0),
        # the reference CLI's defaults (256^3, 128 rays of each of 100 views, 600 samples, TV and
        # beta), past and during progressive growing
        _trainer("trainer_default_full", (256, 256, 256), 128, 0, 600, "nearest", "f32", 100, 800, 230, 0.0075, 1e-5,
                 5e-3, 0.0, 0.0125, 0.0125, 0.0),
        _trainer("trainer_default_pooled", (256, 256, 256), 128, 0, 600, "nearest", "f32", 100, 800, 170, 0.0075, 1e-5,
                 5e-3, 0.0, 0.0125, 0.0125, 0.0),
        # the 512^3 training configuration: BF16 storage, FP32 Adam state, 2^19 rays, 512 samples
        _trainer("trainer_512_bf16", (512, 512, 512), 0, 1 << 19, 512, "trilinear", "bf16", 100, 800, 230, 0.1, 1e-5,
                 0.0, 2.0, 3 / 511, 4 / 512, 1e-4),
        # one 800x800 image of a trained grid kept in half storage
        {"name": "view_800", "kind": "view", "X": 256, "Y": 256, "Z": 256, "res": 800, "samples": 256,
         "interp": "trilinear", "dtype": "f16", "scene": "sparse", "t_stop": 1e-4},
        # the reference's loop with only its imports switched: 121 even-spread rays of 100 views
        {"name": "dropin_default", "kind": "dropin", "X": 256, "Y": 256, "Z": 256, "cams": 100, "rays_per_cam": 121,
         "samples": 600, "res": 800, "tv": 1e-5, "delta": 0.0125, "pd": 0.0125},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dims(rng, lo, hi):
    base = _log_int(rng, lo, hi)
    return [max(lo, min(hi, int(base * rng.uniform(0.75, 1.25)))) for _ in range(3)]


def draw(rng):
    kind = rng.choice(["step", "step", "trainer", "view", "rays", "dropin"])
    interp = rng.choice(["nearest", "trilinear"])
    if kind == "step":
        X, Y, Z = _dims(rng, 32, 256)
        scene = rng.choice(["dense", "sparse"])
        samples = _log_int(rng, 48, 700)
        most = (1 << 26) if scene == "sparse" else (1 << 24)  # samples placed
        rays = _log_int(rng, 2000, min(1 << 18, most // samples))
        c = _step("", (X, Y, Z), rays, samples, interp, rng.choice(["f32", "f32", "bf16", "f16"]), scene,
                  rng.randint(1, 100), _log_int(rng, 64, 800), rng.choice([0.0, 1e-4]))
        del c["name"]
        return c
    if kind == "trainer":
        X, Y, Z = _dims(rng, 96, 300)
        pooled = rng.random() < 0.5
        # steps 170..229: receptive fields 25..3
        step = rng.randint(170, 229) if pooled else rng.randint(230, 400)
        beta = rng.choice([0.0, 5e-3])
        c = _trainer("", (X, Y, Z), rng.randint(40, 400), 0, rng.randint(200, 640), interp,
                     rng.choice(["f32", "bf16"]), rng.randint(20, 100), _log_int(rng, 100, 800), step, 0.0075,
                     rng.choice([0.0, 1e-5]), beta, 2.0, 3.0 / X, 4.0 / 512, 0.0 if beta > 0 else 1e-4)
        del c["name"]
        return c
    if kind == "view":
        X, Y, Z = _dims(rng, 48, 300)
        return {"kind": "view", "X": X, "Y": Y, "Z": Z, "res": _log_int(rng, 64, 800), "samples": _log_int(rng, 64, 512),
                "interp": interp, "dtype": rng.choice(["f32", "bf16", "f16"]), "scene": rng.choice(["dense", "sparse"]),
                "t_stop": rng.choice([0.0, 1e-4])}
    if kind == "rays":
        X, Y, Z = _dims(rng, 32, 200)
        samples = _log_int(rng, 40, 700)
        return {"kind": "rays", "X": X, "Y": Y, "Z": Z, "rays": _log_int(rng, 256, min(1 << 17, (1 << 24) // samples)),
                "samples": samples, "interp": interp, "scene": rng.choice(["dense", "sparse"]),
                "t_stop": rng.choice([0.0, 1e-4])}
    X, Y, Z = _dims(rng, 48, 256)
    cams, samples = rng.randint(4, 100), rng.randint(100, 600)
    side = rng.randint(3, max(3, min(16, int(math.sqrt(8e6 / (cams * samples))))))
    return {"kind": "dropin", "X": X, "Y": Y, "Z": Z, "cams": cams, "rays_per_cam": side * side, "samples": samples,
            "res": _log_int(rng, 64, 800), "tv": rng.choice([0.0, 1e-5]), "delta": 7.0 / 600, "pd": 3.2 / X}


# --------------------------------------------------------------------------- inputs

def _gen(seed, which):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 16 + which)


def _axis(n, pd):
    """World coordinates of an axis' cells, and the first one's float32 value as the layout rounds it."""
    return (torch.arange(n, device="cuda", dtype=torch.float32) - math.ceil(n / 2) + 1) * pd


def _coord(i, n, pd):
    c = np.float32(i) - np.float32(math.ceil(n / 2)) + np.float32(1)
    return float(np.float32(c * np.float32(pd)))


def _density(dims, pd, seed, peak):
    """Sum of six Gaussian blobs (centres in [-1, 1]^3, sigma 0.1 to 0.3) at the cells."""
    g = np.random.default_rng(seed)
    ax = [_axis(n, pd) for n in dims]
    out = torch.zeros(dims, device="cuda")
    for _ in range(6):
        mu, sig = g.uniform(-1, 1, 3), g.uniform(0.1, 0.3)
        e = [torch.exp(-(ax[a] - float(mu[a])) ** 2 / (2 * sig * sig)) for a in range(3)]
        out += peak * (e[0][:, None, None] * e[1][None, :, None] * e[2][None, None, :])
    return out


def _occupied(dims, seed):
    """~5% of the cells, in clumps: value noise on a lattice of one point per 8 cells, thresholded."""
    lat = [max(3, n // 8) for n in dims]
    noise = torch.rand(1, 1, *lat, device="cuda", generator=_gen(seed, 1))
    up = F.interpolate(noise, size=tuple(dims), mode="trilinear", align_corners=True)[0, 0]
    return up > torch.quantile(up.reshape(-1)[:: max(1, up.numel() // 1_000_000)], 0.95)


def _cells_read(occ, interp):
    """Cells whose samples count: the occupied ones, for trilinear those with an occupied corner."""
    if interp == "nearest":
        return occ
    any_ = occ
    for axis in range(3):
        any_ = any_ | any_.roll(-1, axis)
    return any_


def _scene(case, seed):
    """(raw grid (X,Y,Z,4) float32, occupied cells or None, points distance)."""
    dims = (case["X"], case["Y"], case["Z"])
    pd = 3.0 / (max(dims) - 1)
    grid = torch.empty(*dims, 4, device="cuda")
    grid[..., :3] = torch.rand(*dims, 3, device="cuda", generator=_gen(seed, 0))
    grid[..., 3] = _density(dims, pd, seed, 20.0)
    occ = None
    if case["scene"] == "sparse":
        occ = _occupied(dims, seed)
        grid[..., 3] *= occ
    return grid, occ, pd


def _cameras(n, seed):
    """n camera-to-world matrices on the upper hemisphere of radius 4, looking at the origin."""
    g = np.random.default_rng(seed)
    mats = np.tile(np.eye(4), (n, 1, 1))
    for m in mats:
        z = g.normal(size=3)
        z[2] = abs(z[2]) + 0.05
        z /= np.linalg.norm(z)
        x = np.cross([0.0, 0.0, 1.0], z) if abs(z[2]) < 0.999 else np.array([1.0, 0.0, 0.0])
        x /= np.linalg.norm(x)
        m[:3, 0], m[:3, 1], m[:3, 2], m[:3, 3] = x, np.cross(z, x), z, 4 * z
    return torch.from_numpy(mats.astype(np.float32)).to("cuda")


def _even_uv(side):
    ls = torch.linspace(0, end=1, steps=side, device="cuda")
    return torch.cartesian_prod(ls, ls)


def _ray_batch(case, seed, n):
    """(cam_ids, uv) of n rays: every pixel of the view for a single camera (whole images), else
    random cameras and pixels."""
    side = int(round(math.sqrt(n)))
    if case["cams"] == 1 and side * side == n:
        return torch.zeros(n, dtype=torch.int32, device="cuda"), _even_uv(side).contiguous()
    g = _gen(seed, 2)
    cam = torch.randint(0, case["cams"], (n,), device="cuda", generator=g, dtype=torch.int64).to(torch.int32)
    return cam, torch.rand(n, 2, device="cuda", generator=g)


def _images(case, seed):
    return torch.rand(case["cams"], case["res"], case["res"], 4, device="cuda", generator=_gen(seed, 3))


def _trained_grid(dims, pd, seed):
    """A grid in training: blobs of density over a slightly negative floor, colours around [0, 1]."""
    grid = torch.empty(*dims, 4, device="cuda")
    grid[..., :3] = torch.rand(*dims, 3, device="cuda", generator=_gen(seed, 0)) * 1.2 - 0.1
    grid[..., 3] = _density(dims, pd, seed, 1.0).clamp_max(1.0) - 0.02
    return grid


def _inputs(case, seed):
    """Everything a case computes from, made from the seed alone."""
    kind, dims = case["kind"], (case["X"], case["Y"], case["Z"])
    s = {}
    if kind in ("step", "rays", "view"):
        grid, occ, pd = _scene(case, seed)
        s.update(grid=grid if kind == "rays" else grid.to(DTYPES[case["dtype"]]), occ=occ, pd=pd, near=2.0,
                 delta=4.0 / case["samples"])
    else:
        grid = _trained_grid(dims, case["pd"], seed)
        if kind == "trainer":  # exact in half storage, so that the copy it renders from is the same grid
            grid = grid.to(DTYPES[case["dtype"]]).float()
        s.update(grid=grid, occ=None, pd=case["pd"], near=case.get("near", 0.0), delta=case["delta"])
    s["gmin"] = tuple(_coord(0, n, s["pd"]) for n in dims)
    if kind == "step":
        s["c2w"], s["imgs"] = _cameras(case["cams"], seed), _images(case, seed)
        s["cam_ids"], s["uv"] = _ray_batch(case, seed, case["rays"])
    elif kind == "view":
        s["c2w"], n = _cameras(1, seed), case["res"] ** 2
        s["cam_ids"], s["uv"] = torch.zeros(n, dtype=torch.int32, device="cuda"), _even_uv(case["res"]).contiguous()
    elif kind == "rays":
        cam, uv = _ray_batch({"cams": 16}, seed, case["rays"])
        s["o"], s["d"] = _camera_rays(_cameras(16, seed), cam, uv)
        s["targets"] = torch.rand(case["rays"], 4, device="cuda", generator=_gen(seed, 3))
    elif kind == "dropin":
        s["c2w"], s["imgs"] = _cameras(case["cams"], seed), _images(case, seed)
        n = int(round(math.sqrt(case["rays_per_cam"])))
        s["uv"] = _even_uv(n).repeat(case["cams"], 1)
        s["cam_ids"] = torch.repeat_interleave(torch.arange(case["cams"], dtype=torch.int32, device="cuda"), n * n)
    else:
        s["c2w"], s["imgs"] = _cameras(case["cams"], seed), _images(case, seed)
        if case["total_rays"]:
            s["cam_ids"], s["uv"] = _ray_batch(case, seed, case["total_rays"])
        else:
            B, R = case["cams"], case["rays_per_cam"]
            s["cam_ids"] = torch.repeat_interleave(torch.arange(B, dtype=torch.int32, device="cuda"), R)
            s["uv"] = torch.rand(B * R, 2, device="cuda", generator=_gen(seed, 2))
        # moments that dwarf a single step's, as late in a run: the grid barely moves from pass to pass
        g = _gen(seed, 4)
        s["exp_avg"] = torch.randn(s["grid"].shape, device="cuda", generator=g) * 1e-4
        s["exp_avg_sq"] = torch.rand(s["grid"].shape, device="cuda", generator=g) * 1e-4 + 1e-5
    return s


# --------------------------------------------------------------------------- state and one pass

def _march(case, s, samples):
    return MarchConfig(samples, s["delta"], s["gmin"], s["pd"], case["interp"], s["near"], case["t_stop"])


def _occupancy_bits(s, case):
    if s["occ"] is None:
        return None
    bits = pack_occupancy(s["occ"])
    return occupancy_dilate(bits, (case["X"], case["Y"], case["Z"])) if case["interp"] == "trilinear" else bits


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    st = {"case": case}
    if kind == "step":
        st["cfg"], st["grid"], st["bits"] = _march(case, s, case["samples"]), s["grid"], _occupancy_bits(s, case)
        st["camera"] = CameraRays(s["cam_ids"], s["uv"], s["c2w"], THETA, s["imgs"])
        st["grad"] = torch.zeros(s["grid"].shape, device="cuda")
        st["sq"] = torch.empty(case["rays"], device="cuda")
        st["loss_mean"] = LossMean(torch.device("cuda"))
        st["pair"] = CornerBlockPair(s["grid"]) if case["interp"] == "trilinear" else None
    elif kind == "trainer":
        n, B = s["uv"].shape[0], case["cams"]
        rays = (s["cam_ids"], s["uv"]) if case["total_rays"] else s["uv"].reshape(B, n // B, 2)
        tr = Trainer(s["imgs"], s["c2w"], THETA, gridsize=(case["X"], case["Y"], case["Z"]), points_distance=case["pd"],
                     number_of_rays=case["rays_per_cam"] or 1, num_samples=case["samples"], delta_step=case["delta"],
                     lr=case["lr"], tv=case["tv"], beta=case["beta"], interp=case["interp"],
                     storage_dtype=DTYPES[case["dtype"]], uniforms_fn=lambda i: rays, init_grid=s["grid"],
                     near=case["near"], t_stop=case["t_stop"], total_rays=case["total_rays"] or None)
        tr.exp_avg.copy_(s["exp_avg"])
        tr.exp_avg_sq.copy_(s["exp_avg_sq"])
        tr.step_count = ADAM_STEPS
        st["trainer"] = tr
    elif kind == "view":
        st["cfg"], st["grid"], st["bits"] = _march(case, s, case["samples"]), s["grid"], _occupancy_bits(s, case)
        st["camera"] = CameraRays(s["cam_ids"], s["uv"], s["c2w"], THETA)
    elif kind == "rays":
        st.update(o=s["o"], d=s["d"], targets=s["targets"], leaf=s["grid"].requires_grad_(True),
                  kw=dict(num_samples=case["samples"], delta_step=s["delta"], grid_min=s["gmin"],
                          points_distance=s["pd"], interp=case["interp"], near=s["near"], t_stop=case["t_stop"],
                          occupancy=_occupancy_bits(s, case)))
    else:
        st.update(imgs=s["imgs"], c2w=s["c2w"], leaf=s["grid"].requires_grad_(True),
                  grid_indices=generate_grid(case["X"], case["Y"], case["Z"], points_distance=case["pd"])[0])
    return st


def _run_step(st):
    grid, grad, bits, sq, pair = st["grid"], st["grad"], st["bits"], st["sq"], st["pair"]
    if pair is not None:
        train_step(grid, grad, cfg=st["cfg"], camera=st["camera"], occupancy=bits, ray_sq_err=sq, blocks=pair.blocks,
                   clear=pair.other, overwrite=True if bits is None else "reachable")
        pair.flip()
    else:
        if bits is None:
            fill_(grad, 0.0)
        else:
            fill_reachable_(grad, bits, st["cfg"].interp)
        train_step(grid, grad, cfg=st["cfg"], camera=st["camera"], occupancy=bits, ray_sq_err=sq)
    return {"loss": st["loss_mean"](sq), "sq_err": sq, "grad": grad}


def _run_dropin(st):
    c, leaf = st["case"], st["leaf"]
    samples, pixels, _, _ = sample_camera_rays_batched(
        transform_matrices=st["c2w"], camera_angle_x=THETA, imgs=st["imgs"], number_of_rays=c["rays_per_cam"],
        num_samples=c["samples"], delta_step=c["delta"], even_spread=True, camera_ray=False, device="cuda")
    n = normalize_samples_for_indecies(st["grid_indices"], samples, c["pd"])
    values, mask = get_nearest_voxels(n, leaf.clip(0, 1))
    values = (values * mask.unsqueeze(-1)).reshape(c["cams"], c["rays_per_cam"], c["samples"], 4)
    rgba = compute_alpha_weighted_pixels(values).reshape(-1, 4)
    loss = F.mse_loss(rgba, pixels)
    if c["tv"] > 0:
        loss = loss + c["tv"] * tv_loss(leaf)
    leaf.grad = None
    loss.backward()
    return {"rgba": rgba.detach(), "loss": loss.detach(), "grad": leaf.grad}


def run(st):
    kind = st["case"]["kind"]
    if kind == "step":
        return _run_step(st)
    if kind == "trainer":
        tr = st["trainer"]
        out = tr.step(st["case"]["step"])
        return {**out, "grid": tr.grid, "exp_avg": tr.exp_avg, "exp_avg_sq": tr.exp_avg_sq, "grad_abs": tr.grad_abs}
    if kind == "view":
        return render_camera(st["grid"], st["camera"], st["cfg"], occupancy=st["bits"])
    if kind == "rays":
        leaf = st["leaf"]
        rgba = render_rays(leaf, st["o"], st["d"], **st["kw"])
        leaf.grad = None
        F.mse_loss(rgba, st["targets"]).backward()
        return {"rgba": rgba.detach(), "grad": leaf.grad}
    return _run_dropin(st)


# --------------------------------------------------------------------------- what a pass cannot do without

def _receptive_field(i):
    fields = list(range(93, 2, -2))
    return fields[i // 5] if i // 5 < len(fields) else 0


def work(case):
    kind, cells = case["kind"], case["X"] * case["Y"] * case["Z"]
    tri = case.get("interp") == "trilinear"
    size = 2 if case.get("dtype") in ("bf16", "f16") and kind != "rays" else 4
    rays = case.get("rays") or case.get("total_rays") or case.get("cams", 1) * case.get("rays_per_cam", 0)
    rays = case["res"] ** 2 if kind == "view" else rays
    placed = rays * case["samples"]
    # samples whose values are read, and cells they can lie in: ~6% of the placed samples and ~5%
    # of the cells (~10% with an occupied corner) in a sparse scene, two thirds and all in a dense one
    sparse = case.get("scene") == "sparse"
    kept = placed * (0.06 if sparse else 0.6)
    touched = min(cells * ((0.1 if tri else 0.05) if sparse else 1.0), kept * (8 if tri else 1))
    flops = placed * 25 + kept * (150 if tri else 40)
    if kind == "view":
        return {"bytes": touched * 4 * size + rays * (12 + 16), "flops": flops}
    if kind == "rays":  # rays, targets and RGBA; the dense gradient autograd returns
        return {"bytes": touched * 16 + rays * (24 + 16 + 16) + cells * 16, "flops": flops + kept * (100 if tri else 50)}
    if kind == "step":  # camera index, uniforms, target pixel and squared error per ray
        return {"bytes": touched * (4 * size + 16) + rays * (12 + 16 + 4), "flops": flops + kept * (100 if tri else 50)}
    if kind == "dropin":  # grid, its gradient and the coordinates whose minimum is taken; rays in and out
        return {"bytes": cells * (16 + 16 + 12) + rays * (16 + 16), "flops": placed * 100 + cells * 30}
    # trainer: parameter, moments and |grad| sums read and written, the half copy written
    pooled = _receptive_field(case["step"]) > 1
    adam = cells * (4 * 32 + (8 if size == 2 else 0))
    return {"bytes": adam + rays * (12 + 16),
            "flops": cells * 60 + (placed * 40 if not pooled else placed * 60)}


def tolerance(case):
    """float32 arithmetic with its sums in another order (float atomics): up to 3e-7 in the 2-norm
    was measured against exact() and 1e-7 between runs.  A ray whose transmittance lands within
    rounding of t_stop may keep or drop one more sample, which moves that ray by up to t_stop."""
    if case.get("t_stop"):
        return {"rel": 3e-6, "max": 4 * case["t_stop"]}
    return {"rel": 1.2e-6}


# --------------------------------------------------------------------------- 64-bit evaluation

def _camera_rays(c2w, cam_ids, uv):
    """float32 ray origins and directions of camera-form rays."""
    def norm(v):
        return torch.sqrt((v[..., 0] * v[..., 0] + v[..., 2] * v[..., 2]) + v[..., 1] * v[..., 1])
    cam = cam_ids.long()
    x, y, z = c2w[:, :3, 0], c2w[:, :3, 1], -c2w[:, :3, 2]
    aspect = norm(x) / norm(y)
    us = THETA * (uv[:, 0] - 0.5)
    vs = -((THETA * (1 / aspect))[cam] * (uv[:, 1] - 0.5))
    d = us.unsqueeze(-1) * x[cam] + vs.unsqueeze(-1) * y[cam] + z[cam]
    d = d / norm(d).unsqueeze(-1)
    return c2w[cam, :3, 3].contiguous(), d.contiguous()


def _targets(imgs, cam_ids, uv):
    H, W = imgs.shape[1], imgs.shape[2]
    col = (H * uv[:, 0]).round().clamp(max=H - 1).long()
    row = (W * uv[:, 1]).round().clamp(max=W - 1).long()
    return imgs[cam_ids.long(), row, col]


def _indices(o, d, S, delta, near, gmin, pd):
    """float32 continuous cell coordinates (R,S,3) of the samples, each operation rounded to float32."""
    k = torch.arange(1, S + 1, device="cuda", dtype=torch.float32)
    t = k * float(np.float32(delta)) + float(np.float32(near))
    p = o[:, None, :] + d[:, None, :] * t[None, :, None]
    inv = float(np.float32(1.0) / np.float32(pd))
    return (p - torch.tensor(gmin, device="cuda")) * inv


EPS = 1e-4


def _chain64(grid, reads, o, d, seed_grad, S, delta, near, gmin, pd, interp, t_stop, beta_scale=0.0, grad=True):
    """The render chain in float64 on float32 sample placement: (rgba (R,4), per-ray beta sums,
    d loss / d grid).  grid (X,Y,Z,4) float64 raw; reads: cells whose samples count (None: all);
    seed_grad(rgba, slice) = d loss / d rgba."""
    dims = grid.shape[:3]
    flat = grid.reshape(-1, 4)
    X, Y, Z = dims
    G = torch.zeros_like(flat) if grad else None
    lim = torch.tensor(dims, device="cuda", dtype=torch.float32)
    rgba, bsum = [], []
    f = (lambda a: torch.log(a + EPS) - torch.log(1 - a + EPS))
    f0 = math.log(EPS) - math.log(1 + EPS)
    step = max(1, (1 << 22) // S)
    for r0 in range(0, o.shape[0], step):
        sl = slice(r0, min(o.shape[0], r0 + step))
        n = _indices(o[sl], d[sl], S, delta, near, gmin, pd)
        base = n.round() if interp == "nearest" else n.floor()
        at = base if interp == "nearest" else n
        keep = ((at >= 0) & (at < lim)).all(-1)
        if reads is not None:
            c = base[keep].long()
            keep[keep.clone()] = reads[c[:, 0], c[:, 1], c[:, 2]]
        n = n[keep]
        if interp == "nearest":
            c = n.round().long()
            cells = ((c[:, 0] * Y + c[:, 1]) * Z + c[:, 2]).unsqueeze(1)
            w = torch.ones(1, 1, device="cuda", dtype=torch.float64)
        else:
            fr = (n - n.trunc()).double()
            hi, lo = n.ceil().long() % torch.tensor(dims, device="cuda"), n.floor().long()
            cells, w = [], []
            for bx in (0, 1):
                for by in (0, 1):
                    for bz in (0, 1):
                        b = (bx, by, bz)
                        i = [(hi if b[a] == 0 else lo)[:, a] for a in range(3)]
                        cells.append((i[0] * Y + i[1]) * Z + i[2])
                        q = [fr[:, a] if b[a] == 0 else 1 - fr[:, a] for a in range(3)]
                        w.append(q[0] * q[1] * q[2])
            cells, w = torch.stack(cells, 1), torch.stack(w, 1)
        raw = flat[cells]  # (n, corners, 4)
        v = torch.zeros(*keep.shape, 4, device="cuda", dtype=torch.float64)
        v[keep] = (w.unsqueeze(-1) * raw.clamp(0, 1)).sum(1)
        a = v[..., 3]
        T = torch.cat([torch.ones_like(a[:, :1]), torch.cumprod(1 - a, 1)[:, :-1]], 1)
        proc = keep if t_stop <= 0 else keep & (T >= t_stop)
        colour = torch.cat([v[..., :3], torch.ones_like(v[..., :1])], -1)
        out = (colour * (a * T * proc).unsqueeze(-1)).sum(1)
        rgba.append(out)
        if beta_scale:
            bsum.append(((f(a) - f0) * proc).sum(1))
        if not grad:
            continue
        g = seed_grad(out, sl)
        gv = torch.zeros_like(v)
        Q = torch.zeros_like(out)
        am = a * proc
        for k in range(S - 1, -1, -1):
            ak = am[:, k].unsqueeze(-1)
            gv[:, k, 3] = ((colour[:, k] - Q) * g).sum(-1)
            Q = ak * colour[:, k] + (1 - ak) * Q
        gv[..., 3] *= T
        gv[..., :3] = (am * T).unsqueeze(-1) * g[:, None, :3]
        if beta_scale:
            gv[..., 3] += beta_scale * (1 / (a + EPS) + 1 / (1 - a + EPS))
        gv = gv * proc.unsqueeze(-1)
        inside = (raw >= 0) & (raw <= 1)
        G.index_add_(0, cells.reshape(-1), (gv[keep].unsqueeze(1) * w.unsqueeze(-1) * inside).reshape(-1, 4))
    return torch.cat(rgba), torch.cat(bsum) if bsum else None, G.reshape(grid.shape) if grad else None


def _tv64(grid):
    """(sqrt of the squared neighbour differences' sum, its gradient) in float64."""
    total, g = 0.0, torch.zeros_like(grid)
    for axis in range(3):
        n = grid.shape[axis]
        diff = grid.narrow(axis, 1, n - 1) - grid.narrow(axis, 0, n - 1)
        total = total + (diff * diff).sum()
        g.narrow(axis, 1, n - 1).add_(diff)
        g.narrow(axis, 0, n - 1).sub_(diff)
    tv = torch.sqrt(total)
    return tv, g / tv


def _mse_seed(targets):
    scale = 2.0 / (4.0 * targets.shape[0])
    return lambda rgba, sl: scale * (rgba - targets[sl])


def _trainer64(case, s):
    k = _receptive_field(case["step"])
    gmin, pd, grid = s["gmin"], s["pd"], s["grid"].double()
    full = grid
    if k > 1:
        stride = max(1, k // 4)
        grid = F.avg_pool3d(grid.permute(3, 0, 1, 2).unsqueeze(0), k, stride)[0].permute(1, 2, 3, 0).contiguous()
        gmin = tuple(_coord(k // 2, n, pd) for n in full.shape[:3])
        pd = pd * stride
    o, d = _camera_rays(s["c2w"], s["cam_ids"], s["uv"])
    tgt = _targets(s["imgs"], s["cam_ids"], s["uv"]).double()
    n_s = o.shape[0] * case["samples"]
    beta = case["beta"] / n_s
    # a sample whose cells all have a negative alpha is zero and gets no gradient
    reads = _cells_read(grid[..., 3] >= 0, case["interp"])
    rgba, bsum, G = _chain64(grid, reads, o, d, _mse_seed(tgt), case["samples"], s["delta"], s["near"], gmin, pd,
                             case["interp"], case["t_stop"], beta)
    out = {"closs": ((rgba - tgt) ** 2).mean()}
    out["loss"] = out["closs"]
    if case["tv"] > 0 and k < 19:
        tv, g = _tv64(grid)
        G += case["tv"] * g
        out["tvloss"] = case["tv"] * tv
        out["loss"] = out["loss"] + out["tvloss"]
    if case["beta"] > 0:
        f0 = math.log(EPS) - math.log(1 + EPS)
        out["betaloss"] = case["beta"] * (bsum.sum() + n_s * f0) / n_s
        out["loss"] = out["loss"] + out["betaloss"]
    if k > 1:
        p = full.permute(3, 0, 1, 2).unsqueeze(0).detach().requires_grad_(True)
        F.avg_pool3d(p, k, stride).backward(G.permute(3, 0, 1, 2).unsqueeze(0))
        G = p.grad[0].permute(1, 2, 3, 0)
    t = ADAM_STEPS + 1
    m = 0.9 * s["exp_avg"].double() + 0.1 * G
    v = 0.999 * s["exp_avg_sq"].double() + 0.001 * G * G
    out["grad_abs"] = G.abs()
    out["grid"] = full - case["lr"] / (1 - 0.9 ** t) * m / (torch.sqrt(v) / math.sqrt(1 - 0.999 ** t) + 1e-8)
    out["exp_avg"], out["exp_avg_sq"] = m, v
    return out


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "trainer":
        return _trainer64(case, s)
    S = case["samples"]
    if kind == "dropin":
        grid = s["grid"].double()
        o, d = _camera_rays(s["c2w"], s["cam_ids"], s["uv"])
        tgt = _targets(s["imgs"], s["cam_ids"], s["uv"]).double()
        rgba, _, G = _chain64(grid, None, o, d, _mse_seed(tgt), S, s["delta"], 0.0, s["gmin"], s["pd"], "nearest", 0.0)
        loss = ((rgba - tgt) ** 2).mean()
        if case["tv"] > 0:
            tv, g = _tv64(grid)
            loss, G = loss + case["tv"] * tv, G + case["tv"] * g
        return {"rgba": rgba, "loss": loss, "grad": G}
    reads = None if s["occ"] is None else _cells_read(s["occ"], case["interp"])
    if kind == "rays":
        o, d, tgt = s["o"], s["d"], s["targets"].double()
    else:
        o, d = _camera_rays(s["c2w"], s["cam_ids"], s["uv"])
        tgt = None if kind == "view" else _targets(s["imgs"], s["cam_ids"], s["uv"]).double()
    rgba, _, G = _chain64(s["grid"].double(), reads, o, d, None if tgt is None else _mse_seed(tgt), S, s["delta"],
                          s["near"], s["gmin"], s["pd"], case["interp"], case["t_stop"], grad=tgt is not None)
    if kind == "view":
        return rgba
    if kind == "rays":
        return {"rgba": rgba, "grad": G}
    sq = ((rgba - tgt) ** 2).sum(1)
    return {"loss": sq.mean() / 4, "sq_err": sq, "grad": G}
