"""The work a user of this framework has it do, as cases that can be timed and compared.

Four kinds of use of the ray caster, each through its public entry point, and the other device work
of the training loop:

* ``step``    -- one training iteration through the drop-in autograd boundary
  (``RenderOptixFunction.apply``, a loss, ``torch.autograd.grad``): tree rebuild, colour, forward,
  backward, gradient assembly of all eight parameter tensors;
* ``test``    -- the inference render with caller-computed colours (``launch_pipeline_test``);
* ``frame``   -- one viewer frame: a moved camera, RGBA8 image and depth (``render_frame``);
* ``batch``   -- one batched multi-view training pass (``BatchedTrainer.step``);
* ``loss``    -- L1 + SSIM and its gradient (``l1_ssim_loss``);
* ``adam``    -- the optimiser step over all parameters and the projections after it;
* ``densify`` -- clone / split / prune of every parameter with its Adam moments;
* ``knn``     -- the initialisation's mean squared distance to the three nearest points.

Scenes follow ``ray_gauss_amd.scenes`` (uniform, blob mixture, unbounded: inner blobs and a shell of
growing scales), drawn on the GPU from the seed.
"""

from __future__ import annotations

import math
from types import SimpleNamespace

import numpy as np
import torch

from ray_gauss_amd import densify, loss, optim, optix_utils, render, viewer
from ray_gauss_amd.batch import BatchedTrainer, make_ray_batch
from ray_gauss_amd.cameras import look_at_camera, orbit_eye
from ray_gauss_amd.caster import RayCaster, TuneConfig
from ray_gauss_amd.scenes import RenderParams

DEV = "cuda"
GEOMETRY = ("positions", "scales", "quats", "densities")
BOUNDARY = GEOMETRY + ("sh", "sg", "sharpness", "lobe_axis")

# Mean slab hits per ray and million Gaussians of each scene at its usual view (dt 0.01, 8 samples
# per slab), for the operation counts only.
HITS_PER_MILLION = {"uniform": 6000.0, "blobs": 390.0, "unbounded": 660.0}
# Operations of one slab hit (8 samples): weight, threshold and colour sums; and their gradients.
FORWARD_OPS, BACKWARD_OPS = 120.0, 260.0


def listed():
    return [
        # The smallest call: a training iteration on a toy scene, where launches and host work count.
        {"name": "step 4k 64x64", "kind": "step", "scene": "uniform", "n": 4096, "w": 64, "h": 64, "ss": 1, "deg": 3,
         "lobes": 0, "random": False, "loss": "l2"},
        # An early iteration: low SH degree, two lobes, an odd image with jittered, randomly placed
        # samples and 2x1 supersampling.
        {"name": "step 30k ragged", "kind": "step", "scene": "blobs", "n": 30011, "w": 331, "h": 247, "ss": 2, "deg": 1,
         "lobes": 2, "random": True, "loss": "l1_ssim"},
        # The ordinary iteration on an object scene: 100k Gaussians, one 800x800 view.
        {"name": "step 100k 800x800", "kind": "step", "scene": "blobs", "n": 100_000, "w": 800, "h": 800, "ss": 1,
         "deg": 3, "lobes": 4, "random": False, "loss": "l1_ssim"},
        # Evaluation of a trained object scene: one test view after another.
        {"name": "test 100k 800x800", "kind": "test", "scene": "blobs", "n": 100_000, "w": 800, "h": 800},
        # The interactive viewer on an unbounded scene: a new camera, one frame.
        {"name": "frame 1M 1237x822", "kind": "frame", "scene": "unbounded", "n": 1_000_000, "w": 1237, "h": 822},
        # A batched pass over views of uneven size, each partly sampled.
        {"name": "batch 300k uneven", "kind": "batch", "scene": "blobs", "n": 300_000, "views": 8, "w": 1600, "h": 1200,
         "uneven": True, "lobes": 4},
        # The largest: the batched pass of the benchmark, 8 full views of an unbounded scene.
        {"name": "batch 1M 8 views", "kind": "batch", "scene": "unbounded", "n": 1_000_000, "views": 8, "w": 1237,
         "h": 822, "uneven": False, "lobes": 4},
        # The loss of one training image.
        {"name": "loss 1237x822", "kind": "loss", "w": 1237, "h": 822, "ss": 1},
        # The optimiser's step of an unbounded scene.
        {"name": "adam 1M", "kind": "adam", "n": 1_000_000, "lobes": 4},
        # Densification in the middle of a training, every 100 iterations or so.
        {"name": "densify 400k", "kind": "densify", "n": 400_003, "lobes": 4},
        # Initialisation from a structure-from-motion cloud.
        {"name": "knn 120k", "kind": "knn", "n": 120_011},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "test", "frame", "batch", "batch", "loss", "adam", "densify", "knn"])
    if kind == "step":
        n = _log(rng, 1500, 250_000)
        w = _log(rng, 40, 1000)
        h = max(16, int(w * rng.uniform(0.5, 1.1)))
        scene = "uniform" if n < 5000 else rng.choice(["blobs", "unbounded"])
        return {"kind": kind, "scene": scene, "n": n, "w": w, "h": h, "ss": rng.choice([1, 1, 2]) if w < 500 else 1,
                "deg": rng.choice([0, 1, 2, 3, 3]), "lobes": rng.choice([0, 1, 4, 7]) if n >= 5000 else 0,
                "random": rng.random() < 0.3 and n >= 5000, "loss": "l1_ssim" if n >= 5000 else "l2"}
    if kind == "test":
        w = _log(rng, 200, 1600)
        return {"kind": kind, "scene": rng.choice(["blobs", "unbounded"]), "n": _log(rng, 10_000, 600_000), "w": w,
                "h": max(64, int(w * rng.uniform(0.5, 1.1)))}
    if kind == "frame":
        w = _log(rng, 300, 1920)
        return {"kind": kind, "scene": rng.choice(["blobs", "unbounded"]), "n": _log(rng, 20_000, 1_000_000), "w": w,
                "h": max(64, int(w * 0.5625) + rng.randrange(8))}
    if kind == "batch":
        w = _log(rng, 200, 1250)
        return {"kind": kind, "scene": rng.choice(["blobs", "unbounded"]), "n": _log(rng, 20_000, 900_000),
                "views": rng.randrange(2, 9), "w": w, "h": max(64, int(w * rng.uniform(0.5, 0.7))),
                "uneven": rng.random() < 0.5, "lobes": rng.choice([0, 2, 4, 8])}
    if kind == "loss":
        w = _log(rng, 100, 1600)
        return {"kind": kind, "w": w, "h": max(32, int(w * rng.uniform(0.5, 1.1))), "ss": rng.choice([1, 1, 2])}
    if kind == "adam":
        return {"kind": kind, "n": _log(rng, 10_000, 1_500_000), "lobes": rng.choice([0, 2, 4])}
    if kind == "densify":
        return {"kind": kind, "n": _log(rng, 10_000, 600_000), "lobes": rng.choice([1, 2, 4])}
    return {"kind": kind, "n": _log(rng, 5_000, 160_000)}


# ---------------------------------------------------------------- inputs ---------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _unit(t):
    return t / t.norm(dim=-1, keepdim=True)


def _rotation(q):
    w, x, y, z = q.unbind(-1)
    return torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                        2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                        2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], -1).view(-1, 3, 3)


def _means_and_scales(scene, n, g):
    rn = lambda *s: torch.randn(s, generator=g, device=DEV)  # noqa: E731
    ru = lambda *s: torch.rand(s, generator=g, device=DEV)  # noqa: E731

    def blobs(count, centres):
        k = centres.shape[0]
        std = 0.05 + 0.15 * ru(k, 3)
        rot = _rotation(_unit(rn(k, 4)))
        which = torch.randint(0, k, (count,), generator=g, device=DEV)
        local = rn(count, 3) * std[which]
        return centres[which] + (rot[which] * local[:, None, :]).sum(-1)

    if scene == "uniform":
        return ru(n, 3) * 2 - 1, torch.exp(-3.5 + 0.3 * rn(n, 3))
    if scene == "blobs":
        return blobs(n, ru(32 if n <= 150_000 else 96, 3) * 2 - 1), torch.exp(-4.5 + 0.4 * rn(n, 3))
    inner = int(round(0.6 * n))
    pin = blobs(inner, _unit(rn(64, 3)) * ru(64, 1) ** (1 / 3) * 0.8)
    r = torch.exp(math.log(2.0) + (math.log(50.0) - math.log(2.0)) * ru(n - inner, 1))
    pos = torch.cat([pin, _unit(rn(n - inner, 3)) * r])
    scale = torch.exp(-4.5 + 0.4 * rn(n, 3)) * torch.cat([torch.ones(inner, 1, device=DEV), r])
    return pos, scale


def _scene(scene, n, g, deg=3, lobes=0):
    """The activated parameter tensors of the ray caster's boundary."""
    rn = lambda *s: torch.randn(s, generator=g, device=DEV)  # noqa: E731
    pos, scale = _means_and_scales(scene, n, g)
    K = (deg + 1) ** 2
    sh = 0.05 * rn(n, 3, K)
    sh[:, :, 0] = 0.5 + 0.2 * rn(n, 3)
    return {"positions": pos.contiguous(), "scales": scale.contiguous(), "quats": _unit(rn(n, 4)).contiguous(),
            "densities": torch.nn.functional.softplus(rn(n)).contiguous(), "sh": sh.contiguous(),
            "sg": 0.1 * rn(n, 3, lobes),
            "sharpness": torch.exp(math.log(50.0) * torch.rand((n, lobes), generator=g, device=DEV)),
            "lobe_axis": _unit(rn(n, lobes, 3)) if lobes else torch.zeros((n, 0, 3), device=DEV)}


def _camera(case, azimuth=30.0, elevation=20.0):
    radius = {"uniform": 3.0, "blobs": 4.0, "unbounded": 3.5}[case["scene"]]
    return look_at_camera(orbit_eye(radius, azimuth, elevation), width=case["w"], height=case["h"], fovx_deg=40.0)


def _params(case, white=True):
    if case["scene"] == "uniform":
        return RenderParams(dt=0.01, t_eps=1e-4, t_near=0.5, t_far=6.0, white_background=False)
    return RenderParams(dt=0.01, t_eps=1e-4, white_background=white)


def _views(case):
    """Cameras and pixel lists of a batched pass; sizes and subsets belong to the case."""
    if not case["uneven"]:
        cams = [_camera(case, 360.0 * i / case["views"] + 7.0, 15.0) for i in range(case["views"])]
        return [c.launch_record() for c in cams], None
    rng = np.random.default_rng(case["n"] + case["w"])
    cams, pixels = [], []
    for _ in range(case["views"]):
        w = int(rng.integers(case["w"] // 4, case["w"] + 1))
        h = max(1, int(round(w * case["h"] / case["w"])))
        cam = _camera({**case, "w": w, "h": h}, rng.uniform(0, 360), rng.uniform(-30, 45))
        keep = int(round(rng.uniform(0.25, 1.0) * w * h))
        cams.append(cam.launch_record())
        pixels.append(np.sort(rng.permutation(w * h)[:keep]).astype(np.int32))
    return cams, pixels


def _ray_count(case):
    if not case.get("uneven"):
        return case["w"] * case["h"] * case.get("views", 1) * case.get("ss", 1)
    cams, pixels = _views(case)
    return sum(len(p) for p in pixels)


WIDTHS = (("xyz", "positions", (3,)), ("rgb", "rgb", (3, 1)), ("sh", "spherical_harmonics", (3, 15)),
          ("density", "densities", (1,)), ("scales", "scales", (3,)), ("quaternions", "quaternions", (4,)))
RATES = {"xyz": 1.6e-4, "rgb": 5e-3, "sh": 2.5e-4, "density": 5e-2, "scales": 5e-3, "quaternions": 1e-3,
         "sph_gauss_features": 5e-3, "bandwidth_sharpness": 5e-3, "lobe_axis": 1e-3}


def _cloud(case, g):
    """Raw parameters by optimiser name, as the training loop holds them."""
    n, L = case["n"], case["lobes"]
    rn = lambda *s: torch.randn(s, generator=g, device=DEV)  # noqa: E731
    shapes = [(name, attr, w) for name, attr, w in WIDTHS]
    shapes += [("sph_gauss_features", "sph_gauss_features", (3, L)), ("bandwidth_sharpness", "bandwidth_sharpness", (L,)),
               ("lobe_axis", "lobe_axis", (L, 3))]
    values = {name: 0.1 * rn(n, *w) for name, _, w in shapes}
    values["xyz"] = _means_and_scales("blobs", n, g)[0].contiguous()
    values["scales"] = -4.5 + 0.4 * rn(n, 3)
    values["density"] = 0.5 + 0.4 * rn(n, 1)
    values["quaternions"] = rn(n, 4)
    values["lobe_axis"] = rn(n, L, 3)
    return shapes, values


def _with_optimisers(values, g, step):
    opts = {}
    for name, v in values.items():
        p = v.requires_grad_(True)
        o = optim.FusedAdam([p], lr=RATES[name])
        o.state[p] = {"step": torch.tensor(float(step)),
                      "exp_avg": 1e-3 * torch.randn(v.shape, generator=g, device=DEV),
                      "exp_avg_sq": 1e-6 * torch.rand(v.shape, generator=g, device=DEV)}
        opts[name] = o
    return opts


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    s = SimpleNamespace(kind=kind, case=dict(case))
    if kind == "step":
        s.leaves = _scene(case["scene"], case["n"], g, case["deg"], case["lobes"])
        for k in BOUNDARY:
            s.leaves[k].requires_grad_(case["lobes"] > 0 or k in GEOMETRY or k == "sh")
        s.ctx = optix_utils.create_context()
        s.params, s.cam = _params(case), _camera(case)
        shape = (3, case["h"], case["w"]) if case["loss"] == "l1_ssim" else (case["h"] * case["w"] * case["ss"], 3)
        s.target = torch.rand(shape, generator=g, device=DEV)
    elif kind == "test":
        s.scene = _scene(case["scene"], case["n"], g, 0)
        s.colors = (0.5 + 0.3 * torch.randn((case["n"], 3), generator=g, device=DEV)).contiguous()
        s.ctx = optix_utils.create_context()
        groups = optix_utils.create_program_groups(s.ctx, optix_utils.create_module(s.ctx, None, "test"))
        s.pipeline = optix_utils.create_pipeline(s.ctx, groups, None)
        s.cam = _camera(case)
    elif kind == "frame":
        t = _scene(case["scene"], case["n"], g, 3, 4)
        s.scene = t
        s.caster = RayCaster(_params(case), TuneConfig(tree_builder=1))
        s.caster.prepare(*(t[k] for k in BOUNDARY), rebuild=True)
        s.cam = _camera(case).launch_record()
    elif kind == "batch":
        t = _scene(case["scene"], case["n"], g, 3, case["lobes"])
        cams, pixels = _views(case)
        rv, rp, _ = make_ray_batch(cams, pixels, DEV)
        s.target = torch.rand((rv.shape[0], 3), generator=g, device=DEV)
        s.trainer = BatchedTrainer(RayCaster(_params(case), TuneConfig(tree_builder=1)), t, cams, rv, rp, s.target)
    elif kind == "loss":
        w, h, ss = case["w"], case["h"], case["ss"]
        ramp = torch.linspace(0, 9, w * ss, device=DEV).sin()[None, :, None] * 0.3 + 0.5
        s.rays = (ramp + 0.1 * torch.randn((h * ss, w * ss, 3), generator=g, device=DEV)).view(-1, 3).contiguous()
        s.rays.requires_grad_(True)
        s.target = (ramp.view(w, ss).mean(1)[None, None, :] +
                    0.1 * torch.randn((3, h, w), generator=g, device=DEV)).contiguous()
    elif kind == "adam":
        _, values = _cloud(case, g)
        values = {k: v for k, v in values.items() if v.numel()}
        grads = {k: 1e-3 * torch.randn(v.shape, generator=g, device=DEV) for k, v in values.items()}
        s.values, s.opts = values, _with_optimisers(values, g, 10)
        for k, v in values.items():
            v.grad = grads[k]
        s.filter = (-6.0 + 0.5 * torch.randn((case["n"], 1), generator=g, device=DEV)).contiguous()
    elif kind == "densify":
        shapes, values = _cloud(case, g)
        n = case["n"]
        s.shapes, s.values, s.seed = shapes, values, int(seed)
        moments = [torch.randn(v.shape, generator=g, device=DEV) for v in values.values()]
        s.moments = dict(zip(values, moments))
        # what decides who is cloned, split or pruned: the same population in another order for each
        # seed, so that every seed's outputs have the same size
        fixed, order = _gen(n), torch.randperm(n, generator=g, device=DEV)
        s.accum = (torch.rand(n, generator=fixed, device=DEV) ** 4 * 0.01)[order]
        s.count = torch.randint(0, 30, (n,), generator=fixed, device=DEV).float()[order]
        values["scales"] = (-4.5 + 0.4 * torch.randn((n, 3), generator=fixed, device=DEV))[order].contiguous()
        values["density"] = (0.5 + 0.4 * torch.randn((n, 1), generator=fixed, device=DEV))[order].contiguous()
        s.filter = torch.randn((n, 1), generator=g, device=DEV)
    else:
        s.points = _means_and_scales("blobs", case["n"], g)[0].contiguous()
    return s


# ---------------------------------------------------------------- passes ---------------------------


def _run_step(s):
    c, t = s.case, s.leaves
    settings = render.RenderOptixSettings(s.ctx, False, None, None, None, None, None, s.cam, 0, c["lobes"], 7,
                                          int(c["random"]), int(c["random"]), (c["ss"], 1),
                                          s.params.white_background, None, params=s.params)
    rays = render.RenderOptixFunction.apply(*(t[k] for k in BOUNDARY), settings)
    if c["loss"] == "l1_ssim":
        value = loss.l1_ssim_loss(rays, s.target, c["w"], c["h"], (c["ss"], 1))
    else:
        value = ((rays - s.target) ** 2).sum()
    wanted = [k for k in BOUNDARY if t[k].requires_grad]
    grads = torch.autograd.grad(value, [t[k] for k in wanted])
    return {"rays": rays.detach(), "loss": value.detach(), "grads": dict(zip(wanted, grads))}


def _run_test(s):
    t = s.scene
    return optix_utils.launch_pipeline_test(s.pipeline, None, None, None, None, s.cam, t["densities"], s.colors,
                                            t["positions"], t["scales"], t["quats"], 0, 0, (1, 1), True)


def _run_adam(s):
    optim.step_all(list(s.opts.values()))
    v = {k: t.detach() for k, t in s.values.items()}
    optim.project_params(v["density"], v["scales"], s.filter, 0.5, v["quaternions"], v.get("lobe_axis"))
    return {"params": v, "moments": {k: [o.state[s.values[k]][m] for m in ("exp_avg", "exp_avg_sq")]
                                     for k, o in s.opts.items()}}


def _run_densify(s):
    pc, opts = SimpleNamespace(), {}
    for name, attr, _ in s.shapes:
        p = s.values[name]
        setattr(pc, attr, p)
        opts[name] = SimpleNamespace(optimizer=SimpleNamespace(
            param_groups=[{"params": [p]}], state={p: {"exp_avg": s.moments[name], "exp_avg_sq": s.moments[name]}}))
    pc.optim_managers = SimpleNamespace(optimizer_manager_dict=opts)
    pc.xyz_gradient_accum_norm, pc.num_accum, pc.num_accum_gnv, pc.filter_3D = s.accum, s.count, s.count, s.filter
    counts = densify.densify_and_prune(pc, 4e-5, 0.05, 1.0, generator=_gen(s.seed + 1))
    out = {"counts": list(counts)}
    for name, attr, _ in s.shapes:
        p = getattr(pc, attr)
        m = opts[name].optimizer.state[p]
        out[name] = [p.detach(), m["exp_avg"], m["exp_avg_sq"]]
    out["filter"], out["gnv"] = pc.filter_3D, pc.num_accum_gnv
    return out


def run(state):
    kind = state.kind
    if kind == "step":
        return _run_step(state)
    if kind == "test":
        return _run_test(state)
    if kind == "frame":
        state.caster.set_views([state.cam])
        return viewer.render_frame(state.caster, 0)
    if kind == "batch":
        grads = state.trainer.step()
        return {"loss": state.trainer.loss, "grads": grads}
    if kind == "loss":
        c = state.case
        value = loss.l1_ssim_loss(state.rays, state.target, c["w"], c["h"], (c["ss"], c["ss"]))
        return {"loss": value.detach(), "grad": torch.autograd.grad(value, state.rays)[0]}
    if kind == "adam":
        return _run_adam(state)
    if kind == "densify":
        return _run_densify(state)
    return densify.distCUDA2(state.points)


# ---------------------------------------------------------------- what a pass cannot do without ----


def work(case):
    kind = case["kind"]
    if kind == "loss":
        px, rays = case["w"] * case["h"], case["w"] * case["h"] * case["ss"] ** 2
        return {"bytes": 12.0 * px + 24.0 * rays, "flops": 3.0 * px * 8 * 22 * 2}
    if kind == "knn":  # in and out; about two hundred candidates tested per point
        return {"bytes": 16.0 * case["n"], "flops": 200.0 * 9 * case["n"]}
    if kind in ("adam", "densify"):
        width = 59 + 7 * case["lobes"]
        if kind == "adam":  # parameter, gradient, two moments read; parameter and moments written
            return {"bytes": 28.0 * width * case["n"] + 80.0 * case["n"], "flops": 12.0 * width * case["n"]}
        return {"bytes": 2 * 12.0 * width * case["n"], "flops": 100.0 * case["n"]}
    n, rays = case["n"], _ray_count(case)
    hits = HITS_PER_MILLION[case["scene"]] * n * 1e-6 * rays
    if kind == "test":
        return {"bytes": 56.0 * n + 12.0 * rays, "flops": FORWARD_OPS * hits}
    if kind == "frame":
        return {"bytes": 4.0 * (11 + 48 + 28) * n + 8.0 * rays, "flops": FORWARD_OPS * hits}
    width = 11 + 3 * (case.get("deg", 3) + 1) ** 2 + 7 * case["lobes"]
    return {"bytes": 8.0 * width * n + 24.0 * rays, "flops": (FORWARD_OPS + BACKWARD_OPS) * hits}


# ---------------------------------------------------------------- the same in 64 bits --------------


class _SecondOrderY9(torch.autograd.Function):
    """y (3 x^2 - y^2) with the derivative in y that the reference's colour backward uses."""

    @staticmethod
    def forward(ctx, x, y):
        ctx.save_for_backward(x, y)
        return y * (3 * x * x - y * y)

    @staticmethod
    def backward(ctx, g):
        x, y = ctx.saved_tensors
        return g * 6 * x * y, g * (3 * x * x - y * y)


def _colors64(t, eye):
    """SH colours + 0.5, reference basis, in 64 bits."""
    x, y, z = _unit(t["positions"] - eye).unbind(-1)
    xx, yy, zz = x * x, y * y, z * z
    basis = [torch.full_like(x, 0.28209479177387814), -0.4886025119029199 * y, 0.4886025119029199 * z,
             -0.4886025119029199 * x, 1.0925484305920792 * x * y, -1.0925484305920792 * y * z,
             0.31539156525252005 * (2 * zz - xx - yy), -1.0925484305920792 * x * z, 0.5462742152960396 * (xx - yy),
             -0.5900435899266435 * _SecondOrderY9.apply(x, y), 2.890611442640554 * x * y * z,
             -0.4570457994644658 * y * (4 * zz - xx - yy), 0.3731763325901154 * z * (2 * zz - 3 * xx - 3 * yy),
             -0.4570457994644658 * x * (4 * zz - xx - yy), 1.445305721320277 * z * (xx - yy),
             -0.5900435899266435 * x * (xx - 3 * yy)]
    K = t["sh"].shape[2]
    return 0.5 + (t["sh"] * torch.stack(basis[:K], -1)[:, None, :]).sum(-1)


def _grid32(case, params, t):
    """Ray directions, entry and exit in FP32: the discrete sample positions of the method."""
    cam = _camera(case).launch_record()
    f = lambda v: torch.from_numpy(np.asarray(v, np.float32)).to(DEV)  # noqa: E731
    w, h = cam["width"], cam["height"]
    px = torch.arange(w * h, device=DEV)
    fx = ((px % w).float() + 0.5) / float(w)
    fy = ((px // w).float() + 0.5) / float(h)
    ddx, ddy = (2 * fx - 1) * f(cam["tanx"]), (2 * fy - 1) * f(cam["tany"])
    u, v, fw, eye = f(cam["u"]), f(cam["v"]), f(cam["w"]), f(cam["eye"])
    d = (ddx[:, None] * u + ddy[:, None] * v) + fw
    len2 = (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2]
    d = d * (1.0 / len2.sqrt())[:, None]
    with torch.no_grad():  # the union of the ellipsoids' boxes
        delta = torch.log((t["densities"] / params.sigma_thr) ** 2).clamp(min=0).sqrt()
        half = (_rotation(t["quats"]) * (delta[:, None] * t["scales"])[:, None, :]).norm(dim=-1)
        lo = (t["positions"] - half).amin(0).float()
        hi = (t["positions"] + half).amax(0).float()
    a, b = (lo - eye) / d, (hi - eye) / d
    enter = torch.minimum(a, b).amax(1).clamp(min=params.t_near)
    leave = torch.maximum(a, b).amin(1).clamp(max=params.t_far)
    return eye.double(), d, enter, leave


def _exact_step(case, seed):
    """Every Gaussian at every sample of every ray, with the method's sample grid, thresholds and exit."""
    params = _params(case)
    s = prepare(case, seed)
    t = {k: v.detach().double().requires_grad_(v.requires_grad) for k, v in s.leaves.items()}
    eye, d32, enter, leave = _grid32(case, params, t)
    dt, spb = np.float32(params.dt), params.samples_per_slab
    slabs = int(math.ceil(float((leave - enter).clamp(min=0).amax()) / (params.dt * spb))) + 1
    starts = [enter]
    for _ in range(slabs - 1):
        starts.append(starts[-1] + float(np.float32(dt * np.float32(spb))))
    starts = torch.stack(starts, 1)  # (rays, slabs), accumulated in FP32
    offs = torch.from_numpy((np.arange(spb, dtype=np.float32) * dt)).to(DEV)
    times = (starts[:, :, None] + offs).flatten(1).double()
    inside = (starts < leave[:, None]).double()
    colors = _colors64(t, eye)
    # |M (o + t d - mu)|^2 = a t^2 + 2 b t + c with M = diag(1/s) R^T
    M = _rotation(t["quats"]).transpose(1, 2) / t["scales"][:, :, None]
    o = (M * (eye - t["positions"])[:, None, :]).sum(-1)  # (n, 3)
    total = torch.zeros((), dtype=torch.float64, device=DEV)
    rays = torch.zeros((d32.shape[0], 3), dtype=torch.float64, device=DEV)
    wanted = [k for k in BOUNDARY if t[k].requires_grad]
    inner = [M, o, t["densities"], colors]
    sums = [torch.zeros_like(v) for v in inner]
    for i in range(0, d32.shape[0], 32):
        Mi, oi, si, ci = (v.detach().requires_grad_(True) for v in inner)
        d = d32[i:i + 32].double()
        dp = (Mi[None] * d[:, None, None, :]).sum(-1)  # (r, n, 3)
        b, a = (dp * oi).sum(-1), (dp * dp).sum(-1)
        tc = -b / a
        # distance terms at the closest approach, free of cancellation
        p2 = (oi + tc[:, :, None] * dp).square().sum(-1)
        near = ((p2 < 2 * torch.log(si.abs() / params.sigma_thr)).any(0)).nonzero()[:, 0]
        p2, tc, a = p2[:, near], tc[:, near], a[:, near]
        tt = times[i:i + 32]
        q = p2[:, None, :] + a[:, None, :] * (tt[:, :, None] - tc[:, None, :]).square()
        w = si[near] * torch.exp(-0.5 * q)
        w = torch.where(w > params.sigma_thr, w, 0.0)  # (r, samples, near)
        sigma = w.sum(-1)
        color = (w @ ci[near]) / sigma.clamp(min=1e-300)[:, :, None]
        alpha = 1 - torch.exp(-sigma * params.dt)
        by_slab = torch.cumprod((1 - alpha).view(len(d), slabs, spb).prod(-1), 1)
        before = torch.cat([torch.ones_like(by_slab[:, :1]), by_slab[:, :-1]], 1)
        live = ((before > params.t_eps).double().cumprod(1) * inside[i:i + 32]).repeat_interleave(spb, 1)
        alpha = alpha * live.detach()
        T = torch.cumprod(1 - alpha, 1)
        T0 = torch.cat([torch.ones_like(T[:, :1]), T[:, :-1]], 1)
        out = ((T0 * alpha)[:, :, None] * color).sum(1) + T[:, -1:] * float(params.white_background)
        value = (out - s.target[i:i + 32].double()).square().sum()
        for acc, gr in zip(sums, torch.autograd.grad(value, [Mi, oi, si, ci])):
            acc += gr
        rays[i:i + 32] = out.detach()
        total = total + value.detach()
    grads = torch.autograd.grad(inner, [t[k] for k in wanted], sums)
    return {"rays": rays, "loss": total, "grads": dict(zip(wanted, grads))}


def _exact_loss(case, seed):
    s = prepare(case, seed)
    w, h, ss = case["w"], case["h"], case["ss"]
    rays = s.rays.detach().double().requires_grad_(True)
    x = rays.view(h, ss, w, ss, 3).mean((1, 3)).permute(2, 0, 1)
    y = s.target.double()
    k = torch.exp(-(torch.arange(11, device=DEV).double() - 5) ** 2 / (2 * 1.5 ** 2))
    k = (k / k.sum()).tolist()

    def blur(v):
        v = torch.nn.functional.pad(v, (5, 5, 0, 0))
        v = sum(k[i] * v[:, :, i:i + w] for i in range(11))
        v = torch.nn.functional.pad(v, (0, 0, 5, 5))
        return sum(k[i] * v[:, i:i + h, :] for i in range(11))

    m1, m2 = blur(x), blur(y)
    v1, v2, c = blur(x * x) - m1 * m1, blur(y * y) - m2 * m2, blur(x * y) - m1 * m2
    ssim = ((2 * m1 * m2 + 1e-4) * (2 * c + 9e-4)) / ((m1 * m1 + m2 * m2 + 1e-4) * (v1 + v2 + 9e-4))
    value = 0.8 * (x - y).abs().mean() + 0.2 * (1 - ssim.mean())
    return {"loss": value.detach(), "grad": torch.autograd.grad(value, rays)[0]}


def _exact_adam(case, seed):
    s = prepare(case, seed)
    out, moments = {}, {}
    for k, v in s.values.items():
        st, g = s.opts[k].state[v], v.grad.double()
        m = 0.9 * st["exp_avg"].double() + 0.1 * g
        q = 0.999 * st["exp_avg_sq"].double() + 0.001 * g * g
        step = RATES[k] / (1 - 0.9 ** 11)
        out[k] = v.detach().double() - step * m / (q.sqrt() / math.sqrt(1 - 0.999 ** 11) + 1e-15)
        moments[k] = [m, q]
    out["density"] = out["density"].clamp(min=0)
    out["scales"] = torch.minimum(torch.maximum(out["scales"], s.filter.double()), torch.tensor(0.5, device=DEV).double())
    for k in ("quaternions", "lobe_axis"):
        if k in out:
            out[k] = _unit(out[k])
    return {"params": out, "moments": moments}


def _exact_knn(case, seed):
    p = prepare(case, seed).points.double()
    out = torch.empty(p.shape[0], dtype=torch.float64, device=DEV)
    for i in range(0, p.shape[0], 1024):
        d = sum((p[i:i + 1024, None, k] - p[None, :, k]).square() for k in range(3))
        rows = torch.arange(d.shape[0], device=DEV)
        d[rows, rows + i] = math.inf
        out[i:i + 1024] = torch.topk(d, 3, dim=1, largest=False).values.mean(1)
    return out


def exact(case, seed):
    if case["kind"] == "step" and case["loss"] == "l2" and case["ss"] == 1 and case["n"] * case["w"] * case["h"] < 4e7:
        return _exact_step(case, seed)
    if case["kind"] == "loss":
        return _exact_loss(case, seed)
    if case["kind"] == "adam":
        return _exact_adam(case, seed)
    if case["kind"] == "knn":
        return _exact_knn(case, seed)
    return None  # over the time a check may take, or copies of the inputs (densification)
