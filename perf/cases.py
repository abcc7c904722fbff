"""What the framework's speed is measured on: frames, training passes and steps,
the loss, the optimizers and the densification passes, each through the entry
point a trainer or viewer calls.

A case is a dict of plain values; ``kind`` names the entry point:

  frame   render() under no_grad: a viewer's or an evaluation's frame
  train   render(), photometric_loss() and the backward to every parameter
  step    the same with FusedAdam's update inside the backward: a whole step
  loss    photometric_loss() and its backward alone
  adam    FusedAdam.step(), or with "visible" below 1 SelectiveAdam.step()
  noise   mcmc.add_noise(), every step of an MCMC training
  grow    mcmc.grow(), every densification interval
  filter  compute_3d_filter(), every densification interval of a Mip training

Scenes follow metal_gauss_amd.scenes (the benchmark configurations), drawn on
the GPU so that a state is made in milliseconds. ``exact`` restates each path
in float64 torch, from the formulas and not from this package.
"""

import math
import random

import numpy as np
import torch

import metal_gauss_amd as mg
from metal_gauss_amd import mcmc

DEVICE = "cuda"

# Floats per Gaussian and rate of the trainer's six parameter groups. The
# rates are a hundredth of the configured ones, the end of a decayed
# schedule: a few thousand passes over one state stay in the same scene.
GROUPS = (("means", 3, 1.6e-6), ("log_scales", 3, 5e-5), ("quats", 4, 1e-5),
          ("logit_opac", 1, 5e-4), ("sh_dc", 3, 2.5e-5), ("sh_rest", 45, 1.25e-6))
STEP0 = 1000        # optimizer steps before the measured ones
BETA1, BETA2, EPS = 0.9, 0.999, 1e-15
NOISE_KEY = 0x6E6F697365     # second word of add_noise's Philox key
RENDER_KEYS = ("means", "quats", "log_scales", "logit_opac", "sh_dc", "sh_rest")


# ------------------------------------------------------------------- cases

def listed():
    return [
        # The smallest scene, SH degree 0: a thumbnail or an early preview,
        # where launches and the host read of the list total count.
        dict(name="frame_10k_256", kind="frame", scene="ball", n=10_000, width=256, height=256,
             degree=0, lists="host", antialias=False),
        # A viewer's frame of a trained scene, ragged size, antialiased,
        # enqueued with capacity-sized lists.
        dict(name="frame_600k_1237x823", kind="frame", scene="frustum", n=600_000, width=1237,
             height=823, degree=3, lists="capacity", antialias=True),
        # A training pass of the usual synthetic-object size, white
        # background, gradients to a separate optimizer.
        dict(name="train_300k_800", kind="train", scene="cube", n=300_000, width=800, height=800,
             mip=False, white=True),
        # A training pass at photograph size with both Mip filters; the last
        # tile row is ragged and there are over 4096 tiles.
        dict(name="train_600k_1600x900_mip", kind="train", scene="cube", n=600_000, width=1600,
             height=900, mip=True, white=False),
        # The headline: one whole training step at 1M Gaussians.
        dict(name="step_1m_800", kind="step", scene="cube", n=1_000_000, width=800, height=800),
        # The largest: a camera inside a heavy-tailed cloud with a dense
        # cluster in front of it, tile lists of over 10k entries.
        dict(name="train_3.6m_1080p_crowded", kind="train", scene="crowded", n=3_600_000,
             width=1920, height=1080, mip=False, white=False),
        # The loss by itself at a photograph's ragged size.
        dict(name="loss_1237x823", kind="loss", width=1237, height=823),
        # The dense optimizer over 59M floats.
        dict(name="adam_1m", kind="adam", n=1_000_000, visible=1.0),
        # The visibility-masked optimizer.
        dict(name="selective_adam_1m", kind="adam", n=1_000_000, visible=0.6),
        # Exploration noise, once a step.
        dict(name="noise_1m", kind="noise", n=1_000_000),
        # A tenth more Gaussians, with the optimizer state's rows.
        dict(name="grow_1m", kind="grow", n=1_000_000, fraction=0.1),
        # The 3D filter's sizes over all training views.
        dict(name="filter_1m_100_views", kind="filter", n=1_000_000, views=100, width=800,
             height=800),
    ]


def _log_between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    width = _log_between(rng, lo, hi)
    return width, max(64, int(width * rng.uniform(0.5, 1.0)))


def draw(rng):
    kind = rng.choices(("frame", "train", "step", "loss", "adam", "noise", "grow", "filter"),
                       (8, 8, 4, 3, 3, 2, 2, 2))[0]
    if kind == "frame":
        scene = rng.choice(("ball", "frustum", "cube"))
        width, height = _size(rng, 200, 1600)
        return dict(kind=kind, scene=scene, n=_log_between(rng, 5_000, 1_000_000), width=width,
                    height=height, degree=0 if scene == "ball" else 3,
                    lists=rng.choice(("host", "capacity")), antialias=rng.random() < 0.3)
    if kind in ("train", "step"):
        scene = rng.choice(("cube", "cube", "cloud"))
        lo, hi = (300_000, 3_000_000) if scene == "cloud" else (20_000, 1_000_000)
        width, height = _size(rng, 300, 1920 if scene == "cloud" else 1400)
        case = dict(kind=kind, scene=scene, n=_log_between(rng, lo, hi), width=width,
                    height=height)
        if kind == "train":
            case.update(mip=rng.random() < 0.4, white=rng.random() < 0.3)
        return case
    if kind == "loss":
        width, height = _size(rng, 128, 1920)
        return dict(kind=kind, width=width, height=height)
    n = _log_between(rng, 50_000, 1_500_000)
    if kind == "adam":
        return dict(kind=kind, n=n, visible=rng.choice((1.0, round(rng.uniform(0.3, 0.9), 3))))
    if kind == "grow":
        return dict(kind=kind, n=n, fraction=round(rng.uniform(0.02, 0.2), 3))
    if kind == "filter":
        width, height = _size(rng, 400, 1600)
        return dict(kind=kind, n=n, views=rng.randint(20, 250), width=width, height=height)
    return dict(kind=kind, n=n)


# ------------------------------------------------------------------ inputs

def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _gaussians(n, g, means, ls_mean, ls_sd, logit_mean, logit_sd, heavy=False):
    def randn(*shape):
        return torch.randn(*shape, generator=g, device=DEVICE)

    z = randn(n, 3)
    if heavy:
        # Student-t with three degrees of freedom: a tail of large splats.
        z = z / (randn(n, 3).square().sum(1, keepdim=True) / 3.0).sqrt()
    return {"means": means, "log_scales": z * ls_sd + ls_mean, "quats": randn(n, 4),
            "logit_opac": randn(n) * logit_sd + logit_mean, "sh_dc": randn(n, 1, 3) * 0.3,
            "sh_rest": randn(n, 15, 3) * 0.05}


def _look_at(eye, target, width, height, fov_deg):
    """(K, viewmat) of a look-at pinhole, OpenCV axes, both on the host."""
    eye, target = (np.asarray(v, np.float64) for v in (eye, target))
    fwd = target - eye
    fwd /= np.linalg.norm(fwd)
    up = np.array([0.0, 0.0, 1.0]) if abs(fwd[2]) < 0.999 else np.array([0.0, 1.0, 0.0])
    right = np.cross(fwd, up)
    right /= np.linalg.norm(right)
    R = np.stack([right, np.cross(fwd, right), fwd])
    vm = np.eye(4)
    vm[:3, :3], vm[:3, 3] = R, -R @ eye
    f = 0.5 * width / math.tan(math.radians(0.5 * fov_deg))
    K = torch.tensor([[f, 0.0, width / 2], [0.0, f, height / 2], [0.0, 0.0, 1.0]])
    return K, torch.from_numpy(vm.astype(np.float32))


def _on_sphere(rng, radius):
    v = np.array([rng.gauss(0.0, 1.0) for _ in range(3)])
    return radius * v / np.linalg.norm(v)


def _scene(case, seed):
    """(parameters on the GPU, K, viewmat) of a case's scene."""
    g, rng = _generator(seed), random.Random(seed)
    n, W, H, kind = case["n"], case["width"], case["height"], case["scene"]

    def uniform(m, lo, hi):
        return torch.rand(m, 3, generator=g, device=DEVICE) * (hi - lo) + lo

    if kind == "ball":
        p = _gaussians(n, g, uniform(n, -1.0, 1.0), -4.0, 0.4, 0.0, 1.0)
        return p, *_look_at(_on_sphere(rng, 4.0), (0, 0, 0), W, H, 40.0)
    if kind == "cube":
        p = _gaussians(n, g, uniform(n, -1.3, 1.3), -4.5, 0.5, 0.0, 1.5)
        return p, *_look_at(_on_sphere(rng, 4.0), (0, 0, 0), W, H, 39.6)
    if kind == "frustum":
        u = torch.rand(n, 3, generator=g, device=DEVICE)
        z = u[:, 2] * 4.5 + 1.5
        means = torch.stack([(u[:, 0] * 0.9 - 0.45) * z, (u[:, 1] * 0.9 - 0.45) * z, z], 1)
        p = _gaussians(n, g, means, -4.5, 0.5, 0.0, 1.5)
        f = 0.5 * W / math.tan(math.radians(22.5))
        K = torch.tensor([[f, 0.0, W / 2], [0.0, f, H / 2], [0.0, 0.0, 1.0]])
        return p, K, torch.eye(4)
    a = rng.uniform(0.0, 2.0 * math.pi)
    ahead = (math.cos(a), math.sin(a), 0.0)
    base = n if kind == "cloud" else n - n // 6
    p = _gaussians(base, g, uniform(base, -2.0, 2.0), -5.0, 0.7, 0.5, 1.5, heavy=True)
    if kind == "crowded":
        m = n - base
        d = torch.randn(m, 3, generator=g, device=DEVICE)
        r = 0.2 * torch.rand(m, 1, generator=g, device=DEVICE) ** (1.0 / 3.0)
        centre = torch.tensor(ahead, device=DEVICE)
        more = _gaussians(m, g, centre + r * d / d.norm(dim=1, keepdim=True), -5.0, 0.5, 0.5, 1.5)
        p = {k: torch.cat([p[k], more[k]]) for k in p}
    return p, *_look_at([2.0 * x for x in ahead], (0, 0, 0), W, H, 60.0)


def _target(case, seed):
    """A smooth photograph: an 8 x 8 grid of colours, upsampled."""
    g = _generator(seed + 7919)
    grid = torch.rand(1, 3, 8, 8, generator=g, device=DEVICE)
    t = torch.nn.functional.interpolate(grid, size=(case["height"], case["width"]),
                                        mode="bilinear", align_corners=False)
    return t[0].permute(1, 2, 0).contiguous()


def _filter_sizes(case, seed, K):
    g = _generator(seed + 104729)
    depth = torch.rand(case["n"], generator=g, device=DEVICE) * 2.6 + 2.7
    return depth / float(K[0, 0]) * math.sqrt(0.2)


def _moments(n, seed, scale):
    """exp_avg and exp_avg_sq of every group, as after many steps of
    gradients of size ``scale``."""
    g = _generator(seed + 15485863)
    out = {}
    for k, w, _ in GROUPS:
        shape = {"logit_opac": (n,), "sh_dc": (n, 1, 3), "sh_rest": (n, 15, 3)}.get(k, (n, w))
        m = torch.randn(*shape, generator=g, device=DEVICE) * (0.2 * scale)
        v = (torch.rand(*shape, generator=g, device=DEVICE) + 0.5) * (scale * scale)
        out[k] = (m, v)
    return out


def _optimizer(params, moments, selective=False):
    groups = [{"params": [params[k]], "lr": lr} for k, _, lr in GROUPS]
    opt = mg.SelectiveAdam(groups, eps=EPS) if selective else mg.FusedAdam(groups, eps=EPS)
    for k, _, _ in GROUPS:
        m, v = moments[k]
        state = {"exp_avg": m, "exp_avg_sq": v}
        if selective:
            state["steps"] = torch.full((m.shape[0],), float(STEP0), device=DEVICE)
        else:
            state["step"] = STEP0
        opt.state[params[k]].update(state)
    return opt


def _adam_inputs(case, seed):
    n, g = case["n"], _generator(seed)
    shapes = {"logit_opac": (n,), "sh_dc": (n, 1, 3), "sh_rest": (n, 15, 3)}
    p = {k: torch.randn(*shapes.get(k, (n, w)), generator=g, device=DEVICE) for k, w, _ in GROUPS}
    grads = {k: torch.randn(t.shape, generator=g, device=DEVICE) * 1e-3 for k, t in p.items()}
    visible = torch.rand(n, generator=g, device=DEVICE) < case["visible"]
    return p, grads, visible


def _images(case, seed):
    """A render near its target: the target, blotches of error and noise."""
    g = _generator(seed)
    target = _target(case, seed)
    image = 0.7 * target + 0.3 * _target(case, seed + 1)
    noise = torch.randn(image.shape, generator=g, device=DEVICE)
    return (image + 0.03 * noise).clamp(0.0, 1.0), target


class _View:
    """What compute_3d_filter reads of a training view."""

    def __init__(self, K, viewmat, width, height):
        self.K, self.viewmat = K, viewmat
        self.image = torch.empty(height, width, 0)


def _filter_inputs(case, seed):
    g, rng = _generator(seed), random.Random(seed)
    means = torch.rand(case["n"], 3, generator=g, device=DEVICE) * 2.6 - 1.3
    views = []
    for _ in range(case["views"]):
        # Cameras on a sphere, each looking somewhere inside the object.
        K, vm = _look_at(_on_sphere(rng, 4.0), _on_sphere(rng, 1.0), case["width"],
                         case["height"], 39.6)
        views.append(_View(K, vm, case["width"], case["height"]))
    return means, views


def _mcmc_inputs(case, seed):
    n, g = case["n"], _generator(seed)
    means = torch.rand(n, 3, generator=g, device=DEVICE) * 2.6 - 1.3
    # Many nearly transparent Gaussians, which the noise moves.
    return _gaussians(n, g, means, -4.5, 0.5, -2.0, 2.0)


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case, "seed": seed}
    if kind in ("frame", "train", "step"):
        p, K, viewmat = _scene(case, seed)
        state.update(K=K, viewmat=viewmat, cap=None)
        if kind == "frame":
            # As load_ply hands a viewer its splats.
            sh = p["sh_dc"] if case["degree"] == 0 else torch.cat([p["sh_dc"], p["sh_rest"]], 1)
            state.update(means=p["means"], quats=p["quats"], scales=torch.exp(p["log_scales"]),
                         opacities=torch.sigmoid(p["logit_opac"]), sh=sh)
        else:
            state["params"] = {k: p[k].requires_grad_(True) for k in RENDER_KEYS}
            state["target"] = _target(case, seed)
            state["window"] = mg.gaussian_kernel(device=DEVICE, groups=15)
            state["filter_3d"] = _filter_sizes(case, seed, K) if case.get("mip") else None
            state["opt"] = None
            if kind == "step":
                state["moments"] = _moments(case["n"], seed, 1e-8)
                state["opt"] = _optimizer(state["params"], state["moments"])
        if kind != "frame" or case["lists"] == "capacity":
            # Lists sized by the frames before this one.
            state["cap"] = mg.ListCapacity()
            with torch.no_grad():
                _frame(state) if kind == "frame" else _render(state, None)
                if state["cap"].overflowed():
                    _frame(state) if kind == "frame" else _render(state, None)
    elif kind == "loss":
        image, target = _images(case, seed)
        state.update(image=image.requires_grad_(True), target=target,
                     window=mg.gaussian_kernel(device=DEVICE, groups=15))
    elif kind == "adam":
        p, grads, visible = _adam_inputs(case, seed)
        state["params"] = {k: t.requires_grad_(True) for k, t in p.items()}
        for k, t in state["params"].items():
            t.grad = grads[k]
        state["moments"] = _moments(case["n"], seed, 1e-3)
        state["visible"] = visible if case["visible"] < 1.0 else None
        state["opt"] = _optimizer(state["params"], state["moments"],
                                  selective=state["visible"] is not None)
    elif kind == "noise":
        state["params"] = _mcmc_inputs(case, seed)
    elif kind == "grow":
        state["params"] = _mcmc_inputs(case, seed)
        state["moments"] = _moments(case["n"], seed, 1e-8)
        state["opt"] = _optimizer(state["params"], state["moments"])
    else:
        state["means"], state["views"] = _filter_inputs(case, seed)
    return state


# --------------------------------------------------------------------- run

def _frame(s):
    c = s["case"]
    return mg.render(s["means"], s["quats"], s["scales"], s["opacities"], s["sh"], s["K"],
                     s["viewmat"], c["width"], c["height"], sh_degree=c["degree"],
                     antialias=c["antialias"], list_capacity=s["cap"])


def _render(s, opt):
    c, p = s["case"], s["params"]
    background = (1.0, 1.0, 1.0) if c.get("white") else (0.0, 0.0, 0.0)
    mip = dict(filter_3d=s["filter_3d"], antialias=True) if c.get("mip") else {}
    return mg.render(p["means"], p["quats"], p["log_scales"], p["logit_opac"], p["sh_dc"], s["K"],
                     s["viewmat"], c["width"], c["height"], sh_degree=3, sh_rest=p["sh_rest"],
                     background=background, activations=True, optimizer=opt,
                     list_capacity=s["cap"], **mip)


def run(s):
    kind = s["case"]["kind"]
    if kind == "frame":
        with torch.no_grad():
            while True:
                rgb, alpha, info = _frame(s)
                if s["cap"] is None or not s["cap"].overflowed(info["lists_ticket"]):
                    return {"rgb": rgb, "alpha": alpha}
    if kind in ("train", "step"):
        p, opt = s["params"], s["opt"]
        while True:
            for t in p.values():
                t.grad = None
            rgb, _, info = _render(s, opt)
            loss, _ = mg.photometric_loss(rgb, s["target"], s["window"], 0.2)
            loss.backward()
            if opt is not None:
                opt.step(skip=info["lists_status"])
            if not s["cap"].overflowed(info["lists_ticket"]):
                break
            if opt is not None:
                opt.rewind()
        out = {"rgb": rgb, "loss": loss}
        if opt is None:
            return {**out, "grad": {k: t.grad for k, t in p.items()}}
        return {**out, "param": p, "exp_avg": {k: m for k, (m, _) in s["moments"].items()},
                "exp_avg_sq": {k: v for k, (_, v) in s["moments"].items()}}
    if kind == "loss":
        s["image"].grad = None
        loss, parts = mg.photometric_loss(s["image"], s["target"], s["window"], 0.2)
        loss.backward()
        return {"loss": loss, "parts": parts, "grad": s["image"].grad}
    if kind == "adam":
        if s["visible"] is None:
            s["opt"].step()
        else:
            s["opt"].step(s["visible"])
        return {"param": s["params"], "exp_avg": {k: m for k, (m, _) in s["moments"].items()},
                "exp_avg_sq": {k: v for k, (_, v) in s["moments"].items()}}
    if kind == "noise":
        mcmc.add_noise(s["params"], lr_means=1.6e-4, seed=s["seed"])
        return {"means": s["params"]["means"]}
    if kind == "grow":
        n = s["case"]["n"]
        mcmc.grow(s["params"], target=n, active=_active(s["case"]), opt=s["opt"], seed=s["seed"])
        return {"param": s["params"], "exp_avg": {k: m for k, (m, _) in s["moments"].items()},
                "exp_avg_sq": {k: v for k, (_, v) in s["moments"].items()}}
    return {"filter_3d": mg.compute_3d_filter(s["means"], s["views"])}


def _active(case):
    return case["n"] - int(case["n"] * case["fraction"])


# -------------------------------------------------------------------- work

def work(case):
    """Bytes: inputs read and outputs written once. Flops: the projection
    (about 400 a Gaussian), about 180 listed Gaussians walked a pixel before
    it is opaque, at 25 operations forward and 75 backward; the two 11-tap
    blurs of five moments and their adjoints; 20 operations for each
    (Gaussian, view) pair of the filter."""
    kind, n = case["kind"], case.get("n", 0)
    pixels = case.get("width", 0) * case.get("height", 0)
    if kind == "frame":
        floats = 11 + (3 if case["degree"] == 0 else 48)
        return {"bytes": 4 * floats * n + 16 * pixels, "flops": 400 * n + 25 * 180 * pixels}
    if kind == "train":
        return {"bytes": 4 * (2 * 59 + bool(case["mip"])) * n + 24 * pixels,
                "flops": 1200 * n + 100 * 180 * pixels + 3 * 500 * pixels}
    if kind == "step":
        return {"bytes": 4 * 6 * 59 * n + 24 * pixels,
                "flops": (1200 + 59 * 15) * n + 100 * 180 * pixels + 3 * 500 * pixels}
    if kind == "loss":
        return {"bytes": 36 * pixels, "flops": 3 * 500 * pixels}
    if kind == "adam":
        # Gradient, parameter and both moments read, the last three written;
        # a row's step count read and written in each of the six groups.
        seen = case["visible"]
        rows = 0 if seen == 1.0 else (48 * seen + 1) * n
        return {"bytes": 28 * 59 * n * seen + rows, "flops": 15 * 59 * n * seen}
    if kind == "noise":
        return {"bytes": 56 * n, "flops": 150 * n}
    if kind == "grow":
        added = n - _active(case)
        # Weights; a source row read and a copy written; both moments of the
        # new rows and the sources cleared; the sources' split.
        return {"bytes": 4 * _active(case) + (8 * 59 + 16 * 59 + 32) * added, "flops": 40 * n}
    return {"bytes": 16 * n, "flops": 20 * n * case["views"]}


def tolerance(case):
    """float32 throughout, so about 1e-5 for sums in another order. Rendered
    gradients add up thousands of pixels by atomics, and a splat whose alpha
    lies within rounding of the 1/255 cutoff (or a pixel within rounding of
    opaque) falls to either side: single pixels and Gaussians move by up to
    a cutoff's worth. Against ``exact``, frames are 2e-7 to 1e-5 off, images
    of training passes up to 7e-5, gradients 3e-6 to 1.2e-3."""
    kind = case["kind"]
    if kind == "frame":
        return {"rel": 1e-4, "max": 0.05}
    if kind in ("train", "step"):
        return {"rel": 4e-3, "max": 0.9}
    if kind == "grow":
        # A last-bit difference of a weight moves a few of the draws to the
        # neighbouring row.
        return {"rel": 1e-2, "max": 0.99}
    if kind == "loss":
        # 1.6e-5 off: the variances are differences of blurred squares.
        return {"rel": 6e-5, "max": 5e-3}
    if kind == "filter":
        # A Gaussian within rounding of a view's margin is seen or not: of
        # 1e8 pairs about 20 are, and a hundredth of them are the nearest.
        return {"rel": 1e-3, "max": 0.9}
    return {"rel": 1e-6, "max": 1e-4}


# ------------------------------------------- the same in 64 bits, for the error

def exact(case, seed):
    kind = case["kind"]
    if kind == "frame":
        return _exact_frame(case, seed)
    if kind in ("train", "step"):
        return _exact_train(case, seed)
    if kind == "loss":
        image, target = _images(case, seed)
        image = image.double().requires_grad_(True)
        loss, parts = _loss64(image, target.double())
        loss.backward()
        return {"loss": loss.detach(), "parts": parts, "grad": image.grad}
    if kind == "adam":
        p, grads, visible = _adam_inputs(case, seed)
        moments = _moments(case["n"], seed, 1e-3)
        dense = case["visible"] == 1.0
        return _adam64(p, grads, moments, None if dense else visible)
    if kind == "noise":
        return {"means": _noise64(_mcmc_inputs(case, seed), seed)}
    if kind == "filter":
        return {"filter_3d": _filter64(*_filter_inputs(case, seed))}
    return None     # grow: which rows are drawn hangs on a weight's last bit


def _adam64(p, grads, moments, visible=None):
    """One Adam step; with ``visible`` the masked optimizer's (eps inside the
    bias correction's root, rows not visible as they were)."""
    out = {"param": {}, "exp_avg": {}, "exp_avg_sq": {}}
    k = STEP0 + 1
    for name, _, lr in GROUPS:
        x, g = p[name].detach().double(), grads[name].double()
        m, v = (t.double() for t in moments[name])
        m1 = BETA1 * m + (1.0 - BETA1) * g
        v1 = BETA2 * v + (1.0 - BETA2) * g * g
        c1, c2 = 1.0 - BETA1 ** k, 1.0 - BETA2 ** k
        if visible is None:
            x1 = x - lr / c1 * m1 / ((v1 / c2).sqrt() + EPS)
        else:
            x1 = x - lr * math.sqrt(c2) / c1 * m1 / (v1.sqrt() + EPS)
            rows = visible.view(-1, *[1] * (x.dim() - 1))
            x1, m1, v1 = (torch.where(rows, a, b) for a, b in ((x1, x), (m1, m), (v1, v)))
        out["param"][name], out["exp_avg"][name], out["exp_avg_sq"][name] = x1, m1, v1
    return out


def _philox(i, key):
    """Philox4x64-10 (Salmon et al., SC'11) of counters (i, 0, 0, 0)."""
    mul = (np.uint64(0xD2E7470EE14C6C93), np.uint64(0xCA5A826395121157))
    weyl = (0x9E3779B97F4A7C15, 0xBB67AE8584CAA73B)
    half, low = np.uint64(32), np.uint64(0xFFFFFFFF)

    def wide(a, b):
        a0, a1, b0, b1 = a & low, a >> half, b & low, b >> half
        mid = a1 * b0 + ((a0 * b0) >> half)
        other = a0 * b1 + (mid & low)
        return a1 * b1 + (mid >> half) + (other >> half), a * b

    c = [i.astype(np.uint64)] + [np.zeros(i.shape, np.uint64) for _ in range(3)]
    k = list(key)
    for _ in range(10):
        (h0, l0), (h1, l1) = wide(mul[0], c[0]), wide(mul[1], c[2])
        c = [h1 ^ c[1] ^ np.uint64(k[0]), l1, h0 ^ c[3] ^ np.uint64(k[1]), l0]
        k = [(a + w) % 2 ** 64 for a, w in zip(k, weyl)]
    return c


def _rotation64(q):
    q = q / q.norm(dim=-1, keepdim=True).clamp_min(1e-12)
    w, x, y, z = q.unbind(-1)
    rows = [1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
            2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
            2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)]
    return torch.stack(rows, -1).view(-1, 3, 3)


def _noise64(p, seed):
    n = p["means"].shape[0]
    r = _philox(np.arange(n), (seed, NOISE_KEY))
    # 24-bit uniforms, never 0, and the Box-Muller pairs.
    u = [((x >> np.uint64(40)).astype(np.float64) + 0.5) / 2.0 ** 24 for x in r]
    r0, r1 = np.sqrt(-2.0 * np.log(u[0])), np.sqrt(-2.0 * np.log(u[2]))
    z = np.stack([r0 * np.cos(2.0 * np.pi * u[1]), r0 * np.sin(2.0 * np.pi * u[1]),
                  r1 * np.cos(2.0 * np.pi * u[3])], 1)
    e = torch.from_numpy(z).to(DEVICE) * p["log_scales"].double().exp()
    world = (_rotation64(p["quats"].double()) @ e[:, :, None])[:, :, 0]
    opacity = torch.sigmoid(p["logit_opac"].double())
    gate = torch.sigmoid(-100.0 * (opacity - 0.005))
    return p["means"].double() + world * gate[:, None] * (1.6e-4 * 4e4)


def _filter64(means, views):
    means = means.double()
    best = torch.full_like(means[:, 0], math.inf)
    focal = 0.0
    for v in views:
        vm, (H, W) = v.viewmat.double().to(DEVICE), v.image.shape[:2]
        fx, fy, cx, cy = (float(v.K[i, j]) for i, j in ((0, 0), (1, 1), (0, 2), (1, 2)))
        c = means @ vm[:3, :3].T + vm[:3, 3]
        z = c[:, 2]
        zc = z.clamp_min(1e-6)
        x, y = fx * c[:, 0] / zc + cx, fy * c[:, 1] / zc + cy
        seen = ((z > 0.2) & (x > -0.15 * W) & (x < 1.15 * W) & (y > -0.15 * H) & (y < 1.15 * H))
        best = torch.where(seen, torch.minimum(best, z), best)
        focal = max(focal, fx, fy)
    hit = torch.isfinite(best)
    far = best[hit].max() if bool(hit.any()) else torch.ones((), device=DEVICE)
    return torch.where(hit, best, far) / focal * math.sqrt(0.2)


def _window():
    x = torch.arange(11, dtype=torch.float32, device=DEVICE) - 5
    w = torch.exp(-x ** 2 / (2 * 1.5 ** 2))
    return (w / w.sum()).double()


def _blur64(x, w):
    for d in (0, 1):
        size = x.shape[d]
        pad = torch.nn.functional.pad(x, (0, 0, 0, 0, 5, 5) if d == 0 else (0, 0, 5, 5))
        x = sum(w[k] * pad.narrow(d, k, size) for k in range(11))
    return x


def _loss64(a, b):
    """(0.8 mean|a - b| + 0.2 (1 - mean SSIM), [L1, SSIM])."""
    w = _window()
    ma, mb = _blur64(a, w), _blur64(b, w)
    saa, sbb, sab = (_blur64(x * y, w) - u * v
                     for x, y, u, v in ((a, a, ma, ma), (b, b, mb, mb), (a, b, ma, mb)))
    c1, c2 = 0.01 ** 2, 0.03 ** 2
    s = ((2 * ma * mb + c1) * (2 * sab + c2)
         / ((ma * ma + mb * mb + c1) * (saa + sbb + c2))).mean()
    l1 = (a - b).abs().mean()
    return 0.8 * l1 + 0.2 * (1 - s), torch.stack([l1, s]).detach()


# Real spherical harmonics to degree 3.
_C2 = (1.0925484305920792, 0.31539156525252005, 0.5462742152960396)
_C3 = (0.5900435899266435, 2.890611442640554, 0.4570457994644658, 0.3731763325901154,
       1.445305721320277)


def _colours64(sh, dirs):
    x, y, z = dirs.unbind(1)
    xx, yy, zz = x * x, y * y, z * z
    basis = [torch.full_like(x, 0.28209479177387814)]
    if sh.shape[1] > 1:
        c = 0.4886025119029199
        basis += [-c * y, c * z, -c * x, _C2[0] * x * y, -_C2[0] * y * z,
                  _C2[1] * (2 * zz - xx - yy), -_C2[0] * x * z, _C2[2] * (xx - yy),
                  -_C3[0] * y * (3 * xx - yy), _C3[1] * x * y * z,
                  -_C3[2] * y * (4 * zz - xx - yy), _C3[3] * z * (2 * zz - 3 * xx - 3 * yy),
                  -_C3[2] * x * (4 * zz - xx - yy), _C3[4] * z * (xx - yy),
                  -_C3[0] * x * (xx - 3 * yy)]
    return ((torch.stack(basis, 1)[:, :, None] * sh).sum(1) + 0.5).clamp_min(0.0)


def _project64(means, quats, scales, opacity, sh, K, viewmat, W, H, filter_3d, antialias):
    """Screen-space Gaussians: uv, conic, colour and effective opacity
    (differentiable), depth and each one's box of tiles (empty if culled)."""
    fx, fy, cx, cy = (float(K[i, j]) for i, j in ((0, 0), (1, 1), (0, 2), (1, 2)))
    vm = viewmat.double().to(DEVICE)
    R = vm[:3, :3]
    if filter_3d is not None:
        s2 = scales * scales
        wide = s2 + filter_3d.double()[:, None] ** 2
        opacity = opacity * (s2.prod(1) / wide.prod(1)).clamp(0.0, 1.0).sqrt()
        scales = wide.sqrt()
    c = means @ R.T + vm[:3, 3]
    z = c[:, 2]
    zc = z.clamp_min(0.01)
    lx, ly = 1.3 * 0.5 * W / fx, 1.3 * 0.5 * H / fy
    tx, ty = (c[:, 0] / zc).clamp(-lx, lx) * zc, (c[:, 1] / zc).clamp(-ly, ly) * zc
    M = R @ _rotation64(quats) * scales[:, None, :]
    row0 = (fx / zc)[:, None] * M[:, 0] - (fx * tx / (zc * zc))[:, None] * M[:, 2]
    row1 = (fy / zc)[:, None] * M[:, 1] - (fy * ty / (zc * zc))[:, None] * M[:, 2]
    a0, b, c0 = (row0 * row0).sum(1), (row0 * row1).sum(1), (row1 * row1).sum(1)
    a, d = a0 + 0.3, c0 + 0.3
    det = a * d - b * b
    ds = det.clamp_min(1e-12)
    conic = torch.stack([d / ds, -b / ds, a / ds], 1)
    uv = torch.stack([fx * c[:, 0] / zc + cx, fy * c[:, 1] / zc + cy], 1)
    with torch.no_grad():
        mid = 0.5 * (a + d)
        radius = 3.0 * (mid + (mid * mid - ds).clamp_min(0).sqrt()).clamp_min(1e-12).sqrt()
        reach = (2.0 * torch.log((255.0 * opacity).clamp_min(1.0))).sqrt()
        rx, ry = torch.minimum(reach * a.sqrt(), radius), torch.minimum(reach * d.sqrt(), radius)
        u, v = uv[:, 0], uv[:, 1]
        valid = ((z > 0.01) & (z < 100.0) & (det > 1e-12) & (radius < max(W, H)) & (rx > 0)
                 & (ry > 0) & (u + rx > 0) & (u - rx < W) & (v + ry > 0) & (v - ry < H))
        tiles_x, tiles_y = -(-W // 16), -(-H // 16)
        box = [(t / 16).floor().clamp(0, m - 1).long()
               for t, m in ((u - rx, tiles_x), (u + rx, tiles_x), (v - ry, tiles_y),
                            (v + ry, tiles_y))]
    if antialias:
        det0 = (a0 * c0 - b * b).clamp_min(0.0)
        opacity = opacity * (det0 / ds).clamp(0.0, 1.0).sqrt()
    dirs = means + R.T @ vm[:3, 3]
    dirs = dirs / dirs.norm(dim=1, keepdim=True).clamp_min(1e-12)
    colour = _colours64(sh, dirs)
    return uv, conic, colour, opacity, z.detach(), valid, box


def _lists64(depth, valid, box, W, H):
    """(Gaussian ids by tile and depth, each tile's first entry)."""
    tiles_x, tiles_y = -(-W // 16), -(-H // 16)
    order = torch.argsort(depth, stable=True)
    order = order[valid[order]]
    x0, x1, y0, y1 = (t[order] for t in box)
    w = x1 - x0 + 1
    count = w * (y1 - y0 + 1)
    owner = torch.repeat_interleave(torch.arange(order.numel(), device=DEVICE), count)
    k = torch.arange(owner.numel(), device=DEVICE) - (torch.cumsum(count, 0) - count)[owner]
    w = w[owner]
    tile = ((y0[owner] + k // w) * tiles_x + x0[owner] + k % w).to(torch.int32)
    del k, w
    tile, perm = torch.sort(tile, stable=True)
    first = torch.searchsorted(tile, torch.arange(tiles_x * tiles_y + 1, device=DEVICE,
                                                  dtype=torch.int32))
    return order[owner[perm]], first


def _composite64(scr, ids, first, W, H, background, grad=None):
    """Front-to-back compositing of every tile. Without ``grad``: (rgb,
    alpha). With the loss's gradient to the blended image: the gradients of
    uv, conic, colour and opacity."""
    uv, conic, colour, opacity = (t.detach() for t in scr)
    tiles_x, tiles_y = -(-W // 16), -(-H // 16)
    n_tiles, chunk = tiles_x * tiles_y, 256
    bg = torch.tensor(background, dtype=torch.float64, device=DEVICE)
    px = torch.arange(256, device=DEVICE)
    length = first[1:] - first[:-1]
    by_length = torch.argsort(length, descending=True)

    def to_tiles(t):
        pad = torch.nn.functional.pad(t, (0, 0, 0, tiles_x * 16 - W, 0, tiles_y * 16 - H))
        return (pad.view(tiles_y, 16, tiles_x, 16, -1).transpose(1, 2)
                .reshape(n_tiles, 256, -1))

    def to_image(t):
        return (t.view(tiles_y, tiles_x, 16, 16, -1).transpose(1, 2)
                .reshape(tiles_y * 16, tiles_x * 16, -1)[:H, :W])

    grads = None
    if grad is None:
        rgb = torch.zeros(n_tiles, 256, 3, dtype=torch.float64, device=DEVICE)
        alpha = torch.zeros(n_tiles, 256, 1, dtype=torch.float64, device=DEVICE)
    else:
        g_tiles = to_tiles(grad)
        grads = [torch.zeros_like(t) for t in (uv, conic, colour, opacity)]
    for lo in range(0, n_tiles, 192):
        t = by_length[lo:lo + 192]
        x = ((t % tiles_x) * 16)[:, None] + px % 16 + 0.5
        y = ((t // tiles_x) * 16)[:, None] + px // 16 + 0.5
        inside = (x < W) & (y < H)
        longest = int(length[t].max())

        def entries(at):
            j = at + torch.arange(min(chunk, longest - at), device=DEVICE)
            present = j < length[t][:, None]
            return ids[torch.where(present, first[t][:, None] + j, 0)], present

        def weights(e, present, T):
            dx, dy = x[:, None] - uv[e, 0][..., None], y[:, None] - uv[e, 1][..., None]
            ca, cb, cc = (q[..., None] for q in conic[e].unbind(-1))
            power = -0.5 * (ca * dx * dx + cc * dy * dy) - cb * dx * dy
            gauss = power.exp()
            raw = opacity[e][..., None] * gauss
            a = raw.clamp(max=0.999)
            live = present[..., None] & (power <= 0) & (a >= 1.0 / 255.0)
            a = torch.where(live, a, 0.0)
            after = T[:, None] * torch.cumprod(1.0 - a, 1)
            before = torch.cat([T[:, None], after[:, :-1]], 1)
            a = torch.where(before >= 1e-4, a, 0.0)
            return a, before, after[:, -1], gauss, raw, dx, dy, (ca, cb, cc)

        def walk(visit):
            T = torch.where(inside, 1.0, 0.0).double()
            for at in range(0, longest, chunk):
                e, present = entries(at)
                a, before, T, *rest = weights(e, present, T)
                visit(e, a, before, rest)
                if not bool((T >= 1e-4).any()):
                    break

        if grad is None:
            def add(e, a, before, rest):
                w = (a * before).transpose(1, 2)
                rgb[t] += w @ colour[e].contiguous()
                alpha[t] += w.sum(2, keepdim=True)

            walk(add)
            continue
        g = g_tiles[t]
        total = torch.zeros(t.numel(), 256, dtype=torch.float64, device=DEVICE)

        def shade(e):
            # Each entry's colour over the background, against the gradient.
            return (colour[e] - bg) @ g.transpose(1, 2).contiguous()

        def measure(e, a, before, rest):
            total.add_((a * before * shade(e)).sum(1))

        walk(measure)
        passed = torch.zeros_like(total)

        def back(e, a, before, rest):
            gauss, raw, dx, dy, (ca, cb, cc) = rest
            q = shade(e)
            part = passed[:, None] + torch.cumsum(a * before * q, 1)
            passed.copy_(part[:, -1])
            d_a = before * q - (total[:, None] - part) / (1.0 - a)
            d_a = torch.where((a > 0) & (raw <= 0.999), d_a, 0.0)
            d_pow = d_a * raw
            rows = e.reshape(-1)

            def put(k, columns):
                v = torch.stack([c.sum(2) for c in columns], -1)
                grads[k].index_add_(0, rows, v.reshape(-1, len(columns)))

            put(0, (d_pow * (ca * dx + cb * dy), d_pow * (cb * dx + cc * dy)))
            put(1, (-0.5 * d_pow * dx * dx, -d_pow * dx * dy, -0.5 * d_pow * dy * dy))
            grads[2].index_add_(0, rows, ((a * before) @ g.contiguous()).reshape(-1, 3))
            grads[3].index_add_(0, rows, (d_a * gauss).sum(2).reshape(-1))

        walk(back)
    if grad is not None:
        return grads
    rgb = rgb + (1.0 - alpha).clamp_min(0.0) * bg
    return to_image(rgb), to_image(alpha)[..., 0]


def _exact_frame(case, seed):
    p, K, viewmat = _scene(case, seed)
    sh = p["sh_dc"] if case["degree"] == 0 else torch.cat([p["sh_dc"], p["sh_rest"]], 1)
    W, H = case["width"], case["height"]
    # The activations are the viewer's own, in float32.
    scr = _project64(p["means"].double(), p["quats"].double(),
                     torch.exp(p["log_scales"]).double(), torch.sigmoid(p["logit_opac"]).double(),
                     sh.double(), K, viewmat, W, H, None, case["antialias"])
    rgb, alpha = _composite64(scr[:4], *_lists64(*scr[4:], W, H), W, H, (0.0, 0.0, 0.0))
    return {"rgb": rgb, "alpha": alpha}


def _exact_train(case, seed):
    p, K, viewmat = _scene(case, seed)
    W, H, mip = case["width"], case["height"], bool(case.get("mip"))
    x = {k: p[k].double().requires_grad_(True) for k in RENDER_KEYS}
    scr = _project64(x["means"], x["quats"], x["log_scales"].exp(), torch.sigmoid(x["logit_opac"]),
                     torch.cat([x["sh_dc"], x["sh_rest"]], 1), K, viewmat, W, H,
                     _filter_sizes(case, seed, K) if mip else None, mip)
    lists = _lists64(*scr[4:], W, H)
    background = (1.0, 1.0, 1.0) if case.get("white") else (0.0, 0.0, 0.0)
    rgb, _ = _composite64(scr[:4], *lists, W, H, background)
    image = rgb.requires_grad_(True)
    loss, _ = _loss64(image, _target(case, seed).double())
    loss.backward()
    grads = _composite64(scr[:4], *lists, W, H, background, grad=image.grad)
    torch.autograd.backward(scr[:4], grads)
    out = {"rgb": rgb.detach(), "loss": loss.detach()}
    grads = {k: t.grad for k, t in x.items()}
    if case["kind"] == "train":
        return {**out, "grad": grads}
    return {**out, **_adam64(p, grads, _moments(case["n"], seed, 1e-8))}
