"""Performance cases of the rasterizer: what its users have it do, through its public API.

A case is one view: a rendering (``mode`` "render", under ``torch.no_grad``: a viewer, an
evaluation) or a training step's rasterization (``mode`` "train": the forward and the gradients of
every leaf for given upstream image gradients).  Scenes are synthetic, drawn on the GPU from the
seed with the distributions of the benchmark configurations (``gswarp_amd/configs.py``):

  box     means in a box in front of the camera, small splats: a small object, few tiles in use;
  cloud   normally distributed means around an orbiting camera's target: an ordinary scene;
  splats  the cloud with one splat in ten about 30 times larger: heavy overlap, tens of tiles a
          splat, opaque images;
  slab    many mid-sized splats in a thin slab filling the middle of a small image, with given RGB
          colours: long lists on few tiles.
"""

from __future__ import annotations

import math

import torch

from gswarp_amd import configs, rasterizer, rasterizer_flow
from gswarp_amd.methods import mip_3dgs

FLOW_TOPK = 20  # the flow API's default number of recorded Gaussians per pixel
MIP_VARIANCE = 0.3

# family -> (mean linear scale of a splat, its squared spread factor, mean distance, share in view)
_FOOTPRINT = {
    "box": (math.exp(-4.5), math.exp(2 * 0.5 ** 2), 4.0, 1.0),
    "cloud": (math.exp(-5.0), math.exp(2 * 0.7 ** 2), 6.0, 0.8),
    "splats": (math.exp(-2.0) * math.sqrt(0.1), math.exp(2 * 0.5 ** 2), 6.0, 0.8),
    "slab": (0.0425, 1.06, 2.5, 1.0),
}


def _case(name, family, count, width, height, mode, *, api="standard", degree=3, coeffs=16, upstream="color"):
    """One case.  ``coeffs``: stored SH coefficients per channel (0: given RGB colours);
    ``degree``: the active SH degree; ``api``: standard, flow, mip (the Mip filter's variance) or
    cov (precomputed 3D covariances instead of scales and rotations); ``upstream``: the outputs
    that bring gradients (color, or color + depth + alpha)."""
    case = {"family": family, "count": count, "width": width, "height": height, "mode": mode, "api": api,
            "degree": degree, "coeffs": coeffs, "upstream": upstream}
    return {"name": name, **case} if name else case


def listed():
    return [
        # A preview of a small object: the smallest call, latency and launches.
        _case("preview_10k_256", "box", 10_000, 256, 256, "render", degree=0, coeffs=1),
        # The first thousands of steps of a training, before densification.
        _case("train_100k_800", "box", 100_000, 800, 800, "train"),
        # The same on an ordinary scene at the usual size of synthetic training sets.
        _case("train_300k_800", "cloud", 300_000, 800, 800, "train"),
        # A viewer's frame of a trained scene.
        _case("view_1m_1080p", "cloud", 1_000_000, 1920, 1080, "render"),
        # A training step late in a run, with depth and alpha losses: the benchmark's default.
        _case("train_1m_1080p", "cloud", 1_000_000, 1920, 1080, "train", upstream="all"),
        # The largest: a large scene with big background splats.
        _case("train_splats_5m_1080p", "splats", 5_000_000, 1920, 1080, "train", upstream="all"),
        # A frame of a scene with big splats at a lower resolution.
        _case("view_splats_500k_720p", "splats", 500_000, 1280, 720, "render"),
        # Training with optical flow: the recorded Gaussians of every pixel.
        _case("flow_1m_720p", "cloud", 1_000_000, 1280, 720, "train", api="flow"),
        # The reference's published microbenchmark workloads: given RGB colours, small images.
        _case("slab_256k_384", "slab", 262_144, 384, 384, "train", coeffs=0, degree=0, upstream="all"),
        _case("slab_1m_640", "slab", 1_048_576, 640, 640, "train", coeffs=0, degree=0, upstream="all"),
        # Mip-Splatting training on photographs of odd size, early enough that only the first SH
        # band of the sixteen stored coefficients is active.
        _case("mip_250k_979x546", "cloud", 250_000, 979, 546, "train", api="mip", degree=1),
        # A deformation model that computes covariances and colours itself, small odd images.
        _case("cov_60k_487x273", "cloud", 60_000, 487, 273, "train", api="cov", coeffs=0, degree=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["box", "cloud", "cloud", "cloud", "splats", "slab"])
    mode = rng.choice(["render", "train", "train"])
    upstream = rng.choice(["color", "all"])
    degree = rng.choice([0, 1, 2, 3, 3, 3])
    coeffs = rng.choice([16, 16, 16, 16, 0, (degree + 1) ** 2])
    api = "standard"
    if family == "slab":
        count, width = _log_int(rng, 30_000, 1_200_000), _log_int(rng, 200, 700)
        height = min(700, max(200, int(width * rng.uniform(0.7, 1.4))))
        coeffs = 0
    elif family == "box":
        count, width = _log_int(rng, 5_000, 400_000), _log_int(rng, 200, 1000)
        height = int(width * rng.uniform(0.6, 1.2))
    else:
        count = _log_int(rng, 20_000, 2_000_000)
        width = _log_int(rng, 320, 1920)
        height = int(width * rng.uniform(0.5, 0.8))
        if family == "cloud":
            api = rng.choice(["standard", "standard", "standard", "flow", "mip", "cov"])
    if coeffs == 0:
        degree = 0
    return _case(None, family, count, width, height, mode, api=api, degree=degree, coeffs=coeffs, upstream=upstream)


def _camera(case, seed):
    width, height = case["width"], case["height"]
    if case["family"] == "slab":
        eye = torch.eye(4)
        return {"width": width, "height": height, "tanfovx": 1.0, "tanfovy": 1.0, "viewmatrix": eye,
                "projmatrix": eye.clone(), "campos": torch.zeros(3)}
    if case["family"] == "box":
        fovx = math.radians(60.0 if case["mode"] == "render" else 50.0)
        fovy = 2.0 * math.atan(math.tan(fovx / 2.0) * height / width)
        pose = torch.eye(4, dtype=torch.float64) if case["mode"] == "render" else configs.look_at((0.0, 0.0, -4.0))
        return configs.camera(width, height, fovx, fovy, pose)
    spec = configs.ConfigSpec(2, case["count"], width, height, case["degree"], True)
    return configs.orbit_camera(spec, seed, 0)


def _inputs(case, seed):
    """The scene's tensors on the GPU, all float32, from the seed alone."""
    device = torch.device("cuda:0")
    g = torch.Generator(device=device).manual_seed(seed * 7919 + 17)
    n, family, coeffs = case["count"], case["family"], case["coeffs"]
    height, width = case["height"], case["width"]

    def normal(*shape):
        return torch.randn(shape, generator=g, device=device)

    def uniform(lo, hi, *shape):
        return torch.rand(shape, generator=g, device=device) * (hi - lo) + lo

    bg = torch.zeros(3, device=device)
    if family == "slab":
        means = torch.cat([uniform(-0.65, 0.65, n, 2), uniform(2.0, 3.0, n, 1)], 1)
        scales = uniform(0.025, 0.06, n, 3)
        rotations = torch.zeros(n, 4, device=device)
        rotations[:, 0] = 1.0
        opacities = uniform(0.1, 0.9, n, 1)
        bg = torch.tensor((0.05, 0.15, 0.25), device=device)
    else:
        if family == "box":
            means = torch.cat([uniform(-1.0, 1.0, n, 2), uniform(2.0, 6.0, n, 1)], 1)
            log_scales = normal(n, 3) * 0.5 - 4.5
        else:
            means = normal(n, 3) * torch.tensor((3.0, 1.5, 3.0), device=device).sqrt()
            if family == "splats":
                large = uniform(0.0, 1.0, n, 1) < 0.1
                log_scales = normal(n, 3) * 0.5 + torch.where(large, -2.0, -5.5)
            else:
                log_scales = normal(n, 3) * 0.7 - 5.0
        scales = log_scales.exp()
        rotations = torch.nn.functional.normalize(normal(n, 4), dim=1)
        opacities = torch.sigmoid(normal(n, 1) + (1.0 if family == "splats" else 0.0))
    leaves = {"means3D": means, "means2D": torch.zeros(n, 3, device=device), "opacities": opacities}
    if coeffs:
        leaves["shs"] = torch.cat([normal(n, 1, 3) * 0.3, normal(n, coeffs - 1, 3) * 0.05], 1)
    else:
        leaves["colors_precomp"] = uniform(0.0, 1.0, n, 3)
    if case["api"] == "cov":
        leaves["cov3D_precomp"] = _upper(_covariance(scales, rotations)).contiguous()
    else:
        leaves["scales"], leaves["rotations"] = scales, rotations
    upstream = [normal(3, height, width)]
    if case["upstream"] == "all":
        upstream += [normal(1, height, width), normal(1, height, width)]
    return {k: v.contiguous() for k, v in leaves.items()}, bg, upstream


def prepare(case, seed):
    """The model's leaves, the view's rasterizer settings and the loss's image gradients."""
    leaves, bg, upstream = _inputs(case, seed)
    device = bg.device
    cam = _camera(case, seed)
    fields = dict(image_height=cam["height"], image_width=cam["width"], tanfovx=cam["tanfovx"],
                  tanfovy=cam["tanfovy"], bg=bg, scale_modifier=1.0, viewmatrix=cam["viewmatrix"].to(device),
                  projmatrix=cam["projmatrix"].to(device), sh_degree=case["degree"],
                  campos=cam["campos"].to(device), prefiltered=False, auto_tune=False, auto_tune_verbose=False)
    if case["api"] == "flow":
        make, settings = rasterizer_flow.GaussianRasterizer, rasterizer_flow.GaussianRasterizationSettings(**fields)
    elif case["api"] == "mip":
        make = mip_3dgs.MipGaussianRasterizer
        settings = mip_3dgs.MipGaussianRasterizationSettings(**fields, filter_variance=MIP_VARIANCE)
    else:
        make, settings = rasterizer.GaussianRasterizer, rasterizer.GaussianRasterizationSettings(**fields)
    train = case["mode"] == "train"
    for leaf in leaves.values():
        leaf.requires_grad_(train)
    return {"make": make, "settings": settings, "leaves": leaves, "upstream": upstream, "train": train,
            "flow": case["api"] == "flow"}


def _forward(state):
    leaves = state["leaves"]
    out = state["make"](state["settings"])(**leaves)
    if state["flow"]:
        names = ("color", "radii", "depth", "alpha", "proj_2D", "conic_2D", "conic_2D_inv", "gs_per_pixel",
                 "weight_per_gs_pixel", "x_mu")
        return dict(zip(names, out))
    color, radii, meta = out
    return {"color": color, "radii": radii, **meta._asdict()}


def run(state):
    """One pass: the rasterizer's outputs, and in training the gradient of every leaf."""
    if not state["train"]:
        with torch.no_grad():
            return _forward(state)
    out = _forward(state)
    losses = [out[k] for k in ("color", "depth", "alpha")[:len(state["upstream"])]]
    leaves = state["leaves"]
    grads = torch.autograd.grad(losses, list(leaves.values()), state["upstream"])
    result = {k: v.detach() for k, v in out.items()}
    result.update({f"grad_{k}": v for k, v in zip(leaves, grads)})
    return result


def work(case):
    """Inputs read once, outputs written once; per Gaussian about 500 operations forward and 900
    backward, per blended pixel about 25 and 60.  Blended pixels: the area in which a splat's alpha
    passes 1/255, bounded by 40 layers a pixel, where an image of such splats is opaque."""
    n, pixels = case["count"], case["width"] * case["height"]
    train = case["mode"] == "train"
    leaf = 3 + 1 + (3 * case["coeffs"] if case["coeffs"] else 3) + (6 if case["api"] == "cov" else 7)
    words = n * (leaf + 9) + 5 * pixels
    if case["api"] == "flow":
        words += 4 * FLOW_TOPK * pixels
    if train:
        words += n * (leaf + 3) + pixels * (5 if case["upstream"] == "all" else 3)
    scale, spread, distance, share = _FOOTPRINT[case["family"]]
    focal = case["width"] / 2.0 if case["family"] == "slab" else case["width"] * 0.9
    area = math.pi * 2.0 * math.log(0.5 * 255.0) * (0.3 + spread * (scale * focal / distance) ** 2)
    blended = min(n * share * area, 40.0 * pixels)
    flops = n * (1400.0 if train else 500.0) + blended * (85.0 if train else 25.0)
    return {"bytes": 4.0 * words, "flops": flops}


def tolerance(case):
    """Four times the largest error against ``exact`` seen over the listed and forty drawn cases.

    Images differ by up to 4e-5, from blend decisions (alpha >= 1/255) that rounding turns.
    Gradients differ by up to 1.9e-3: the backward divides by the transmittance 1 - alpha, which for
    an opaque pixel is a float32 difference near 1e-4.  The float atomics' order alone gives 7e-5.
    (The flow API's recorded slots differ by 8e-3: one turned decision shifts all later slots of
    its pixel.  They are held to the same bound, being the same in every run.)"""
    return {"rel": 6.0e-3 if case["mode"] == "train" else 1.6e-4}


# --- the same view in 64 bits, in plain torch ---------------------------------------------------

_SH1 = 0.4886025119029199
_SH2 = (1.0925484305920792, -1.0925484305920792, 0.31539156525252005, -1.0925484305920792, 0.5462742152960396)
_SH3 = (-0.5900435899266435, 2.890611442640554, -0.4570457994644658, 0.3731763325901154, -0.4570457994644658,
        1.445305721320277, -0.5900435899266435)


def _covariance(scales, rotations):
    w, x, y, z = rotations.unbind(1)
    rot = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                       2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                       2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], 1).reshape(-1, 3, 3)
    m = rot * scales[:, None, :]
    return (m[:, :, None, :] * m[:, None, :, :]).sum(-1)


def _upper(sigma):
    return torch.stack([sigma[:, 0, 0], sigma[:, 0, 1], sigma[:, 0, 2], sigma[:, 1, 1], sigma[:, 1, 2],
                        sigma[:, 2, 2]], 1)


def _sh_color(means, campos, shs, degree):
    d = torch.nn.functional.normalize(means - campos, dim=1)
    x, y, z = d.unbind(1)
    basis = [torch.full_like(x, 0.28209479177387814)]
    if degree > 0:
        basis += [-_SH1 * y, _SH1 * z, -_SH1 * x]
    if degree > 1:
        basis += [_SH2[0] * x * y, _SH2[1] * y * z, _SH2[2] * (2 * z * z - x * x - y * y), _SH2[3] * x * z,
                  _SH2[4] * (x * x - y * y)]
    if degree > 2:
        basis += [_SH3[0] * y * (3 * x * x - y * y), _SH3[1] * x * y * z, _SH3[2] * y * (4 * z * z - x * x - y * y),
                  _SH3[3] * z * (2 * z * z - 3 * x * x - 3 * y * y), _SH3[4] * x * (4 * z * z - x * x - y * y),
                  _SH3[5] * z * (x * x - y * y), _SH3[6] * x * (x * x - 3 * y * y)]
    rgb = 0.5
    for k, b in enumerate(basis):
        rgb = rgb + b[:, None] * shs[:, k]
    return torch.clamp(rgb, min=0.0)


def _tile_lists(pix, cov, radius, opac, visible, gx, gy):
    """(tile, Gaussian) pairs of the visible Gaussians: the 16 x 16 tiles that meet both the square
    of the radius and (one pixel wider) the box in which alpha can reach 1/255."""
    reach = torch.sqrt(2.0 * torch.log(torch.clamp(255.0 * opac, min=1.0)))
    lo, hi = [], []
    for axis, (diag, size) in enumerate(((0, gx), (2, gy))):
        c = pix[:, axis]
        box = torch.ceil(reach * torch.sqrt(cov[:, diag])) + 1.0
        lo.append(torch.maximum(((c - radius) / 16).trunc(), ((c - box) / 16).trunc()).clamp(0, size).long())
        hi.append(torch.minimum(((c + radius + 15) / 16).trunc(), ((c + box + 15) / 16).trunc()).clamp(0, size).long())
    nx, ny = (hi[0] - lo[0]).clamp(min=0), (hi[1] - lo[1]).clamp(min=0)
    area = torch.where(visible & (reach > 0), nx * ny, torch.zeros_like(nx))
    gauss = torch.repeat_interleave(torch.arange(len(area), device=area.device), area)
    cell = torch.arange(len(gauss), device=area.device) - (torch.cumsum(area, 0) - area)[gauss]
    tile = (lo[1][gauss] + cell // nx[gauss]) * gx + lo[0][gauss] + cell % nx[gauss]
    return tile, gauss


def exact(case, seed):
    if case["family"] == "splats" and case["count"] > 1_000_000:
        return None  # about 2 * 10^10 pixel evaluations, each kept in 64 bits
    leaves, bg, upstream = _inputs(case, seed)
    cam = _camera(case, seed)
    with torch.enable_grad():
        return _exact_view(case, {k: v.double() for k, v in leaves.items()}, bg.double(),
                           [u.double() for u in upstream], cam)


def _exact_view(case, leaves, bg, upstream, cam):
    device = bg.device
    width, height, n = case["width"], case["height"], case["count"]
    train = case["mode"] == "train"
    leaves = {k: v.requires_grad_(train) for k, v in leaves.items()}
    means, opac = leaves["means3D"], leaves["opacities"].reshape(-1)
    view, proj = cam["viewmatrix"].to(device).double(), cam["projmatrix"].to(device).double()
    tanx, tany = cam["tanfovx"], cam["tanfovy"]
    ones = torch.ones(n, 1, dtype=torch.float64, device=device)
    cam_pos = torch.cat([means, ones], 1) @ view
    hom = torch.cat([means, ones], 1) @ proj
    depth = cam_pos[:, 2]
    ndc = hom[:, :2] / (hom[:, 3:] + 1.0e-7)
    size = torch.tensor((width, height), dtype=torch.float64, device=device)
    pix = ((ndc + 1.0) * size - 1.0) * 0.5
    sigma = leaves.get("cov3D_precomp")
    if sigma is None:
        sigma = _upper(_covariance(leaves["scales"], leaves["rotations"]))
    sigma = sigma[:, [0, 1, 2, 1, 3, 4, 2, 4, 5]].reshape(-1, 3, 3)
    jac = []
    for axis, (tan, extent) in enumerate(((tanx, width), (tany, height))):
        focal = extent / (2.0 * tan)
        ratio = cam_pos[:, axis] / depth
        t = torch.clamp(ratio, -1.3 * tan, 1.3 * tan) * depth
        t = torch.where(ratio.abs() > 1.3 * tan, t.detach(), t)  # a clamped coordinate is a constant
        jac.append((focal / depth)[:, None] * view[:3, axis] - (focal * t / (depth * depth))[:, None] * view[:3, 2])
    sx = (sigma * jac[0][:, None, :]).sum(-1)
    sy = (sigma * jac[1][:, None, :]).sum(-1)
    blur = 0.3 + (MIP_VARIANCE if case["api"] == "mip" else 0.0)
    cov = torch.stack([(sx * jac[0]).sum(-1) + blur, (sx * jac[1]).sum(-1), (sy * jac[1]).sum(-1) + blur], 1)
    rgb = leaves["colors_precomp"] if case["coeffs"] == 0 else _sh_color(
        means, cam["campos"].to(device).double(), leaves["shs"], case["degree"])

    with torch.no_grad():
        a, b, c = cov.unbind(1)
        base_a, base_c = a - (blur - 0.3), c - (blur - 0.3)
        mid, det = 0.5 * (base_a + base_c), base_a * base_c - b * b
        radius = torch.ceil(3.0 * torch.sqrt(mid + torch.sqrt(torch.clamp(mid * mid - det, min=0.1))))
        gx, gy = (width + 15) // 16, (height + 15) // 16
        lo = ((pix - radius[:, None]) / 16).trunc().clamp(min=0)
        hi = ((pix + radius[:, None] + 15) / 16).trunc().clamp(min=0)
        grid = torch.tensor((gx, gy), dtype=torch.float64, device=device)
        lo, hi = torch.minimum(lo, grid), torch.minimum(hi, grid)
        visible = (depth > 0.2) & (det.abs() > 1.0e-7) & ((hi - lo) > 0).all(1)
        det = a * c - b * b
        if case["api"] == "mip":
            lam = 0.5 * (a + c) + torch.sqrt(torch.clamp(0.25 * (a - c) ** 2 + b * b, min=0.0))
            radius = torch.ceil(3.0 * torch.sqrt(torch.clamp(lam, min=0.1)))
        conic = torch.stack([c, -b, a], 1) / det[:, None]
        tile, gauss = _tile_lists(pix, cov, radius, opac, visible, gx, gy)
        order = torch.argsort(depth[gauss].float(), stable=True)
        order = order[torch.argsort(tile[order], stable=True)]
        lists = gauss[order]
        lengths = torch.bincount(tile, minlength=gx * gy)
        del tile, gauss, order
        flow = case["api"] == "flow"
        result, grads = _exact_blend(lists, lengths, pix, conic, opac, rgb, depth, bg,
                                     upstream if train else None, width, height, FLOW_TOPK if flow else 0)
        keep = visible[:, None]
        out = {"color": result["color"], "radii": None, "depth": result["depth"], "alpha": result["alpha"],
               "proj_2D": torch.where(keep, pix, 0.0), "conic_2D": torch.where(keep, conic, 0.0),
               "conic_2D_inv": torch.where(keep, cov, 0.0)}
        if flow:
            out.update(gs_per_pixel=None, weight_per_gs_pixel=result["weight"], x_mu=result["x_mu"])
        if not train:
            return out
        # The gradients of the means and conics on the image enter the chain twice with the flow API.
        twice = 2.0 if flow else 1.0
        grad_pix, grad_conic = twice * grads["pix"], twice * grads["conic"]
        inv2 = 1.0 / (det * det + 1.0e-7)
        t0, t1, t2 = grad_conic.unbind(1)
        grad_cov = torch.stack([inv2 * (-c * c * t0 + 2 * b * c * t1 - b * b * t2),
                                2 * inv2 * (b * c * t0 - (a * c + b * b) * t1 + a * b * t2),
                                inv2 * (-a * a * t2 + 2 * a * b * t1 - b * b * t0)], 1)
        # what no pixel blends adds nothing (behind the camera the chain need not even be finite)
        grad_cov = torch.where(visible[:, None], grad_cov, 0.0)
    used = [k for k in leaves if k != "means2D"]
    leaf_grads = torch.autograd.grad([pix, cov, depth, rgb, opac], [leaves[k] for k in used],
                                     [grad_pix, grad_cov, grads["depth"], grads["rgb"], grads["opac"]])
    out.update({f"grad_{k}": g for k, g in zip(used, leaf_grads)})
    means2d = torch.zeros(n, 3, dtype=torch.float64, device=device)
    means2d[:, :2] = grads["pix"] * size * 0.5
    out["grad_means2D"] = means2d
    return out


def _exact_blend(lists, lengths, pix, conic, opac, rgb, depth, bg, upstream, width, height, top_k):
    """Front-to-back blend of every tile's list, and with ``upstream`` its gradients to the
    Gaussians' image quantities (conic's as half its matrix's: the off-diagonal once)."""
    device, f64 = pix.device, dict(dtype=torch.float64, device=pix.device)
    gx = (width + 15) // 16
    n = pix.shape[0]
    padded_h, padded_w = (height + 15) // 16 * 16, gx * 16
    image = torch.zeros(5, padded_h * padded_w, **f64)
    image[:3] = bg[:, None]
    flow = torch.zeros(3, max(top_k, 1), padded_h * padded_w, **f64) if top_k else None
    up = torch.zeros(5, padded_h, padded_w, **f64)
    if upstream is not None:
        up[:3, :height, :width] = upstream[0]
        for k, u in enumerate(upstream[1:]):
            up[3 + k, :height, :width] = u[0]
    up = up.reshape(5, -1)
    grads = torch.zeros(n, 10, **f64)  # x, y, conic 3, opacity, r, g, b, depth
    features = torch.cat([rgb, depth[:, None], torch.ones(n, 1, **f64)], 1)
    starts = torch.cumsum(lengths, 0) - lengths
    cell = torch.arange(256, device=device)
    by_length = torch.argsort(lengths, descending=True)
    sizes = lengths[by_length].tolist()
    at = 0
    while at < len(sizes) and sizes[at] > 0:
        longest = sizes[at]
        take = max(1, min(len(sizes) - at, (1 << 25) // (256 * longest)))
        tiles = by_length[at:at + take]
        at += take
        slot = torch.arange(longest, device=device)
        present = slot < lengths[tiles][:, None]
        ids = lists[torch.where(present, starts[tiles][:, None] + slot, 0)]  # (tiles, list)
        px = (tiles % gx)[:, None] * 16 + cell % 16
        py = torch.div(tiles, gx, rounding_mode="floor")[:, None] * 16 + cell // 16
        where = py * padded_w + px  # (tiles, 256)
        inside = (px < width) & (py < height)
        dx = pix[ids, 0][:, :, None] - px[:, None, :]
        dy = pix[ids, 1][:, :, None] - py[:, None, :]
        ca, cb, cc = (conic[ids, k][:, :, None] for k in range(3))
        o = opac[ids][:, :, None]
        power = -0.5 * (ca * dx * dx + cc * dy * dy) - cb * dx * dy
        gauss = torch.exp(power)
        alpha = torch.clamp(o * gauss, max=0.99)
        alpha = torch.where(present[:, :, None] & inside[:, None, :] & (power <= 0.0) & (alpha >= 1.0 / 255.0),
                            alpha, 0.0)
        behind = torch.cumprod(1.0 - alpha, 1)
        alpha = torch.where(behind >= 1.0e-4, alpha, 0.0)
        behind = torch.cumprod(1.0 - alpha, 1)
        front = torch.cat([torch.ones_like(behind[:, :1]), behind[:, :-1]], 1)
        weight = alpha * front
        f = features[ids]  # (tiles, list, 5)
        sums = torch.bmm(f.transpose(1, 2).contiguous(), weight).transpose(0, 1)  # (5, tiles, 256)
        sums[:3] += behind[:, -1] * bg[:, None, None]
        image[:, where.reshape(-1)] = sums.reshape(5, -1)
        if top_k:
            rank = torch.cumsum((alpha > 0).int(), 1) - 1
            t, k, p = torch.nonzero((alpha > 0) & (rank < top_k), as_tuple=True)
            for plane, value in enumerate((weight, dx, dy)):
                flow[plane, rank[t, k, p].long(), where[t, p]] = value[t, k, p]
        if upstream is None:
            continue
        u = up[:, where.reshape(-1)].reshape(5, len(tiles), 256).transpose(0, 1).contiguous()
        fu = torch.bmm(f, u)
        wfu = weight * fu
        rest = torch.flip(torch.cumsum(torch.flip(wfu, [1]), 1), [1]) - wfu
        rest = rest + (behind[:, -1] * (bg[:, None] * u[:, :3]).sum(1))[:, None, :]
        v = torch.where(alpha > 0, gauss * (front * fu - rest / (1.0 - alpha)), 0.0)
        vdx, vdy = v * dx, v * dy
        o, ca, cb, cc = o[..., 0], ca[..., 0], cb[..., 0], cc[..., 0]
        mx, my = vdx.sum(2), vdy.sum(2)
        part = torch.stack([-o * (ca * mx + cb * my), -o * (cc * my + cb * mx), -0.5 * o * (vdx * dx).sum(2),
                            -0.5 * o * (vdx * dy).sum(2), -0.5 * o * (vdy * dy).sum(2), v.sum(2)], 2)
        part = torch.cat([part, torch.bmm(weight, u[:, :4].transpose(1, 2).contiguous())], 2)
        grads.index_add_(0, ids[present], part[present])
    image = image.reshape(5, padded_h, padded_w)[:, :height, :width]
    result = {"color": image[:3].contiguous(), "depth": image[3:4].contiguous(), "alpha": image[4:].contiguous()}
    if top_k:
        flow = flow.reshape(3, top_k, padded_h, padded_w)[..., :height, :width]
        result.update(weight=flow[0].contiguous(), x_mu=flow[1:].contiguous())
    return result, {"pix": grads[:, :2], "conic": grads[:, 2:5], "opac": grads[:, 5], "rgb": grads[:, 6:9],
                    "depth": grads[:, 9]}
