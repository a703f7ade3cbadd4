"""Performance cases of the gs3d rasterizer, through its public entry points.

A case is a dict of plain values; ``kind`` names the call that a program makes:

  train    gs3d.rasterize and its backward from upstream image gradients: one
           optimisation step without the optimiser (SH colours, plain features
           or features with an extra channel; absolute gradients, camera
           gradients, several cameras, batches of scenes, every tile mode)
  gsplat   gs3d.gsplat.rasterization with that signature's defaults (packed
           metadata) and its backward
  render   gs3d.rasterize without gradients: novel-view rendering, with
           ``requests`` contribution statistics when a program scores
           Gaussians for densification or pruning
  staged   gs3d.ops: prepare_gaussians, bin_and_sort, rasterize_to_pixels and
           the backward through all three
  sh       gs3d.ops.spherical_harmonics and its backward

Scenes: ``uniform`` (a box in front of the camera), ``ball``, ``clusters`` (64
clusters, cameras on a ring around them) and ``fanout`` (5% of the Gaussians
are large and reach thousands of tiles).  Scene and cameras both come from the
seed; upstream gradients are normal.
"""

import math

import torch

from dsl_splat_amd import gs3d
from dsl_splat_amd.cameras import PinholeCamera
from dsl_splat_amd.gs3d import gsplat, ops
from dsl_splat_amd.statistics import MaskedContributionCount, WeightedContributionSum

_DEFAULTS = dict(batch=0, cameras=1, channels=3, sh_degree=-1, extra=False, absgrad=False, pose=False,
                 background=False, tile_mode="radius", requests=0, scene="ball")


def _case(kind, n, width, height, **options):
    return dict(_DEFAULTS, kind=kind, n=n, width=width, height=height, **options)


def listed():
    return [
        # The smallest optimisation step: launches and host work count.
        dict(_case("train", 10_000, 256, 256, scene="uniform"), name="train_10k_256"),
        # Feed-forward models: a batch of small scenes, each seen by two cameras.
        dict(_case("train", 4_096, 128, 128, batch=4, cameras=2, scene="uniform"), name="train_batch4_4k_128"),
        # One mid-size scene per step with the densification signal.
        dict(_case("train", 500_000, 1280, 720, sh_degree=3, absgrad=True), name="train_500k_720p"),
        # The largest step: four full-HD views of a 3M-Gaussian scene.
        dict(_case("train", 3_000_000, 1920, 1080, cameras=4, sh_degree=3, scene="clusters"), name="train_3m_4x1080p"),
        # Feature distillation: 32 channels and the camera depth as an extra one.
        dict(_case("train", 1_000_000, 1600, 1200, channels=32, extra=True), name="train_feat32_1m_1600x1200"),
        # Pose refinement on a scene with very large Gaussians.
        dict(_case("train", 2_000_000, 1920, 1080, sh_degree=3, absgrad=True, pose=True, scene="fanout"),
             name="train_pose_2m_1080p"),
        # Exact tile lists on two cameras.
        dict(_case("train", 1_000_000, 1920, 1080, cameras=2, sh_degree=3, tile_mode="accutile", scene="clusters"),
             name="train_accutile_1m_2x1080p"),
        # Another library's trainer, early in its SH schedule, odd sizes, a background.
        dict(_case("gsplat", 300_001, 801, 601, cameras=3, sh_degree=1, background=True, scene="clusters"),
             name="gsplat_packed_300k_3x801x601"),
        # A viewer: one frame, no gradients.
        dict(_case("render", 1_000_000, 1920, 1080, sh_degree=3, background=True), name="render_1m_1080p"),
        # Scoring Gaussians for densification: a masked count and a weighted sum.
        dict(_case("render", 400_000, 1237, 822, sh_degree=2, requests=2, scene="clusters"),
             name="render_statistics_400k_1237x822"),
        # The staged calls with a short feature vector, ragged sizes.
        dict(_case("staged", 77_777, 637, 421, channels=8, background=True), name="staged_78k_637x421"),
        # SH colours evaluated outside the rasterizer.
        dict(_case("sh", 1_000_000, 0, 0, sh_degree=3), name="sh3_1m"),
    ]


def _log_int(rng, lo, hi):
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return min(hi, max(lo, v + rng.randint(-3, 3)))


def draw(rng):
    kind = rng.choice(("train", "train", "train", "train", "gsplat", "render", "render", "staged", "sh"))
    if kind == "sh":
        return _case("sh", _log_int(rng, 1_000, 2_000_000), 0, 0, sh_degree=rng.randint(0, 3))
    n = _log_int(rng, 2_000, 1_500_000)
    width = _log_int(rng, 96, 1920)
    height = max(64, min(1200, int(width * rng.uniform(0.5, 1.0))))
    options = dict(scene=rng.choice(("uniform", "ball", "clusters")), background=rng.random() < 0.4,
                   tile_mode=rng.choice(("radius", "radius", "snugbox", "accutile")))
    if kind == "staged":
        return _case(kind, min(n, 400_000), width, height, channels=rng.choice((1, 3, 5, 8, 13)), **options)
    options["cameras"] = rng.choice((1, 1, 2, 3, 4)) if n * width * height < 4e11 else 1
    if kind == "train" and rng.random() < 0.3:
        options.update(channels=rng.choice((1, 3, 7, 16, 32, 40)), extra=rng.random() < 0.5)
    else:
        options["sh_degree"] = rng.randint(0, 3)
    if kind != "render":
        options.update(absgrad=rng.random() < 0.5, pose=rng.random() < 0.3)
    elif rng.random() < 0.5:
        options["requests"] = rng.choice((1, 2, 3))
    if kind == "train" and n < 20_000 and rng.random() < 0.3:
        options["batch"] = rng.choice((2, 3))
    return _case(kind, n, width, height, **options)


# --------------------------------------------------------------------------
# Inputs


def _look_at(eye, target=(0.0, 0.0, 0.0)):
    eye = torch.tensor(eye, dtype=torch.float64)
    z = torch.tensor(target, dtype=torch.float64) - eye
    z = z / z.norm()
    x = torch.linalg.cross(z, torch.tensor([0.0, 1.0, 0.0], dtype=torch.float64))
    x = x / x.norm()
    view = torch.eye(4, dtype=torch.float64)
    view[:3, :3] = torch.stack([x, torch.linalg.cross(z, x), z])
    view[:3, 3] = -view[:3, :3] @ eye
    return view.float()


def _uniform(g, shape, lo, hi):
    return torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _scene(case, g, n):
    """means, log scales, opacity logits, the cameras' distance and the focal
    length over the image width."""
    scene = case["scene"]
    if scene == "uniform":
        return _uniform(g, (n, 3), -1.0, 1.0), _uniform(g, (n, 3), -4.5, -2.5), _normal(g, n), 4.0, 1.0
    if scene == "ball":
        d = _normal(g, n, 3)
        means = d / d.norm(dim=-1, keepdim=True) * 1.5 * _uniform(g, (n, 1), 0.0, 1.0) ** (1.0 / 3.0)
        return means, _uniform(g, (n, 3), -5.0, -3.0), _normal(g, n), 4.0, 0.77
    if scene == "clusters":
        centres = _uniform(g, (64, 3), -2.0, 2.0)
        assign = torch.randint(0, 64, (n,), generator=g, device="cuda")
        return centres[assign] + 0.3 * _normal(g, n, 3), _uniform(g, (n, 3), -5.5, -3.0), 1.5 * _normal(g, n), 5.0, 0.73
    log_scales = _uniform(g, (n, 3), -7.0, -5.0)
    large = torch.randperm(n, generator=g, device="cuda")[:max(1, n // 20)]
    log_scales[large] = _uniform(g, (len(large), 3), -1.0, 0.0)
    return _uniform(g, (n, 3), -2.0, 2.0), log_scales, _normal(g, n), 5.0, 0.73


def _stack(items, batch):
    return torch.stack(items) if batch else items[0]


def prepare(case, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    n, width, height, cameras, batch = case["n"], case["width"], case["height"], case["cameras"], case["batch"]
    state = dict(case=case)
    rows = 16 if case["sh_degree"] >= 0 else 0

    def sh_coefficients():
        sh = 0.05 * _normal(g, n, rows, 3)
        sh[:, 0] *= 10.0
        return sh

    if case["kind"] == "sh":
        state.update(sh=sh_coefficients().requires_grad_(), dirs=_normal(g, n, 3).requires_grad_(),
                     upstream=_normal(g, n, 3))
        return state
    parts = {k: [] for k in ("means", "quats", "scales", "opacities", "colors", "viewmats", "Ks", "extra")}
    turn = torch.rand(max(1, batch), generator=torch.Generator().manual_seed(seed)).tolist()
    for b in range(max(1, batch)):
        means, log_scales, logits, distance, focal = _scene(case, g, n)
        angles = [2 * math.pi * (turn[b] + c / cameras) for c in range(cameras)]
        views = torch.stack([_look_at((distance * math.sin(a), 0.0, -distance * math.cos(a))) for a in angles]).cuda()
        K = torch.tensor([[focal * width, 0.0, width / 2], [0.0, focal * width, height / 2], [0.0, 0.0, 1.0]])
        parts["means"].append(means)
        parts["quats"].append(_normal(g, n, 4))
        parts["scales"].append(torch.exp(log_scales))
        parts["opacities"].append(torch.sigmoid(logits))
        parts["colors"].append(sh_coefficients() if rows else _uniform(g, (n, case["channels"]), 0.0, 1.0))
        parts["viewmats"].append(views)
        parts["Ks"].append(K.repeat(cameras, 1, 1).cuda())
        if case["extra"]:
            parts["extra"].append((means @ views[0, 2, :3] + views[0, 2, 3])[:, None])
    for name, items in parts.items():
        if items:
            state[name] = _stack(items, batch).contiguous()
    lead = ((batch,) if batch else ()) + (cameras, height, width)
    channels = 3 if rows else case["channels"]
    if case["background"]:
        state["background"] = torch.rand(((batch,) if batch else ()) + (cameras, channels), generator=g, device="cuda")
    if case["kind"] == "render":
        if case["requests"]:
            weights = torch.rand(lead, generator=g, device="cuda")
            state["statistics"] = [
                MaskedContributionCount("count", weights > 0.5),
                WeightedContributionSum("error", weights),
                MaskedContributionCount("edges", weights > 0.9),
            ][:case["requests"]]
        return state
    if case["kind"] == "staged":
        state["camera"] = PinholeCamera(state["viewmats"][0].contiguous(), state["Ks"][0].contiguous(), width, height)
        lead = (height, width)
    grads = ["means", "quats", "scales", "opacities", "colors"]
    if case["extra"]:
        grads.append("extra")
    if case["pose"]:
        grads.append("viewmats")
    for name in grads:
        state[name].requires_grad_()
    state["grads"] = grads
    state["upstream"] = [_normal(g, *lead, channels), _normal(g, *lead, 1)]
    if case["extra"]:
        state["upstream"].append(_normal(g, *lead, 1))
    return state


# --------------------------------------------------------------------------
# One pass


def _backward(state, outputs):
    torch.autograd.backward(outputs, state["upstream"])
    grads = {}
    for name in state["grads"]:
        grads[name] = state[name].grad
        state[name].grad = None
    return grads


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "sh":
        colors = ops.spherical_harmonics(state["sh"], state["dirs"], case["sh_degree"])
        colors.backward(state["upstream"])
        out = dict(colors=colors, sh=state["sh"].grad, dirs=state["dirs"].grad)
        state["sh"].grad = state["dirs"].grad = None
        return out if out["dirs"] is not None else dict(colors=colors, sh=out["sh"])
    if kind == "staged":
        geometry = ops.prepare_gaussians(state["means"], state["quats"], state["scales"], state["opacities"],
                                         state["camera"], tile_mode=case["tile_mode"])
        tiles = ops.bin_and_sort(geometry)
        background = state["background"][0] if case["background"] else None
        pixels = ops.rasterize_to_pixels(geometry, tiles, state["colors"], background)
        grads = _backward(state, [pixels.features, pixels.alpha])
        return dict(features=pixels.features, alpha=pixels.alpha, radii=geometry.radii, grads=grads)
    geometry = [state[k] for k in ("means", "quats", "scales", "opacities")]
    sh = case["sh_degree"] >= 0
    if kind == "gsplat":
        features, alpha, meta = gsplat.rasterization(
            *geometry, state["colors"], state["viewmats"], state["Ks"], case["width"], case["height"],
            sh_degree=case["sh_degree"] if sh else None, backgrounds=state.get("background"),
            absgrad=case["absgrad"], tile_mode=case["tile_mode"])
        grads = _backward(state, [features, alpha])
        # The trainer's densification state, from the packed rows.
        rows, ids = meta["means2d"], meta["gaussian_ids"]
        signal = rows.absgrad if case["absgrad"] else rows.grad
        moved = torch.zeros(case["n"], device="cuda").index_add_(0, ids, signal.norm(dim=-1))
        views = torch.zeros(case["n"], device="cuda").index_add_(0, ids, torch.ones_like(ids, dtype=torch.float32))
        return dict(features=features, alpha=alpha, grads=grads, moved=moved, views=views)
    colors = dict(sh_coeffs=state["colors"], sh_degree=case["sh_degree"]) if sh else dict(features=state["colors"])
    options = dict(backgrounds=state.get("background"), extra_features=state.get("extra"),
                   tile_mode=case["tile_mode"], **colors)
    if kind == "render":
        with torch.no_grad():
            result = gs3d.rasterize(*geometry, state["viewmats"], state["Ks"], case["width"], case["height"],
                                    statistics=state.get("statistics", ()), **options)
        return dict(features=result.features, alpha=result.alpha, radii=result.radii,
                    statistics=result.statistics)
    result = gs3d.rasterize(*geometry, state["viewmats"], state["Ks"], case["width"], case["height"],
                            absgrad=case["absgrad"], **options)
    meta = result.meta
    outputs = [result.features, result.alpha] + ([result.extra_features] if case["extra"] else [])
    grads = _backward(state, outputs)
    out = dict(features=result.features, alpha=result.alpha, radii=result.radii, grads=grads)
    if case["extra"]:
        out["extra"] = result.extra_features
    out["means2d_grad"] = meta["means2d"].grad
    if case["absgrad"]:
        out["absgrad"] = meta["means2d"].absgrad
    return out


# --------------------------------------------------------------------------
# Sizes and tolerances

# (pixel, Gaussian) pairs that a pixel blends before it is opaque, by scene.
_BLENDED = dict(uniform=22, ball=37, clusters=64, fanout=40)


def work(case):
    n, rows = case["n"], (case["sh_degree"] + 1) ** 2 if case["sh_degree"] >= 0 else 0
    colour = 3 * rows if rows else case["channels"]
    train = case["kind"] in ("train", "gsplat", "staged")
    if case["kind"] == "sh":
        return dict(bytes=4.0 * n * (2 * 48 + 12), flops=float(n * rows * 24))
    items, cameras = max(1, case["batch"]), case["cameras"]
    channels = (3 if rows else case["channels"]) + (1 if case["extra"] else 0) + 1
    pixels = cameras * case["width"] * case["height"]
    gaussian = n * (11 + colour + (1 if case["extra"] else 0)) * (2 if train else 1)
    # radii, and a training program's screen gradients
    screen = cameras * n * (1 + (2 if train else 0) + (2 if train and case["absgrad"] else 0) + case["requests"])
    image = pixels * (channels * (2 if train else 1) + case["requests"])
    blended = pixels * min(_BLENDED[case["scene"]], 1 + cameras * n // 64)
    flops = blended * ((24 + 2 * channels) + (train and 48 + 4 * channels)) + cameras * n * (250 + (train and 600))
    return dict(bytes=4.0 * items * (gaussian + screen + image), flops=float(items * flops))


def tolerance(case):
    # 32-bit sums throughout.  Images hold one fixed order of operations per
    # pixel; gradients are sums over pixels in any order: two passes over the
    # same inputs differ by up to 1.5e-6 (largest 2.7e-4 of the root mean
    # square), and by 4e-6 with camera gradients, which are sums over all
    # Gaussians that largely cancel.
    if case["pose"]:
        return dict(rel=2e-5, max=2e-3, differ=0.0)
    return dict(rel=1e-5, max=1.2e-3, differ=0.0)


# --------------------------------------------------------------------------
# The same results in 64 bits, in plain torch


class _Inverse(torch.autograd.Function):
    """(a, b, c) -> (c, -b, a) / det of a symmetric 2x2 matrix; original 3DGS
    takes the gradient with 1 / (det^2 + 1e-7)."""

    @staticmethod
    def forward(ctx, a, b, c):
        ctx.save_for_backward(a, b, c)
        det = a * c - b * b
        return c / det, -b / det, a / det

    @staticmethod
    def backward(ctx, ga, gb, gc):
        a, b, c = ctx.saved_tensors
        det = a * c - b * b
        s = 1.0 / (det * det + 1e-7)
        da = s * (-c * c * ga + b * c * gb - b * b * gc)
        db = s * (2 * b * c * ga - (a * c + b * b) * gb + 2 * a * b * gc)
        dc = s * (-b * b * ga + a * b * gb - a * a * gc)
        return da, db, dc


def _sh_colors(coefficients, directions, degree):
    x, y, z = (directions / directions.norm(dim=-1, keepdim=True)).unbind(-1)
    xx, yy, zz = x * x, y * y, z * z
    basis = [0.28209479177387814 * torch.ones_like(x)]
    if degree > 0:
        k = 0.4886025119029199
        basis += [-k * y, k * z, -k * x]
    if degree > 1:
        k = 1.0925484305920792
        basis += [k * x * y, -k * y * z, 0.31539156525252005 * (2 * zz - xx - yy), -k * x * z, k / 2 * (xx - yy)]
    if degree > 2:
        k, m = 0.5900435899266435, 0.4570457994644658
        basis += [-k * y * (3 * xx - yy), 2.890611442640554 * x * y * z, -m * y * (4 * zz - xx - yy),
                  0.3731763325901154 * z * (2 * zz - 3 * xx - 3 * yy), -m * x * (4 * zz - xx - yy),
                  1.445305721320277 * z * (xx - yy), -k * x * (xx - 3 * yy)]
    weights = torch.stack(basis, -1)
    return ((coefficients[:, :len(basis)] * weights[..., None]).sum(-2) + 0.5).clamp_min(0)


def _project(means, quats, scales, view, K, width, height, near):
    w, x, y, z = (quats / quats.norm(dim=-1, keepdim=True).clamp_min(1e-12)).unbind(-1)
    rotation = torch.stack([
        1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
        2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
        2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], -1).reshape(-1, 3, 3)
    fx, fy = K[0, 0], K[1, 1]
    p = means @ view[:3, :3].T + view[:3, 3]
    tz = p[:, 2]

    def clamped(v, limit):
        ratio = v / tz
        return torch.where(ratio.abs() > limit, (ratio.clamp(-limit, limit) * tz).detach(), v)

    tx, ty = clamped(p[:, 0], 1.3 * width / (2 * fx)), clamped(p[:, 1], 1.3 * height / (2 * fy))
    zero = torch.zeros_like(tz)
    J = torch.stack([fx / tz, zero, -fx * tx / tz ** 2, zero, fy / tz, -fy * ty / tz ** 2], -1).reshape(-1, 2, 3)
    half = J @ view[:3, :3] @ (rotation * scales[:, None, :])
    cov = half @ half.transpose(-1, -2)
    a, b, c = cov[:, 0, 0] + 0.3, cov[:, 0, 1], cov[:, 1, 1] + 0.3
    conic = torch.stack(_Inverse.apply(a, b, c), -1)
    center = torch.stack([fx * p[:, 0] / tz + K[0, 2] - 0.5, fy * p[:, 1] / tz + K[1, 2] - 0.5], -1)
    with torch.no_grad():
        mid = 0.5 * (a + c)
        radius = torch.ceil(3 * torch.sqrt(mid + torch.sqrt((mid * mid - (a * c - b * b)).clamp_min(0.1))))
        gx, gy = (width + 15) // 16, (height + 15) // 16
        lo = torch.stack([((center[:, k] - radius) / 16).trunc().clamp(0, m) for k, m in ((0, gx), (1, gy))], -1)
        hi = torch.stack([((center[:, k] + radius + 15) / 16).trunc().clamp(0, m) for k, m in ((0, gx), (1, gy))], -1)
        seen = (tz > near) & ((hi - lo) > 0).all(-1)
    return center, conic, tz.detach(), lo.long(), hi.long(), seen


_CHUNK = 1 << 24  # (pixel, Gaussian) pairs evaluated together
_MOST_PAIRS = 60_000_000


def _exact_view(leaves, upstream, statistics, lists, width, height, background):
    """One camera's image, the gradients of the leaves (centres, conics,
    opacities, channels) and the statistics, tile by tile."""
    center, conic, opacity, channels = leaves
    pairs, first, count = lists
    gx, gy = (width + 15) // 16, (height + 15) // 16
    n, depth = channels.shape
    device = center.device
    image = torch.zeros((gy * 16, gx * 16, depth + 1), dtype=torch.float64, device=device)
    image[..., :depth] = background
    if upstream is not None:
        padded = torch.zeros_like(image)
        padded[:height, :width] = upstream
    totals = [torch.zeros(n + 1, dtype=torch.float64, device=device) for _ in statistics]
    maps = []
    for _, values in statistics:
        m = torch.zeros((gy * 16, gx * 16), dtype=torch.float64, device=device)
        m[:height, :width] = values
        maps.append(m)
    order = torch.argsort(count, descending=True)
    lengths = count[order].tolist()
    pixel = torch.arange(256, device=device)
    at = 0
    while at < len(lengths) and lengths[at] > 0:
        longest = lengths[at]
        end = min(len(lengths), at + max(1, _CHUNK // (longest * 256)))
        tiles = order[at:end]
        at = end
        slot = torch.arange(longest, device=device)
        member = slot[None] < count[tiles][:, None]
        ids = pairs[(first[tiles][:, None] + slot[None]).clamp_max(len(pairs) - 1)]
        x = (tiles % gx * 16)[:, None] + pixel[None] % 16
        y = (tiles // gx * 16)[:, None] + pixel[None] // 16
        inside = (x < width) & (y < height)
        with torch.enable_grad():
            dx = center[ids, 0][..., None] - x[:, None]
            dy = center[ids, 1][..., None] - y[:, None]
            k = conic[ids]
            power = -0.5 * (k[..., 0, None] * dx * dx + k[..., 2, None] * dy * dy) - k[..., 1, None] * dx * dy
            alpha = (opacity[ids][..., None] * torch.exp(power.clamp_max(0.0))).clamp_max(0.99)
            keep = (power <= 0) & (alpha >= 1 / 255) & member[..., None] & inside[:, None]
            decay = torch.log1p(-torch.where(keep, alpha, torch.zeros_like(alpha)))
            after = torch.exp(torch.cumsum(decay, 1))
            keep = keep & (after.detach() >= 1e-4)
            weight = torch.where(keep, alpha * torch.exp(torch.cumsum(decay, 1) - decay), torch.zeros_like(alpha))
            colour = weight.transpose(1, 2) @ channels[ids]
            covered = weight.sum(1)[..., None]
            out = torch.cat([colour + (1 - covered) * background, covered], -1)
            if upstream is not None:
                out.backward(padded[y, x] * inside[..., None])
        image[y, x] = out.detach()
        for total, m, (is_sum, _) in zip(totals, maps, statistics):
            v = m[y, x][:, None]
            part = v * weight.detach() if is_sum else ((v != 0) & keep).double()
            total.index_add_(0, torch.where(member, ids, n).reshape(-1), part.sum(-1).reshape(-1))
    return image[:height, :width], [t[:n] for t in totals]


def exact(case, seed):
    state = prepare(case, seed)
    degree = case["sh_degree"]
    double = lambda t: t.detach().double()
    if case["kind"] == "sh":
        sh, dirs = double(state["sh"]).requires_grad_(), double(state["dirs"]).requires_grad_()
        colors = _sh_colors(sh, dirs, degree)
        colors.backward(double(state["upstream"]))
        out = dict(colors=colors.detach(), sh=sh.grad)
        return dict(out, dirs=dirs.grad) if degree > 0 else out
    width, height, batch = case["width"], case["height"], case["batch"]
    train = "grads" in state
    near = 0.2 if case["kind"] in ("train", "render") else 0.01
    names = [k for k in ("means", "quats", "scales", "opacities", "colors", "extra", "viewmats") if k in state]
    leaf = {k: double(state[k]).requires_grad_() for k in names}
    images, totals, screens = [], [], []
    budget = _MOST_PAIRS
    for b in range(max(1, batch)):
        pick = lambda t: t[b] if batch else t
        for c in range(case["cameras"]):
            view, K = pick(leaf["viewmats"])[c], double(pick(state["Ks"])[c])
            means = pick(leaf["means"])
            center, conic, depth, lo, hi, seen = _project(means, pick(leaf["quats"]), pick(leaf["scales"]), view, K,
                                                          width, height, near)
            channels = pick(leaf["colors"])
            if degree >= 0:
                channels = _sh_colors(channels, means - torch.linalg.inv(view)[:3, 3], degree)
            if "extra" in leaf:
                channels = torch.cat([channels, pick(leaf["extra"])], -1)
            # Depth-ordered lists of every tile: pairs in depth order, stably
            # sorted by tile.
            rank = torch.argsort(depth.float(), stable=True)
            rank = rank[seen[rank]]
            span = (hi - lo)[rank]
            per_row = span[:, 0] * span[:, 1]
            budget -= int(per_row.sum())
            if budget < 0:
                return None
            ids = torch.repeat_interleave(rank, per_row)
            offset = torch.arange(len(ids), device=ids.device) - torch.repeat_interleave(
                torch.cumsum(per_row, 0) - per_row, per_row)
            wide = (hi - lo)[ids, 0]
            gx, gy = (width + 15) // 16, (height + 15) // 16
            tile = (lo[ids, 1] + offset // wide.clamp_min(1)) * gx + lo[ids, 0] + offset % wide.clamp_min(1)
            tile, by_tile = torch.sort(tile, stable=True)
            count = torch.bincount(tile, minlength=gx * gy)
            lists = (ids[by_tile], torch.cumsum(count, 0) - count, count)
            background = torch.zeros(channels.shape[1], dtype=torch.float64, device=ids.device)
            if case["background"]:
                background[:state["background"].shape[-1]] = double(pick(state["background"])[c])
            upstream = None
            if train:
                planes = [state["upstream"][i] for i in ((0, 2, 1) if case["extra"] else (0, 1))]
                if case["kind"] != "staged":
                    planes = [pick(p)[c] for p in planes]
                upstream = torch.cat([double(p) for p in planes], -1)
            requests = [(isinstance(r, WeightedContributionSum),
                         (r.pixel_weights if isinstance(r, WeightedContributionSum) else r.mask)[c].double())
                        for r in state.get("statistics", ())]
            stage = [t.detach().requires_grad_(train) for t in (center, conic, pick(leaf["opacities"]), channels)]
            image, counted = _exact_view(stage, upstream, requests, lists, width, height, background)
            images.append(image)
            totals.append(counted)
            if train:
                grads = [torch.zeros_like(t) if t.grad is None else t.grad for t in stage]
                for grad in grads:
                    grad[~seen] = 0
                screens.append(grads[0])
                finite = lambda t: torch.where(seen.reshape(-1, *[1] * (t.ndim - 1)), t, torch.zeros_like(t))
                torch.autograd.backward([finite(center), finite(conic), pick(leaf["opacities"]), channels], grads)
    lead = ((batch,) if batch else ()) + (() if case["kind"] == "staged" else (case["cameras"],))
    image = torch.stack(images).reshape(lead + images[0].shape)
    colours = 3 if degree >= 0 else case["channels"]
    out = dict(features=image[..., :colours], alpha=image[..., -1:])
    if train:
        out["grads"] = {k: leaf[k].grad for k in state["grads"]}
        if case["extra"]:
            out["extra"] = image[..., colours:-1]
        if case["kind"] == "train":
            screen = torch.stack(screens)
            out["means2d_grad"] = screen.reshape(lead + screen.shape[1:])
    elif case["requests"]:
        # Counts are whole numbers; sums are computed ones.
        out["statistics"] = {r.name: torch.stack([t[i] for t in totals])
                             for i, r in enumerate(state["statistics"]) if isinstance(r, WeightedContributionSum)}
    return out
