"""The renderer's work as its users call it, for timing and for checking results.

Every case is a grid of ``svox2_amd.scenes``' blob family and one call, or one
training step, through ``svox2_amd.SparseGrid``.  The kinds:

  image     one rendered image without gradients (viewer, test-set evaluation,
            a request of the serving loop)
  depth     one depth image (geometry export, depth supervision)
  fused     one fused forward + MSE backward on a batch of camera rays, the
            core of a training step; cuvol or nvol compositing, with or without
            the beta and sparsity terms, in front of an MSI background or not
  train     one whole training step: fused, both TV terms, both RMSprop steps
  autograd  ``volume_render``, a loss in torch and ``backward``, with per-ray
            clips (the differentiable path of programs with losses of their own)
  sample    trilinear samples at free points and their backward

``exact`` restates the same quantities in plain float64 torch: samples lie on
the lattice t_min + k step of each ray (skipping empty space removes only
samples that read zeros), so no skip distance enters.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import svox2_amd
from svox2_amd import scenes

DEV = "cuda"
STEP = 0.5           # march step, in voxels
SIGMA_THRESH = 1e-8
STOP = 1e-7
# The regularised training step: late in a run, when steps are small.
TV_DENSITY, TV_SH, TV_FRAC = 1e-5, 1e-3, 0.01
LR_DENSITY, LR_SH, BETA, EPS = 1e-3, 1e-5, 0.95, 1e-8
BG_RESO, BG_LAYERS = 256, 64

_DEFAULTS = {"kind": "fused", "reso": 512, "storage": "f32", "backend": "cuvol", "rays": 0,
             "beta": 0.0, "sparsity": 0.0, "background": False, "width": 0, "height": 0}


def _case(name=None, **kw):
    c = dict(_DEFAULTS, **kw)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # The smallest request of the serving mix: launch latency.
        _case("image_128_256_bf16", kind="image", reso=256, storage="bf16", width=128, height=128),
        # A test view of the 512^3 grid.
        _case("image_800_512", kind="image", reso=512, width=800, height=800),
        # Its depth map.
        _case("depth_800_512", kind="depth", reso=512, width=800, height=800),
        # The first, coarse stage: a small dense grid, every sample contributes.
        _case("fused_4096_dense64", reso=64, rays=4096),
        # The usual training batch on the final grid.
        _case("fused_5000_512", reso=512, rays=5000),
        # The benchmark's batch.
        _case("fused_65536_512", reso=512, rays=65536),
        # A large odd batch in bfloat16 with the regularisers folded into it.
        _case("fused_200003_512_bf16", reso=512, rays=200003, storage="bf16", beta=1e-3,
              sparsity=1e-11),
        # The training step of the middle stage, 256^3.
        _case("train_5000_256", kind="train", reso=256, rays=5000),
        # A step of a program with its own loss, clipped rays.
        _case("autograd_262144_512", kind="autograd", reso=512, rays=262144),
        # An unbounded scene: the grid in front of an MSI background.
        _case("background_65536_512", reso=512, rays=65536, background=True),
        # The opacity-accumulating backend.
        _case("nvol_30000_256", reso=256, rays=30000, backend="nvol"),
        # A million free points, forward and backward.
        _case("sample_1m_512", kind="sample", reso=512, rays=1 << 20),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["image", "depth", "fused", "fused", "fused", "train", "autograd",
                       "background", "nvol", "sample"])
    reso = _log_int(rng, 64, 512)
    storage = rng.choice(["f32", "f32", "bf16"])
    if kind in ("image", "depth"):
        return _case(kind=kind, reso=reso, storage=storage, width=_log_int(rng, 100, 800),
                     height=_log_int(rng, 100, 800))
    if kind == "fused":
        reg = rng.random() < 0.4
        return _case(reso=reso, storage=storage, rays=_log_int(rng, 500, 200000),
                     beta=1e-3 if reg else 0.0, sparsity=1e-11 if reg else 0.0)
    if kind == "train":
        return _case(kind="train", reso=min(reso, 320), rays=_log_int(rng, 2000, 20000))
    if kind == "autograd":
        return _case(kind="autograd", reso=reso, storage=storage, rays=_log_int(rng, 2000, 262144))
    if kind == "background":
        return _case(reso=reso, rays=_log_int(rng, 2000, 60000), background=True)
    if kind == "nvol":
        return _case(reso=reso, storage=storage, rays=_log_int(rng, 2000, 50000), backend="nvol")
    return _case(kind="sample", reso=reso, storage=storage, rays=_log_int(rng, 10000, 1 << 20))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _scene(reso, dgen):
    """A blob grid (dense up to 96^3, about 3 % of the cells from 384^3 on, 8 %
    between).  One scene per resolution, so that its row count is its own; the
    opacity of the whole and the SH rows come from the seed."""
    spec = scenes.DENSE64 if reso <= 96 else scenes.SPARSE256 if reso < 384 else scenes.SPARSE512
    blobs = scenes.draw_blobs(spec, torch.Generator().manual_seed(reso))
    field = scenes.blob_field(reso, *blobs, device=DEV)
    if reso <= 96:
        links = torch.arange(reso ** 3, dtype=torch.int32, device=DEV).view(reso, reso, reso)
        density = field.reshape(-1, 1)
    else:
        links, rows = scenes.morton_rows(field > spec.threshold)
        cells = torch.nonzero(links.flatten() >= 0).flatten()
        density = torch.empty(rows, 1, dtype=torch.float64, device=DEV)
        density[links.flatten()[cells].long(), 0] = field.flatten()[cells]
    density *= 0.75 + 0.5 * torch.rand(1, generator=dgen, device=DEV).double()
    sh = torch.randn(density.size(0), 27, generator=dgen, device=DEV) * 0.1
    dc = torch.randn(density.size(0), 3, generator=dgen, device=DEV) * 0.2 + 0.5
    sh[:, [0, 9, 18]] = dc
    return scenes.SceneData(links, density, sh, 9, density.size(0) / reso ** 3)


def prepare(case, seed):
    gen = torch.Generator().manual_seed(seed)
    dgen = torch.Generator(device=DEV).manual_seed(seed)
    scene = _scene(case["reso"], dgen)
    grid = scenes.to_sparse_grid(scene, device=DEV, dtype=torch.bfloat16
                                 if case["storage"] == "bf16" else torch.float32)
    del scene
    grid.opt.sigma_thresh, grid.opt.stop_thresh = SIGMA_THRESH, STOP
    grid.opt.backend = case["backend"]
    if case["background"]:
        columns = 2 * BG_RESO * BG_RESO
        data = torch.empty(columns, BG_LAYERS, 4, device=DEV)
        data[..., :3] = torch.randn(columns, BG_LAYERS, 3, generator=dgen, device=DEV) * 0.5
        data[..., 3] = torch.rand(columns, BG_LAYERS, generator=dgen, device=DEV) * 2.0
        grid.background_nlayers, grid.background_reso = BG_LAYERS, BG_RESO
        grid.background_links = torch.arange(columns, dtype=torch.int32, device=DEV).view(
            2 * BG_RESO, BG_RESO)
        grid.background_data = torch.nn.Parameter(data)
    s = {"kind": case["kind"], "grid": grid, "beta": case["beta"], "sparsity": case["sparsity"]}
    cams = scenes.CameraSet(scenes.hemisphere_cameras(20, gen))
    n = case["rays"]
    if case["kind"] in ("image", "depth"):
        cam = cams.camera(0, width=case["width"], height=case["height"])
        if case["kind"] == "depth":
            cam.c2w = cam.c2w.to(DEV)  # its rays are generated on the device
        s["camera"] = cam
    elif case["kind"] == "sample":
        s["points"] = torch.rand(n, 3, generator=dgen, device=DEV) * 2 - 1
        s["grad_density"] = torch.randn(n, 1, generator=dgen, device=DEV)
        s["grad_sh"] = torch.randn(n, 27, generator=dgen, device=DEV)
    else:
        # Camera rays; on the small dense grid rays aimed into it from close by.
        o, d = (scenes.sphere_rays(n, gen) if case["reso"] <= 96 else cams.random_batch(n, gen))
        clip = scenes.config_clip(n, gen).to(DEV) if case["kind"] == "autograd" else None
        s["rays"] = svox2_amd.Rays(o.to(DEV), d.to(DEV), clip)
        s["gt"] = torch.rand(n, 3, generator=dgen, device=DEV)
    if case["kind"] == "train":
        # RMSprop state as a run in progress has it: about the gradients' squares.
        for name, data in (("density_rms", grid.density_data), ("sh_rms", grid.sh_data)):
            rms = torch.rand(data.shape, generator=dgen, device=DEV).add_(0.5).mul_(1e-5).square_()
            s[name] = rms
        from svox2_amd.svox2 import interleaved_rows
        grid.density_rms, grid.sh_rms = interleaved_rows(
            grid.sh_data.size(0), grid.sh_data.size(1), torch.float32, DEV)
        grid.density_rms.copy_(s.pop("density_rms"))
        grid.sh_rms.copy_(s.pop("sh_rms"))
        np.random.seed(seed)  # the regularisers draw their cells from numpy, as in training
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(s):
    grid, kind = s["grid"], s["kind"]
    if kind == "image":
        with torch.no_grad():
            return grid.volume_render_image(s["camera"])
    if kind == "depth":
        with torch.no_grad():
            return grid.volume_render_depth_image(s["camera"])
    if kind == "sample":
        grid.density_data.grad = grid.sh_data.grad = None
        density, sh = grid.sample(s["points"])
        torch.autograd.backward([density, sh], [s["grad_density"], s["grad_sh"]])
        return {"density": density, "sh": sh, "grad_density": grid.density_data.grad,
                "grad_sh": grid.sh_data.grad}
    if kind == "autograd":
        grid.density_data.grad = grid.sh_data.grad = None
        rgb = grid.volume_render(s["rays"])
        torch.nn.functional.mse_loss(rgb, s["gt"]).backward()
        return {"rgb": rgb, "grad_density": grid.density_data.grad, "grad_sh": grid.sh_data.grad}
    rgb = grid.volume_render_fused(s["rays"], s["gt"], beta_loss=s["beta"],
                                   sparsity_loss=s["sparsity"])
    if kind == "train":
        grid.inplace_tv_grad(grid.density_data.grad, scaling=TV_DENSITY, sparse_frac=TV_FRAC)
        grid.inplace_tv_color_grad(grid.sh_data.grad, scaling=TV_SH, sparse_frac=TV_FRAC)
        grid.optim_density_step(LR_DENSITY, beta=BETA, epsilon=EPS)
        grid.optim_sh_step(LR_SH, beta=BETA, epsilon=EPS)
        return {"rgb": rgb, "density": grid.density_data, "sh": grid.sh_data,
                "density_rms": grid.density_rms, "sh_rms": grid.sh_rms}
    out = {"rgb": rgb, "grad_density": grid.density_data.grad, "grad_sh": grid.sh_data.grad,
           "touched": grid.sparse_grad_indexer}
    if grid.use_background:
        out["grad_background"] = grid.background_data.grad
    return out


# ---------------------------------------------------------------------------
# Work
# ---------------------------------------------------------------------------
def work(case):
    """Bytes each pass must move: its rays or pixels, each data row its samples
    read once, each gradient row written once (read and written where a batch
    adds to a gradient that is there), cell links of the occupied cells passed.
    A camera ray of these scenes has about 17 contributing samples at 512^3 on
    average (a third of the rays has all of them), in proportion at other
    resolutions, 60 in the small dense grid; a sample enters about 2 rows no
    other sample of its ray has entered."""
    reso, n = case["reso"], case["rays"] or case["width"] * case["height"]
    rows = reso ** 3 * (1.0 if reso <= 96 else 0.084 if reso < 384 else 0.032)
    row = 28 * (2 if case["storage"] == "bf16" else 4)
    flops_sample = 8 * 2 + 8 * 27 * 2 + 27 * 2
    if case["kind"] == "sample":
        hit = n * 8 * rows / reso ** 3
        used = rows * (1 - math.exp(-hit / rows))
        return {"bytes": n * (12 + 2 * 112) + 32 * n + used * row + rows * 112,
                "flops": n * 2 * flops_sample}
    samples = n * (60 if reso <= 96 else (45.0 if reso < 384 else 17.0) * reso
                   / (256 if reso < 384 else 512))
    used = rows * (1 - math.exp(-2 * samples / rows))
    if case["kind"] == "depth":
        return {"bytes": 16 * n + used * row / 28 + 4 * samples, "flops": samples * 40}
    if case["kind"] == "image":
        return {"bytes": 12 * n + used * row + 4 * samples, "flops": samples * flops_sample}
    moved = n * 48 + used * row + 4 * samples
    if case["kind"] == "autograd":
        moved += rows * 112 + 8 * n
    else:
        moved += used * 2 * 112 + rows
    if case["kind"] == "train":
        moved += used * 112 * 4 + TV_FRAC * reso ** 3 * 16
    flops = samples * 3 * flops_sample
    if case["background"]:
        layers = n * BG_LAYERS
        cells = 2 * BG_RESO * BG_RESO * BG_LAYERS
        bg_used = cells * (1 - math.exp(-4 * layers / cells))
        moved += bg_used * 16 * 3 + cells
        flops += layers * 200
    return {"bytes": moved, "flops": flops}


# ---------------------------------------------------------------------------
# The same in float64
# ---------------------------------------------------------------------------
def _affine(grid):
    n = torch.tensor(grid.links.shape, dtype=torch.float64, device=DEV)
    radius, center = grid.radius.double().to(DEV), grid.center.double().to(DEV)
    scaling = 0.5 / radius * n
    return n, scaling, 0.5 * (1 - center / radius) * n - 0.5


def _cells(links, n, pos):
    """(rows (.., 8) with -1 for empty, weights (.., 8)) of grid positions."""
    pos = torch.minimum(pos.clamp_min(0.0), n - 1)
    low = torch.minimum(pos.long(), (n - 2).long())
    f = pos - low
    flat = links.reshape(-1)
    base = (low[..., 0] * links.size(1) + low[..., 1]) * links.size(2) + low[..., 2]
    rows, weights = [], []
    for k in range(8):
        dx, dy, dz = k >> 2, (k >> 1) & 1, k & 1
        rows.append(flat[base + (dx * links.size(1) + dy) * links.size(2) + dz].long())
        weights.append((f[..., 0] if dx else 1 - f[..., 0]) * (f[..., 1] if dy else 1 - f[..., 1])
                       * (f[..., 2] if dz else 1 - f[..., 2]))
    return torch.stack(rows, -1), torch.stack(weights, -1)


def _sh_basis(d):
    x, y, z = (d / d.norm(dim=1, keepdim=True)).unbind(1)
    c = (0.28209479177387814, 0.4886025119029199, 1.0925484305920792, 0.31539156525252005,
         0.5462742152960396)
    return torch.stack([torch.full_like(x, c[0]), -c[1] * y, c[1] * z, -c[1] * x, c[2] * x * y,
                        -c[2] * y * z, c[3] * (2 * z * z - x * x - y * y), -c[2] * x * z,
                        c[4] * (x * x - y * y)], 1)


def _march(grid, o, d, clip, density):
    """The rays' contributing samples, in order: (ray, t, rows, weights, world
    step of each ray); rows are -1 where a corner is empty."""
    n, scaling, offset = _affine(grid)
    go, gd = o * scaling + offset, d * scaling
    per = 1.0 / gd.norm(dim=1)
    gd = gd * per[:, None]
    t1, t2 = (-0.5 - go) / gd, (n - 0.5 - go) / gd
    tmin = torch.minimum(t1, t2).amax(1).clamp_min(0.0)
    tmax = torch.maximum(t1, t2).amin(1).clamp_max(2e3)
    if clip is not None:
        tmin = torch.maximum(tmin, clip[:, 0].double() / per)
        tmax = torch.minimum(tmax, clip[:, 1].double() / per)
    last = int(((tmax - tmin) / STEP).clamp_min(0).max()) + 1
    found = []
    for k0 in range(0, last, 128):
        k = torch.arange(k0, min(k0 + 128, last), device=DEV)
        t = tmin[:, None] + k * STEP
        ray, at = torch.nonzero(t <= tmax[:, None], as_tuple=True)
        t = t[ray, at]
        rows, w = _cells(grid.links, n, go[ray] + t[:, None] * gd[ray])
        w = torch.where(rows >= 0, w, torch.zeros_like(w))
        keep = (w * density[rows.clamp_min(0)]).sum(1) > SIGMA_THRESH
        found.append([x[keep] for x in (ray, t, rows, w)])
    ray, t, rows, w = (torch.cat(x) for x in zip(*found))
    order = torch.argsort(ray, stable=True)
    return ray[order], t[order], rows[order], w[order], per * STEP


def _before(ray, n, x):
    """Sum of x over the earlier samples of the same ray."""
    incl = torch.cumsum(x, 0)
    count = torch.bincount(ray, minlength=n)
    start = (torch.cumsum(count, 0) - count)[ray]
    return incl - x - torch.where(start > 0, incl[(start - 1).clamp_min(0)],
                                  torch.zeros_like(x))


def _composite(grid, backend, d, m, density, sh, bg):
    """(colours, per-sample opacity sums for the regularisers, log T at the end)."""
    ray, _, rows, w, ws = m
    n = d.size(0)
    rows = rows.clamp_min(0)
    sigma = (w * density[rows]).sum(1)
    depth = ws[ray] * sigma
    before = _before(ray, n, depth)
    if backend == "cuvol":
        alive = (before.detach() <= -math.log(STOP))
        weight = torch.exp(-before) * (1 - torch.exp(-depth))
        dead = torch.zeros(n, device=DEV, dtype=torch.bool)
        dead[ray[(before + depth).detach() > -math.log(STOP)]] = True
        total = torch.zeros(n, dtype=torch.float64, device=DEV).index_add(0, ray, depth * alive)
        left = torch.exp(-total) * ~dead
    else:
        a = 1 - torch.exp(-depth)
        earlier = _before(ray, n, a)
        alive = earlier.detach() < 1
        weight = (earlier + a).clamp_max(1.0) - earlier.clamp_max(1.0)
        total = torch.zeros(n, dtype=torch.float64, device=DEV).index_add(0, ray, a)
        left = 1 - total.clamp_max(1.0)
    ray, rows, w, weight, alive_sigma = (x[alive] for x in (ray, rows, w, weight, sigma))
    basis = _sh_basis(d)[ray]
    coeff = (w[..., None] * sh[rows]).sum(1).view(-1, 3, 9)
    colour = ((coeff * basis[:, None]).sum(2) + 0.5).clamp_min(0.0)
    rgb = torch.zeros(n, 3, dtype=torch.float64, device=DEV).index_add(0, ray,
                                                                       weight[:, None] * colour)
    return rgb + left[:, None] * bg, alive_sigma, total, left, (rows, w, alive)


def _behind(grid, o, d, left, data):
    """The MSI background's colour behind each ray (differentiable in data and
    in the transmittance left)."""
    n, scaling, offset = _affine(grid)
    gd = d * scaling
    per = 1.0 / gd.norm(dim=1)
    so, sd = (o * scaling + offset + 0.5) * 2 / n - 1, gd * per[:, None] * 2 / n
    unit = 1.0 / sd.norm(dim=1)
    per, sd = per * unit, sd * unit[:, None]
    half_b = (so * sd).sum(1)
    gap = half_b * half_b - (so * so).sum(1)
    inner = (torch.linalg.cross(so, sd).norm(dim=1) + 1e-3).clamp_min(1.0)
    columns, layers = 2 * BG_RESO, BG_LAYERS
    steps = int(layers / STEP) + 2
    flat = data.reshape(-1, 4)
    live = left.detach() > math.exp(-25.0)
    trans, last = left, 1.0 / inner
    out = torch.zeros(o.size(0), 3, dtype=torch.float64, device=DEV)
    for i in range(steps):
        r = steps / (steps - i - 0.5)
        det = gap + r * r
        ok = live & (inner <= r) & (det >= 0)
        p = so + (det.clamp_min(0).sqrt() - half_b)[:, None] * sd
        inv = 1.0 / p.norm(dim=1)
        u = p * inv[:, None]
        x = columns * (0.5 + torch.atan2(u[:, 0], u[:, 2]) / (2 * math.pi))
        y = BG_RESO * (0.5 - torch.asin(u[:, 1].clamp(-1, 1)) / math.pi)
        z = ((1 - inv) * layers - 0.5).clamp(0, layers - 1)
        x0, y0 = x.long().clamp(0, columns - 1), y.long().clamp(0, BG_RESO - 1)
        z0 = z.long().clamp(0, layers - 2)
        fx, fy, fz = ((a - b)[:, None] for a, b in ((x, x0), (y, y0), (z, z0)))
        value = 0.0
        for cx, wx in ((x0, 1 - fx), ((x0 + 1) % columns, fx)):
            for cy, wy in ((y0, 1 - fy), ((y0 + 1) % BG_RESO, fy)):
                at = (cx * BG_RESO + cy) * layers + z0
                value = value + wx * wy * ((1 - fz) * flat[at] + fz * flat[at + 1])
        sigma = value[:, 3]
        use = ok & (sigma.detach() > 0)
        depth = torch.where(use, (last - inv) * per * sigma, torch.zeros_like(sigma))
        colour = (value[:, :3] * 0.28209479177387814 + 0.5).clamp_min(0.0)
        out = out + (trans * (1 - torch.exp(-depth)) * use)[:, None] * colour
        trans = trans * torch.exp(-depth)
        live = live & ~(use & (trans.detach() < STOP))
        last = torch.where(ok, inv, last)
    shown = (left.detach() > math.exp(-25.0))
    return out + (trans * shown)[:, None]


def _render_grads(case, s):
    """Colours, gradients and touched rows of the mean squared error with the
    folded regularisers, block of rays by block of rays."""
    grid, rays = s["grid"], s["rays"]
    n = rays.origins.size(0)
    density = grid.density_data.detach().double().view(-1).requires_grad_()
    sh = grid.sh_data.detach().double().requires_grad_()
    data = grid.background_data.detach().double().requires_grad_() if case["background"] else None
    touched = torch.zeros(density.numel(), dtype=torch.bool, device=DEV)
    colours = []
    for b in range(0, n, 16384):
        o, d = (x[b:b + 16384].double() for x in (rays.origins, rays.dirs))
        clip = None if rays.clip is None else rays.clip[b:b + 16384]
        m = _march(grid, o, d, clip, density.detach())
        rgb, sigma, total, left, (rows, w, alive) = _composite(
            grid, case["backend"], d, m, density, sh, 0.0 if data is not None else 1.0)
        if data is not None:
            rgb = rgb + _behind(grid, o, d, left, data)
        loss = (rgb - s["gt"][b:b + 16384].double()).square().sum() / (3 * n)
        if case["beta"] > 0:
            t = left.detach()
            loss = loss - (case["beta"] / n * (1 - t / (1 - t + 1e-3)) * total).sum()
        if case["sparsity"] > 0:
            loss = loss + case["sparsity"] * torch.log1p(2 * sigma * sigma).sum()
        loss.backward()
        real = m[2][alive]
        touched[real[real >= 0]] = True
        colours.append(rgb.detach())
    return (torch.cat(colours), density.grad[:, None], sh.grad, touched,
            None if data is None else data.grad)


def _tv(grid, data, first, scale, edge):
    """The total-variation gradient over a run of cells from `first`, and the
    rows it touches; a neighbour past the grid's end is row 0; an empty one
    reads 0, or with `edge` the cell's own value (and row 0's cell is left out)."""
    links = grid.links
    flat = links.reshape(-1).long()
    count = max(int(TV_FRAC * flat.numel()), 1)
    cell = (first + torch.arange(count, device=DEV)) % flat.numel()
    sizes = links.shape
    at = torch.stack([cell // (sizes[1] * sizes[2]), cell // sizes[2] % sizes[1], cell % sizes[2]])
    own = flat[cell]
    use = own != 0 if edge else torch.ones_like(own, dtype=torch.bool)
    near = []
    for a, stride in enumerate((sizes[1] * sizes[2], sizes[2], 1)):
        inside = at[a] + 1 < sizes[a]
        near.append(torch.where(inside, flat[(cell + stride).clamp_max(flat.numel() - 1)], 0))
    own, near = own[use], [x[use] for x in near]
    live = (own >= 0) | torch.stack([x >= 0 for x in near]).any(0)
    own, near = own[live], [x[live] for x in near]

    def value(row, null):
        v = data[row.clamp_min(0)]
        return torch.where((row >= 0)[:, None], v, null)

    v0 = value(own, torch.zeros((), dtype=torch.float64, device=DEV))
    null = v0 if edge else torch.zeros_like(v0)
    diff = [value(x, null) - v0 for x in near]
    scaled = [x * (sizes[a] / 256.0) for a, x in enumerate(diff)]
    norm = scale / count / torch.sqrt(1e-9 + sum(x * x for x in diff))
    grad, touched = torch.zeros_like(data), torch.zeros(data.size(0), dtype=torch.bool, device=DEV)
    for row, term in zip([own] + near, [-sum(scaled)] + scaled):
        there = row >= 0
        grad.index_add_(0, row[there], (term * norm)[there])
        touched[row[there & (term != 0).any(1)]] = True
    return grad, touched


def _image_rays(cam):
    pix = torch.arange(cam.width * cam.height, device=DEV)
    x = ((pix % cam.width).double() + 0.5 - cam.cx_val) / cam.fx_val
    y = ((pix // cam.width).double() + 0.5 - cam.cy_val) / cam.fy_val
    d = torch.stack([x, y, torch.ones_like(x)], 1)
    d = d / d.norm(dim=1, keepdim=True)
    c2w = cam.c2w.double().to(DEV)
    return c2w[:3, 3].expand_as(d), d @ c2w[:3, :3].T


def exact(case, seed):
    s = prepare(case, seed)
    grid, kind = s["grid"], case["kind"]
    density = grid.density_data.detach().double().view(-1)
    sh = grid.sh_data.detach().double()
    if kind in ("image", "depth"):
        o, d = _image_rays(s["camera"])
        parts = []
        with torch.no_grad():
            for b in range(0, o.size(0), 16384):
                ob, db = o[b:b + 16384], d[b:b + 16384]
                m = _march(grid, ob, db, None, density)
                if kind == "image":
                    parts.append(_composite(grid, "cuvol", db, m, density, sh, 1.0)[0])
                    continue
                ray, t, rows, w, ws = m
                depth = ws[ray] * (w * density[rows.clamp_min(0)]).sum(1)
                before = _before(ray, ob.size(0), depth)
                weight = torch.exp(-before) * (1 - torch.exp(-depth)) * (before <= -math.log(STOP))
                parts.append(torch.zeros(ob.size(0), dtype=torch.float64, device=DEV).index_add(
                    0, ray, weight * t / STEP * ws[ray]))
        return torch.cat(parts).view(case["height"], case["width"],
                                     *([3] if kind == "image" else []))
    if kind == "sample":
        n, scaling, offset = _affine(grid)
        rows, w = _cells(grid.links, n, s["points"].double() * scaling + offset)
        w = torch.where(rows >= 0, w, torch.zeros_like(w))
        rows = rows.clamp_min(0)
        out = {"density": torch.zeros(w.size(0), 1, dtype=torch.float64, device=DEV),
               "sh": torch.zeros(w.size(0), 27, dtype=torch.float64, device=DEV),
               "grad_density": torch.zeros_like(density)[:, None],
               "grad_sh": torch.zeros_like(sh)}
        for k in range(8):
            wk, rk = w[:, k:k + 1], rows[:, k]
            out["density"] += wk * density[rk][:, None]
            out["sh"] += wk * sh[rk]
            out["grad_density"].index_add_(0, rk, wk * s["grad_density"].double())
            out["grad_sh"].index_add_(0, rk, wk * s["grad_sh"].double())
        return out
    rgb, g_density, g_sh, touched, g_data = _render_grads(case, s)
    if kind == "autograd":
        return {"rgb": rgb, "grad_density": g_density, "grad_sh": g_sh}
    if kind == "train":
        draws = np.random.RandomState(seed)
        cells = grid.links.numel()
        out = {"rgb": rgb}
        for name, data, grad, rms, scale, edge, lr in (
                ("density", density[:, None], g_density, grid.density_rms, TV_DENSITY, False,
                 LR_DENSITY),
                ("sh", sh, g_sh, grid.sh_rms, TV_SH, True, LR_SH)):
            tv, marked = _tv(grid, data, int(draws.randint(0, cells)), scale, edge)
            g, rms = grad + tv, rms.double()
            on = (touched | marked)[:, None]
            new = torch.where(rms == 0, g * g, BETA * rms + (1 - BETA) * g * g)
            out[name] = torch.where(on, data - lr * g / (new.sqrt() + EPS), data)
            out[name + "_rms"] = torch.where(on, new, rms)
        return out
    out = {"rgb": rgb, "grad_density": g_density, "grad_sh": g_sh, "touched": None}
    if g_data is not None:
        out["grad_background"] = g_data
    return out
