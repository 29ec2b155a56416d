"""Kernel variants at the sizes where their tiling can go wrong: point sets
around the sampler's 16 points per wavefront and its cell-map thresholds, MSI
backgrounds whose layers and columns do not fill the scatter's 8-layer window or
wrap onto slots of the same parity, launches on both sides of the ray count
from which a march's start is searched by a lane per ray."""
import numpy as np
import pytest
import torch

import oracle.oracle as O
import svox2_amd
from svox2_amd import _C, scenes
from tests.conftest import assert_grad_close, host_grid

pytestmark = pytest.mark.gpu


def _grid(sc, dev, dtype=torch.float32):
    g = scenes.to_sparse_grid(sc, device=dev, dtype=dtype)
    g.opt.sigma_thresh, g.opt.stop_thresh = 1e-8, 1e-7
    return g


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 1000, 32768])
@pytest.mark.parametrize("kind", ["dense", "sparse"])
def test_sample_point_sets(gpu, kind, n):
    """Values within 1e-5 and gradients within 1e-5 of the largest (float32
    sums of at most a few hundred terms, 2^-24 each) of float64 sampling, with
    and without the cell map; points outside the grid clamp to its border."""
    gen = torch.Generator().manual_seed(n)
    spec = scenes.BlobSpec(4, (0.2, 0.2), (20.0, 20.0))
    sc = scenes.make_blob_grid(20, spec, gen, dense=kind == "dense")
    grid = _grid(sc, gpu)
    pts = torch.rand(n, 3, generator=gen) * 2.2 - 1.1
    gd, gs = torch.randn(n, 1, generator=gen), torch.randn(n, 27, generator=gen)
    links, dens = sc.links.numpy(), sc.density.double().float().double().requires_grad_()
    sh = sc.sh.float().double().requires_grad_()
    N = np.array(links.shape, np.float64)
    f32 = np.float32
    pg = (pts.numpy() * f32(0.5 * N[0]) + f32(0.5 * N[0] - 0.5)).astype(f32)
    d64, s64 = O.sample_trilerp(links, dens, sh, pg)
    torch.autograd.backward([d64, s64], [gd.double(), gs.double()])
    for cmap in (None, False):
        s = grid._to_cpp()
        s.cell_map = False if cmap is False else _C.build_cell_map(s.links, grid.sh_data.size(0))
        p = pts.to(gpu)
        d, c = _C.sample_grid(s, p, True)
        only, _ = _C.sample_grid(s, p, False)
        assert torch.equal(only, d)
        assert (d.cpu().double() - d64.detach()).abs().max() <= 1e-5 * 20
        assert (c.cpu().double() - s64.detach()).abs().max() <= 1e-5
        out = [torch.zeros(grid.sh_data.size(0), k, device=gpu) for k in (1, 27)]
        _C.sample_grid_backward(s, p, gd.to(gpu), gs.to(gpu), out[0], out[1], True)
        for got, want in zip(out, (dens.grad, sh.grad)):
            assert (got.cpu().double() - want).abs().max() <= 1e-5 * want.abs().max().clamp_min(1)


@pytest.mark.parametrize("n", [10, 40000, 600000])
def test_sample_gradients_are_contiguous(gpu, n):
    """Whatever layout the backward adds into, .grad is contiguous and equals
    the explicit call's."""
    gen = torch.Generator().manual_seed(3)
    sc = scenes.make_blob_grid(96, scenes.BlobSpec(4, (0.1, 0.1), (20.0, 20.0)), gen)
    grid = _grid(sc, gpu)
    pts = (torch.rand(n, 3, generator=gen) * 2 - 1).to(gpu)
    d, s = grid.sample(pts)
    (d.sum() + s.sum()).backward()
    want = [torch.zeros(grid.sh_data.size(0), k, device=gpu) for k in (1, 27)]
    _C.sample_grid_backward(grid._to_cpp(), pts, torch.ones_like(d), torch.ones_like(s),
                            want[0], want[1], True)
    for p, w in ((grid.density_data, want[0]), (grid.sh_data, want[1])):
        assert p.grad.is_contiguous()
        assert (p.grad - w).abs().max() <= 1e-5 * w.abs().max()


@pytest.mark.parametrize("reso,layers", [(4, 2), (5, 7), (7, 8), (6, 9), (9, 17), (33, 64)])
def test_background_backward_windows(gpu, reso, layers):
    """Background gradients of the fused step for odd and even reso (columns
    wrap onto a slot of the same parity when reso is odd) and layer counts around
    multiples of 8, a third of the columns empty: within 2e-5 of the largest of
    float64 autograd; touched layers: nothing outside the trilinear cells of
    live samples, every layer with a gradient marked."""
    gen = torch.Generator().manual_seed(reso * 100 + layers)
    sc = scenes.make_blob_grid(16, scenes.BlobSpec(3, (0.2, 0.2), (3.0, 3.0)), gen)
    grid = _grid(sc, gpu)
    links = torch.arange(2 * reso * reso, dtype=torch.int32).view(2 * reso, reso)
    empty = torch.rand(2 * reso, reso, generator=gen) < 0.33
    links[empty] = -1
    links[~empty] = torch.arange(int((~empty).sum()), dtype=torch.int32)
    rows = int((~empty).sum())
    data = torch.randn(rows, layers, 4, generator=gen) * 0.5
    data[..., 3] = torch.rand(rows, layers, generator=gen)
    grid.background_nlayers, grid.background_reso = layers, reso
    grid.background_links = links.to(gpu)
    grid.background_data = torch.nn.Parameter(data.to(gpu))
    o, d = scenes.sphere_rays(300, gen, radius=0.7, target=0.6)
    gt = torch.rand(300, 3, generator=gen)
    grid.volume_render_fused(svox2_amd.Rays(o.to(gpu), d.to(gpu)), gt.to(gpu))
    g = host_grid(sc, links=grid.links.cpu().numpy())
    bg = O.Background(links.numpy(), data.double().numpy())
    data64 = data.double().requires_grad_()
    rgb = O.render_bg_fp64(g, bg, o.numpy(), d.numpy(), O.Opts(sigma_thresh=1e-8, stop_thresh=1e-7),
                           torch.from_numpy(g.density), torch.from_numpy(g.sh), data64)
    ((rgb - gt.double()) ** 2).sum().div(3 * 300).backward()
    got, want = grid.background_data.grad.cpu().double(), data64.grad
    assert (got - want).abs().max() <= 2e-5 * want.abs().max()
    marked = grid.sparse_background_indexer.cpu()
    assert marked[(want.abs() > 1e-6 * want.abs().max()).any(-1)].all()
    assert not (got[~marked] != 0).any()


@pytest.mark.parametrize("n", [1, 63, 65, 700, 4096])
@pytest.mark.parametrize("factor", [1.0, 1.7, 4.0, 12.0])
def test_fused_record_capacity(gpu, dense64, n, factor):
    """The fused call on a dense grid with workspaces from the least to twelve
    times it (records of all, some or few rays fit; one counter or one per 64
    rays): colours and touched rows those of the call without a workspace,
    gradients within 1e-5 of the largest (the order of float32 atomics)."""
    import ctypes
    _, o, d, gt, sc = dense64
    grid = _grid(sc, gpu)
    rays = svox2_amd.Rays(torch.from_numpy(o[:n]).to(gpu), torch.from_numpy(d[:n]).to(gpu))
    gt_t = torch.from_numpy(gt[:n]).to(gpu)
    lib = _C.load_library()
    least = lib.svox2_volume_render_cuvol_fused_workspace_bytes(n)
    out = []
    for nbytes in (0, int(least * factor) // 4 * 4):
        gd, gs, _, _ = grid._get_data_grads()
        gd.zero_()
        gs.zero_()
        holder = _C.GridOutputGrads()
        holder.grad_density_out, holder.grad_sh_out = gd, gs
        holder.mask_out = torch.zeros(gd.size(0), dtype=torch.bool, device=gpu)
        g = _C._grid_struct(grid._to_cpp())
        oo, dd, clip = _C._rays(rays._to_cpp())
        gstruct = _C._grads_struct(holder, g.rows, g.sh_data_dim)
        rgb = torch.empty(n, 3, device=gpu)
        ws = torch.full((max(nbytes // 4, 1),), -1, dtype=torch.int32, device=gpu)
        st = lib.svox2_volume_render_cuvol_fused(
            ctypes.byref(g), _C._ptr(oo), _C._ptr(dd), _C._ptr(clip), n,
            ctypes.byref(_C._opt_struct(grid.opt._to_cpp())), _C._ptr(gt_t), 0.0, 0.0,
            _C._ptr(rgb), None, ctypes.byref(gstruct), _C._ptr(ws) if nbytes else None, nbytes,
            _C._stream(oo))
        assert st == 0, lib.svox2_last_error()
        out.append([x.clone() for x in (rgb, holder.mask_out, gd, gs)])
    a, b = out
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    for x, y in zip(a[2:], b[2:]):
        assert (x - y).abs().max() <= 1e-5 * x.abs().max()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [100000, 100033])
def test_march_start(gpu, dtype, n):
    """The start searched for, and rays that it finds nothing on written without
    a march: colours have the same bits as in calls of fewer rays, which march
    from the grid's edge.  Depths sum the same terms in chunks that begin
    elsewhere: two float32 sums, each a tree of 5 levels and at most 20 chunks
    (96^3: under 640 samples), differ by at most 2 * 25 * 2^-24 of the depth."""
    gen = torch.Generator().manual_seed(n)
    spec = scenes.BlobSpec(3, (0.1, 0.15), (20.0, 20.0))
    grid = _grid(scenes.make_blob_grid(96, spec, gen), gpu, dtype)
    origins = torch.randn(n, 3, generator=gen)
    origins = origins / origins.norm(dim=1, keepdim=True) * 2.5
    dirs = torch.rand(n, 3, generator=gen) * 1.6 - 0.8 - origins
    dirs = dirs / dirs.norm(dim=1, keepdim=True)
    origins, dirs = origins.to(gpu), dirs.to(gpu)
    with torch.no_grad():
        rays = svox2_amd.Rays(origins, dirs)
        rgb, depth = grid.volume_render(rays), grid.volume_render_depth(rays)
        parts = [svox2_amd.Rays(origins[i:i + 30000].contiguous(), dirs[i:i + 30000].contiguous())
                 for i in range(0, n, 30000)]
        assert torch.equal(rgb, torch.cat([grid.volume_render(p) for p in parts]))
        want = torch.cat([grid.volume_render_depth(p) for p in parts])
        assert ((depth - want).abs() <= 50 * 2.0 ** -24 * want).all()
    assert 0.2 < (depth == 0).float().mean() < 0.98


def test_march_start_image(gpu):
    """An image of 317 x 331 pixels against its rays in smaller calls."""
    gen = torch.Generator().manual_seed(1)
    spec = scenes.BlobSpec(3, (0.1, 0.15), (20.0, 20.0))
    grid = _grid(scenes.make_blob_grid(96, spec, gen), gpu)
    c2w = torch.eye(4)
    c2w[2, 3] = -2.5
    cam = svox2_amd.Camera(c2w.to(gpu), 400.0, 400.0, width=317, height=331)
    with torch.no_grad():
        img = grid.volume_render_image(cam).view(-1, 3)
        rays = cam.gen_rays()
        want = torch.cat([grid.volume_render(svox2_amd.Rays(rays.origins[i:i + 30000],
                                                            rays.dirs[i:i + 30000]))
                          for i in range(0, img.size(0), 30000)])
    # The camera's rays are formed in the kernel: float32 rounding apart.
    assert (img - want).abs().max() <= 2e-4
    assert (img == grid.opt.background_brightness).all(1).float().mean() > 0.2


@pytest.mark.parametrize("width,height,batch", [(8, 4, 0), (8, 4, -1), (0, 4, 5), (8, 4, 2.5)])
def test_depth_image_refuses(gpu, dense64, width, height, batch):
    """Batches that hold no ray stay refused, though the image is one launch."""
    grid = _grid(dense64[4], gpu)
    cam = svox2_amd.Camera(torch.eye(4, device=gpu), 10.0, 10.0, width=width, height=height)
    with pytest.raises((ValueError, RuntimeError, TypeError)):
        grid.volume_render_depth_image(cam, batch_size=batch)


@pytest.mark.parametrize("n", [1, 2, 3, 33, 65])
def test_nvol_ray_counts(gpu, n):
    """Few and odd rays through both forms of the nvol backward: the fused colours
    are the forward's bits, the gradients the oracle's to the shared tolerances."""
    gen = torch.Generator().manual_seed(n)
    sc = scenes.make_blob_grid(24, scenes.BlobSpec(4, (0.2, 0.2), (20.0, 20.0)), gen)
    grid = _grid(sc, gpu)
    grid.opt.backend = "nvol"
    hg = host_grid(sc, links=grid.links.cpu().numpy())
    o, d = scenes.sphere_rays(n, gen, radius=1.8, target=0.4)
    rays = svox2_amd.Rays(o.to(gpu), d.to(gpu))
    gt = torch.rand(n, 3, generator=gen)
    spec, opt = grid._to_cpp(), grid.opt._to_cpp()
    rgb_f = _C.volume_render_nvol(spec, rays._to_cpp(), opt)
    gout = ((rgb_f.cpu().double() - gt.double()) * (2.0 / (3 * n))).numpy()
    op = grid.opt
    opts = O.Opts(op.background_brightness, op.step_size, op.sigma_thresh, op.stop_thresh,
                  op.near_clip, op.use_spheric_clip, op.last_sample_opaque)
    rgd, rgs, rmask = O.nvol_grads_fp64(hg, o.numpy(), d.numpy(), opts, gout)
    for fused in (False, True):
        gd, gs, _, _ = grid._get_data_grads()
        gd.zero_()
        gs.zero_()
        mask = torch.zeros(gd.size(0), dtype=torch.bool, device=gpu)
        holder = _C.GridOutputGrads()
        holder.grad_density_out, holder.grad_sh_out, holder.mask_out = gd, gs, mask
        if fused:
            rgb = torch.empty(n, 3, device=gpu)
            _C.volume_render_nvol_fused(spec, rays._to_cpp(), opt, gt.to(gpu), 0.0, 0.0, rgb,
                                        holder)
            assert torch.equal(rgb, rgb_f)
        else:
            _C.volume_render_nvol_backward(spec, rays._to_cpp(), opt,
                                           torch.from_numpy(gout).float().to(gpu), rgb_f, holder)
        assert_grad_close(gd.cpu().numpy().reshape(-1), rgd, "grad density")
        assert_grad_close(gs.cpu().numpy(), rgs, "grad sh")
        assert np.array_equal(mask.cpu().numpy(), rmask)


def test_cell_map_follows_its_links(gpu):
    """Links allocated where others were freed get a cell map of their own."""
    gen = torch.Generator().manual_seed(5)
    sc = scenes.make_blob_grid(64, scenes.BlobSpec(4, (0.1, 0.1), (20.0, 20.0)), gen)
    grid = _grid(sc, gpu)
    pts = (torch.rand(1 << 19, 3, generator=gen) * 2 - 1).to(gpu)
    spec = grid._to_cpp()
    for links in (grid.links.clone(), grid.links.flip(0).clone()):
        spec.links = torch.empty_like(links)
        at = spec.links.data_ptr()
        spec.links.copy_(links)
        del links
        spec.cell_map = None
        got = _C.sample_grid(spec, pts, True)
        spec.cell_map = False
        assert all(torch.equal(a, b) for a, b in zip(got, _C.sample_grid(spec, pts, True))), at
        spec.links = None
