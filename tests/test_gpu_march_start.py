"""The search for a march's start (launches of 100000 rays or more with a cell
map) under every render option, against the same calls without a map, which march
from the grid's edge."""
import pytest
import torch

import svox2_amd
from svox2_amd import _C, scenes

pytestmark = pytest.mark.gpu

N = 100033
OPTIONS = {
    "spheric": {"use_spheric_clip": True},
    "spheric_near": {"use_spheric_clip": True, "near_clip": 0.35},
    "near": {"near_clip": 1.7},
    "opaque": {"last_sample_opaque": True},
    "step": {"step_size": 0.37},  # its sums round
    "thresh": {"sigma_thresh": 0.3},
    "black": {"background_brightness": 0.0},
    "background": {},
    "bf16": {"step_size": 0.7, "last_sample_opaque": True},
}


def _grid(gpu, name):
    gen = torch.Generator().manual_seed(5)
    sc = scenes.make_blob_grid(96, scenes.BlobSpec(3, (0.1, 0.15), (20.0, 20.0)), gen)
    grid = scenes.to_sparse_grid(sc, device=gpu,
                                 dtype=torch.bfloat16 if name == "bf16" else torch.float32)
    grid.opt.sigma_thresh, grid.opt.stop_thresh = 1e-8, 1e-7
    for key, value in OPTIONS[name].items():
        setattr(grid.opt, key, value)
    if name == "background":
        grid.background_nlayers, grid.background_reso = 6, 16
        grid.background_links = torch.arange(512, dtype=torch.int32, device=gpu).view(32, 16)
        data = torch.randn(512, 6, 4, generator=gen)
        data[..., 3] = data[..., 3].abs()
        grid.background_data = torch.nn.Parameter(data.to(gpu))
    return grid, gen


def _rays(gpu, gen):
    o = torch.randn(N, 3, generator=gen)
    o = o / o.norm(dim=1, keepdim=True) * 2.5
    d = torch.rand(N, 3, generator=gen) * 1.8 - 0.9 - o
    return svox2_amd.Rays(o.to(gpu), (d / d.norm(dim=1, keepdim=True)).to(gpu))


def _specs(grid):
    spec, bare = grid._to_cpp(), grid._to_cpp()
    spec.cell_map = _C.build_cell_map(spec.links, grid.sh_data.size(0))
    bare.cell_map = False
    return spec, bare


@pytest.mark.parametrize("name", list(OPTIONS))
def test_rays(gpu, name):
    """Colours: the same bits.  First crossings: the same bits.  Expected depths
    sum the same terms in chunks that begin elsewhere, each a tree of 5 levels and
    at most 30 chunks (96^3 at a step of 0.37: under 960 samples): two such float32
    sums differ by at most 2 * 35 * 2^-24 of the depth."""
    grid, gen = _grid(gpu, name)
    rays = _rays(gpu, gen)._to_cpp()
    spec, bare = _specs(grid)
    opt = grid.opt._to_cpp()
    for ordered in (False, True):
        got = _C.volume_render_cuvol(spec, rays, opt, ordered=ordered)
        want = _C.volume_render_cuvol(bare, rays, opt, ordered=ordered)
        assert torch.equal(got, want)
    got = _C.volume_render_sigma_thresh(spec, rays, opt, 0.5)
    want = _C.volume_render_sigma_thresh(bare, rays, opt, 0.5)
    assert torch.equal(got, want) and 0.02 < (want > 0).float().mean() < 0.98
    got = _C.volume_render_expected_term(spec, rays, opt)
    want = _C.volume_render_expected_term(bare, rays, opt)
    assert ((got - want).abs() <= 70 * 2.0 ** -24 * want.abs()).all()


@pytest.mark.parametrize("name", list(OPTIONS))
@pytest.mark.parametrize("record", [True, False])  # with the chunk log, without
def test_fused(gpu, name, record):
    """The fused call: colours and touched rows the same, gradients within 1e-5 of
    the largest (the order of float32 atomics)."""
    grid, gen = _grid(gpu, name)
    rays = _rays(gpu, gen)._to_cpp()
    gt = torch.rand(N, 3, generator=gen).to(gpu)
    out = []
    for spec in _specs(grid):
        holder = _C.GridOutputGrads()
        rows = grid.sh_data.size(0)
        holder.grad_density_out = torch.zeros(rows, 1, device=gpu)
        holder.grad_sh_out = torch.zeros(rows, 27, device=gpu)
        holder.mask_out = torch.zeros(rows, dtype=torch.bool, device=gpu)
        sums = [holder.grad_density_out, holder.grad_sh_out]
        if name == "background":
            holder.grad_background_out = torch.zeros_like(grid.background_data.data)
            sums.append(holder.grad_background_out)
        rgb = torch.empty(N, 3, device=gpu)
        _C.volume_render_cuvol_fused(spec, rays, grid.opt._to_cpp(), gt, 1e-3, 1e-11, rgb, holder,
                                     record=record)
        out.append(([rgb, holder.mask_out], sums))
    assert all(torch.equal(a, b) for a, b in zip(out[0][0], out[1][0]))
    for a, b in zip(out[0][1], out[1][1]):
        assert b.abs().max() > 0 and (a - b).abs().max() <= 1e-5 * b.abs().max()


@pytest.mark.parametrize("ndc", [False, True])
@pytest.mark.parametrize("name", ["spheric", "near", "opaque", "step", "background", "bf16"])
def test_image(gpu, name, ndc):
    """An image of 331 x 303 pixels, its rays warped to NDC or not."""
    grid, _ = _grid(gpu, name)
    c2w = torch.eye(4)
    c2w[:3, 3] = torch.tensor([0.1, -0.2, 0.3 if ndc else -2.4])
    cam = svox2_amd.Camera(c2w, 300.0, 310.0, width=331, height=303,
                           ndc_coeffs=(2 * 300.0 / 331, 2 * 310.0 / 303) if ndc else (-1.0, -1.0))
    spec, bare = _specs(grid)
    got = _C.volume_render_cuvol_image(spec, cam._to_cpp(), grid.opt._to_cpp())
    want = _C.volume_render_cuvol_image(bare, cam._to_cpp(), grid.opt._to_cpp())
    assert torch.equal(got, want)
    seen = (want - want[0, 0]).abs().amax(2) > 0
    assert 0.02 < seen.float().mean()
