"""The fused call's workspace: what is asked for, and the record stream at its
limits, looked into from outside ([order | per-ray state | counters | ...])."""
import ctypes

import numpy as np
import pytest
import torch

import svox2_amd
from svox2_amd import _C, scenes

pytestmark = pytest.mark.gpu


def _align(b):
    return (b + 255) // 256 * 256


def _fused(grid, rays, gt, nbytes):
    """One fused call through the C ABI with a workspace of nbytes, filled with
    ones: (colours, mask, density and SH gradients) and the workspace's words."""
    lib, n = _C.load_library(), gt.size(0)
    gd, gs, _, _ = grid._get_data_grads()
    gd.zero_()
    gs.zero_()
    holder = _C.GridOutputGrads()
    holder.grad_density_out, holder.grad_sh_out = gd, gs
    holder.mask_out = torch.zeros(gd.size(0), dtype=torch.bool, device=gd.device)
    g = _C._grid_struct(grid._to_cpp())
    o, d, _ = _C._rays(rays._to_cpp())
    gstruct = _C._grads_struct(holder, g.rows, g.sh_data_dim)
    rgb = torch.empty(n, 3, device=gd.device)
    ws = torch.full((max(nbytes // 4, 1),), -1, dtype=torch.int32, device=gd.device)
    st = lib.svox2_volume_render_cuvol_fused(
        ctypes.byref(g), _C._ptr(o), _C._ptr(d), None, n,
        ctypes.byref(_C._opt_struct(grid.opt._to_cpp())), _C._ptr(gt), 0.0, 0.0, _C._ptr(rgb),
        None, ctypes.byref(gstruct), _C._ptr(ws) if nbytes else None, nbytes, _C._stream(o))
    assert st == 0, lib.svox2_last_error()
    return (rgb, holder.mask_out, gd.clone(), gs.clone()), ws.cpu().numpy()


def _states(ws, n):
    """(per-ray states, overflow slots taken per counter)."""
    at = _align((3 * 1024 + 2 * n) * 4) // 4
    counters = at + _align(4 * n) // 4
    return ws[at:at + n], ws[counters:counters + 64]


def _grid(sc, dev, accelerate=True):
    grid = scenes.to_sparse_grid(sc, device=dev, accelerate=accelerate)
    grid.opt.sigma_thresh, grid.opt.stop_thresh = 1e-8, 1e-7
    return grid


def _with_background(grid, dev):
    grid.background_nlayers, grid.background_reso = 4, 8
    grid.background_links = torch.arange(128, dtype=torch.int32, device=dev).view(16, 8)
    grid.background_data = torch.nn.Parameter(torch.rand(128, 4, 4, device=dev))


@pytest.mark.parametrize("background,n", [(False, 4096), (True, 5000), (False, 90000)])
def test_room_is_asked_for_records_alone(gpu, dense64, background, n):
    """On a dense grid the call asks for more than the least only where it
    records: not with a background, not for batches that keep a chunk log."""
    grid = _grid(dense64[4], gpu)
    if background:
        _with_background(grid, gpu)
    lib = _C.load_library()
    o, d = scenes.sphere_rays(n, torch.Generator().manual_seed(n))
    rays, gt = svox2_amd.Rays(o.to(gpu), d.to(gpu)), torch.rand(n, 3, device=gpu)
    grid.volume_render_fused(rays, gt)  # gradients and the cell map are there
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    grid.volume_render_fused(rays, gt)
    torch.cuda.synchronize()
    used = torch.cuda.max_memory_allocated() - before
    least = lib.svox2_volume_render_cuvol_fused_workspace_bytes(n)
    beside = 24 * n + 4 * grid.sh_data.size(0) + (4 << 20)  # colours, masks, rounding
    if not background and n == 4096:
        assert used > 4 * least
    else:
        room = lib.svox2_background_workspace_bytes(n) if background else least
        assert used <= room + beside


@pytest.mark.parametrize("n", [50000, 65537])
def test_overflow_in_a_large_ordered_batch(gpu, dense64, n):
    """A dense grid and the least workspace: some rays' records fit and others'
    do not, in a batch that is ordered and whose counters are split.  Colours and
    touched rows of the call without a workspace, gradients within 1e-5 of the
    largest (the order of float32 atomics)."""
    sc = dense64[4]
    sc = scenes.SceneData(sc.links, sc.density.clamp_min(0.05), sc.sh, 9, sc.occupancy)
    grid = _grid(sc, gpu)
    gen = torch.Generator().manual_seed(n)
    o, d = scenes.sphere_rays(n, gen)
    # Half of the rays cut across an edge of the grid: about ten samples each.
    o[::2] = torch.tensor([-1.5, 0.0, 0.2])
    o[::2, 1] = torch.rand((n + 1) // 2, generator=gen) * 1.6 - 0.8
    d[::2] = torch.tensor([0.6, 0.0, 0.8])
    rays = svox2_amd.Rays(o.to(gpu), d.to(gpu))
    gt = torch.rand(n, 3, generator=gen).to(gpu)
    least = _C.load_library().svox2_volume_render_cuvol_fused_workspace_bytes(n)
    a, _ = _fused(grid, rays, gt, 0)
    b, ws = _fused(grid, rays, gt, least)
    states, _ = _states(ws, n)
    assert set(np.unique(states)) == {1, 2} and (states[::2] == 1).any()
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    for x, y in zip(a[2:], b[2:]):
        assert (x - y).abs().max() <= 1e-5 * x.abs().max()


@pytest.mark.parametrize("samples,blocks", [(7, 0), (9, 1)])
def test_a_ray_fills_its_own_slots(gpu, samples, blocks):
    """A ray has 8 slots of its own: a chunk of 7 samples and its header stay in
    them, a longer one takes an overflow block of 64."""
    planes = (samples - 1) // 2  # rows in the z planes 8 ..: samples at 7.5, 8, ...
    links = torch.full((16, 16, 16), -1, dtype=torch.int32)
    links[:, :, 8:8 + planes] = torch.arange(256 * planes, dtype=torch.int32).view(16, 16, planes)
    gen = torch.Generator().manual_seed(samples)
    sc = scenes.SceneData(links, torch.full((256 * planes, 1), 0.5, dtype=torch.float64),
                          torch.randn(256 * planes, 27, generator=gen).double(), 9, 0.2)
    grid = _grid(sc, gpu, accelerate=False)
    n = 20
    o = torch.rand(n, 3, generator=gen) - 0.5
    o[:, 2] = -1.5
    d = torch.tensor([0.0, 0.0, 1.0]).expand(n, 3).contiguous()
    rays = svox2_amd.Rays(o.to(gpu), d.to(gpu))
    gt = torch.rand(n, 3, generator=gen).to(gpu)
    a, _ = _fused(grid, rays, gt, 0)
    least = _C.load_library().svox2_volume_render_cuvol_fused_workspace_bytes(n)
    b, ws = _fused(grid, rays, gt, 4 * least)
    states, taken = _states(ws, n)
    assert (states == 1).all() and taken[0] == 64 * blocks * n
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    for x, y in zip(a[2:], b[2:]):
        assert (x - y).abs().max() <= 1e-5 * x.abs().max()
