"""The fused call's workspace: what is asked for."""
import pytest
import torch

import svox2_amd
from svox2_amd import _C, scenes

pytestmark = pytest.mark.gpu


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
