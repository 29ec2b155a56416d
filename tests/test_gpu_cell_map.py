"""Which calls take a cell map, and whose: sampling only the one its spec
carries, so that it follows links however they were written; the renderers one
that is cached per links tensor, built before it is read on every stream."""
import pytest
import torch

from svox2_amd import _C, scenes

pytestmark = pytest.mark.gpu


def _grid(dev, reso=64, seed=7):
    gen = torch.Generator().manual_seed(seed)
    sc = scenes.make_blob_grid(reso, scenes.BlobSpec(4, (0.1, 0.1), (20.0, 20.0)), gen)
    grid = scenes.to_sparse_grid(sc, device=dev)
    grid.opt.sigma_thresh, grid.opt.stop_thresh = 1e-8, 1e-7
    return grid


def _rays(dev, n=2000, seed=3):
    import svox2_amd
    o, d = scenes.sphere_rays(n, torch.Generator().manual_seed(seed), radius=1.8, target=0.6)
    return svox2_amd.Rays(o.to(dev), d.to(dev))


def _fill_empty(links, rows):
    """Gives every empty cell some row, through .data: the version stays."""
    version = links._version
    some = torch.arange(links.numel(), dtype=torch.int32, device=links.device) % rows
    links.data.copy_(torch.where(links < 0, some.view(links.shape), links))
    assert links._version == version


@pytest.mark.parametrize("n", [40000, 600000])
def test_sample_follows_links_without_a_version(gpu, n):
    """Links changed through .data after a render: samples (and their adjoint)
    are those of the links as they are, the same bits as without any map."""
    grid = _grid(gpu)
    with torch.no_grad():
        grid.volume_render(_rays(gpu))
    pts = torch.rand(n, 3, generator=torch.Generator().manual_seed(n)).to(gpu) * 2 - 1
    _C.sample_grid(grid._to_cpp(), pts, True)
    _fill_empty(grid.links, grid.sh_data.size(0))
    bare = grid._to_cpp()
    bare.cell_map = False
    got, want = _C.sample_grid(grid._to_cpp(), pts, True), _C.sample_grid(bare, pts, True)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    grid.sample(pts)[0].sum().backward()
    weight = grid.density_data.grad.double().sum().item()
    # Every point lies among cells with rows: its 8 weights sum to 1.
    assert abs(weight - n) <= 1e-4 * n


def test_sample_inference_links(gpu):
    """Links made under inference mode have no version; they are sampled as any."""
    grid = _grid(gpu)
    pts = torch.rand(40000, 3, generator=torch.Generator().manual_seed(1)).to(gpu) * 2 - 1
    spec = grid._to_cpp()
    want = _C.sample_grid(spec, pts, True)
    with torch.inference_mode():
        spec.links = grid.links.clone()
    assert all(torch.equal(a, b) for a, b in zip(_C.sample_grid(spec, pts, True), want))


def test_captured_sample_follows_links(gpu):
    """A captured sample reads the links at each replay, whatever became of the
    renderers' cached maps in between."""
    grid = _grid(gpu)
    rays = _rays(gpu)
    pts = torch.rand(1 << 19, 3, generator=torch.Generator().manual_seed(2)).to(gpu) * 2 - 1
    spec, bare = grid._to_cpp(), grid._to_cpp()
    bare.cell_map = False
    with torch.no_grad():
        grid.volume_render(rays)
    _C.sample_grid(spec, pts, True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = _C.sample_grid(spec, pts, True)
    for step in range(4):
        graph.replay()
        want = _C.sample_grid(bare, pts, True)
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, want)), step
        if step == 0:
            grid.links[grid.links < 0] = 0
        elif step == 1:
            grid.accelerate()
        else:
            for seed in range(20 + 5 * step, 25 + 5 * step):  # drops the cached maps
                with torch.no_grad():
                    _grid(gpu, seed=seed).volume_render(rays)


@pytest.mark.parametrize("n", [1, 15, 17, 65, 1000, 40001])
def test_sample_own_map(gpu, n):
    """A spec's own map is used whatever the point count, also where the last
    wavefront's 16 points are not full: the same bits as without."""
    grid = _grid(gpu)
    pts = torch.rand(n, 3, generator=torch.Generator().manual_seed(n)).to(gpu) * 2.2 - 1.1
    spec = grid._to_cpp()
    out = []
    for cmap in (False, _C.build_cell_map(spec.links, grid.sh_data.size(0))):
        spec.cell_map = cmap
        assert bool(_C._grid_struct(spec, own_map=True).cell_map) == (cmap is not False)
        out.append(_C.sample_grid(spec, pts, True) + _C.sample_grid(spec, pts, False)[:1])
    assert all(torch.equal(a, b) for a, b in zip(*out))


@pytest.mark.parametrize("warm", [False, True])
def test_captured_render(gpu, warm):
    """A render captured before or after an eager one: an eager render between
    the capture and the first replay, and every replay, have the bits of a render
    without a map, also when the cached maps are dropped or the links change in
    between."""
    grid = _grid(gpu)
    rays = _rays(gpu)
    bare = grid._to_cpp()
    bare.cell_map = False

    def plain():
        return _C.volume_render_cuvol(bare, rays._to_cpp(), grid.opt._to_cpp())

    with torch.no_grad():
        _grid(gpu, seed=9).volume_render(rays)  # kernels loaded
        if warm:
            grid.volume_render(rays)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = grid.volume_render(rays)
        assert torch.equal(grid.volume_render(rays), plain())
        for step in range(4):
            graph.replay()
            want = plain()
            torch.cuda.synchronize()
            assert torch.equal(out, want), step
            if step == 0:
                for seed in range(30, 36):  # drops the cached map
                    _grid(gpu, seed=seed).volume_render(rays)
            elif step == 1:
                _fill_empty(grid.links, grid.sh_data.size(0))
                assert not torch.equal(plain(), want)


def test_render_on_several_streams(gpu):
    """Renders on streams that take turns without waiting for each other, each
    new grid's map wanted on all of them: the bits of a render without a map."""
    rays = _rays(gpu)
    streams = [torch.cuda.Stream() for _ in range(3)]
    grids = [_grid(gpu, seed=40 + k) for k in range(3)]
    out = []
    torch.cuda.synchronize()
    with torch.no_grad():
        for k in range(9):
            for grid in grids:
                with torch.cuda.stream(streams[k % 3]):
                    out.append((grid, grid.volume_render(rays)))
    torch.cuda.synchronize()
    for grid, got in out:
        bare = grid._to_cpp()
        bare.cell_map = False
        assert torch.equal(got, _C.volume_render_cuvol(bare, rays._to_cpp(), grid.opt._to_cpp()))


def test_map_ends_with_its_storage(gpu):
    """Two links tensors that take turns at one address (both are views of the
    same memory, each with a storage of its own) get a map each."""
    grid = _grid(gpu)
    rays = _rays(gpu)
    memory = grid.links.clone()
    spec = grid._to_cpp()
    for flip in (False, True):
        memory.copy_(grid.links.flip(0) if flip else grid.links)
        spec.links = torch.from_dlpack(memory)
        assert spec.links.data_ptr() == memory.data_ptr() and spec.links._version == 0
        out = []
        for cmap in (None, False):
            spec.cell_map = cmap
            out.append(_C.volume_render_cuvol(spec, rays._to_cpp(), grid.opt._to_cpp()))
        assert torch.equal(out[0], out[1])
        spec.links = None
