"""The gathered transposes of the backprojection and of the matched projector
against the scattering kernels, which a graph capture on a fresh plan records
(no scratch may be allocated inside a capture).  Both take the same FP32
selection and weights, so they differ by summation order and by the products'
rounding only: a few ulps of a detector sample's sum of up to a few thousand
terms, bounded here by 1e-5 of the largest sample.  The shapes are those where
the gather can go wrong: detector rows that leave a remainder after 16 or 32,
an off-centre row, more slices than one chunk of 64, matrices of one column
group more than 64, fine and coarse voxels, a falling slice grid, FFS.
"""
import pytest

from freect_amd import scans as S
from helpers import gpu_ctx

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return gpu_ctx()


CASES = [dict(nx=32, ny=32, n_slices=8, n_rows=8),
         dict(nx=65, ny=20, n_slices=9, n_rows=17, fov=350.0),
         dict(nx=20, ny=70, n_slices=66, n_rows=16, fov=120.0, rotations=6.0, tile_z=4),
         dict(nx=40, ny=40, n_slices=12, n_rows=33, cr=0.3, rotation=-1),
         dict(nx=130, ny=130, n_slices=3, n_rows=9, fov=200.0, flip=True),
         dict(nx=24, ny=31, n_slices=10, n_rows=12, ffs=3, ppr=192),
         dict(nx=16, ny=16, n_slices=1, n_rows=5, rotations=0.3)]


def _plan(ctx, nx, ny, n_slices, n_rows, fov=400.0, rotations=2.3, tile_z=8, cr=0.0, rotation=1,
          flip=False, ffs=0, ppr=96):
    from freect_amd import wfbp
    w = S.tiny(nx=nx, n_slices=n_slices, n_channels=96, n_rows=n_rows, ppr=ppr,
               rotations=rotations, ffs_mode=ffs)
    sc = w.scan.replace(rotation=rotation, central_row=w.scan.central_row + cr)
    rc = w.recon.replace(ny=ny, recon_fov=fov, x_origin=3.0)
    if flip:
        rc = rc.replace(start_pos=rc.end_pos, end_pos=rc.start_pos)
    return wfbp.Plan(ctx, sc, rc, tile_z=tile_z)


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("op", ["backproject_adjoint", "matched_project"])
def test_gather_equals_scatter(ctx, case, op):
    p, general = _plan(ctx, **CASES[case]), _plan(ctx, **CASES[case])
    gen = torch.Generator(device="cuda").manual_seed(case)
    x = torch.rand((p.info.n_slices_native, p.recon.ny, p.recon.nx), device="cuda",
                   generator=gen) + 0.1
    got, ref = p.alloc_lines().fill_(float("nan")), p.alloc_lines()
    for _ in range(2):   # with and without the first use's allocation
        getattr(p, op)(x, got)
    s = torch.cuda.Stream()
    general.set_stream(s)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        getattr(general, op)(x, ref)
    for _ in range(2):
        g.replay()
        torch.cuda.synchronize()
        assert ref.abs().max() > 0
        assert (got - ref).abs().max() <= 1e-5 * ref.abs().max()


@pytest.mark.parametrize("views,channels,rows,ffs", [(1, 70, 3, 0), (5, 96, 8, 0), (40, 200, 5, 0),
                                                     (8, 64, 4, 3), (130, 65, 9, 2)])
def test_rebin_transpose_at_the_scan_ends(ctx, oracle, views, channels, rows, ffs):
    # Scans shorter than the fan's reach, where most samples go to a clamped
    # first or last projection.  Sums of at most `views` terms per entry, FP32
    # weights: 1e-5 of the largest.
    import numpy as np

    from freect_amd import wfbp
    w = S.tiny(nx=8, n_slices=2, n_channels=channels, n_rows=rows, ppr=192, rotations=1.0,
               ffs_mode=ffs)
    sc = w.scan.replace(n_views=views)
    p = wfbp.Plan(ctx, sc, w.recon)
    i = p.info
    g = np.random.RandomState(views).standard_normal(
        (i.n_parallel_views, i.n_filtered_rows, i.channel_pitch)).astype(np.float32)
    out = p.alloc_raw().fill_(float("nan"))
    p.rebin_adjoint(torch.from_numpy(g).cuda(), out)
    p.synchronize()
    ref = oracle.rebin_adjoint(sc, g[..., : i.n_filtered_channels].astype(np.float64))
    assert np.abs(out.cpu().numpy() - ref).max() <= 1e-5 * np.abs(ref).max()


def test_weights_are_divided(ctx):
    # xbar scale / sum W, correctly rounded, as the scattering kernel divides:
    # one voxel on the axis and on a channel, in the plane of a view's focal
    # spot (row 3.5, both halves exact).  Three views of that theta~ see it, all
    # in the flat part of W, so that sum W = 3 and each W = 1 exactly: the two
    # samples of the middle view are x / 3 / 2 to the bit.
    import math

    import numpy as np

    from freect_amd import wfbp
    w = S.tiny(nx=9, n_slices=4, n_rows=8, ppr=96, rotations=4.0)
    dz, v = 0.1875, 200   # (half a feed: 9 mm, 0.514 of the 17.5 mm cone at the axis)
    sc = w.scan.replace(feed=dz * 96, z0=-dz * v, central_channel=48.0)
    rc = w.recon.replace(start_pos=0.0, end_pos=4 * sc.csw, recon_fov=200.0)
    p = wfbp.Plan(ctx, sc, rc)
    x, g = p.alloc_native().zero_(), p.alloc_lines()
    scale = np.float32(2.0 * math.pi / 96)
    for xb in np.random.RandomState(0).uniform(1.0, 2.0, 64).astype(np.float32):
        x[0, 4, 4] = float(xb)
        p.backproject_adjoint(x, g)
        p.synchronize()
        got = g[v, :, 48].cpu().numpy()
        want = np.zeros(8, np.float32)
        want[3:5] = xb * scale / np.float32(3.0) / np.float32(2.0)
        assert np.array_equal(got, want), (got, want)


@pytest.mark.parametrize("bad", ["inf", "-inf", "nan"])
@pytest.mark.parametrize("op", ["backproject_adjoint", "matched_project", "ray_project",
                                "ray_backproject"])
def test_nonfinite_samples(ctx, op, bad):
    # One sample that is not finite: the gathers and the table projector give
    # infinities and NaNs where the general kernels (a capture on a fresh plan)
    # give them, an infinite sample no NaN.
    from freect_amd import wfbp
    w = S.tiny(nx=40, n_slices=12, rotations=2.5)
    sc, rc = w.scan.replace(angle0=0.4), w.recon.replace(x_origin=3.1)
    p, general = wfbp.Plan(ctx, sc, rc), wfbp.Plan(ctx, sc, rc)
    x = (p.alloc_raw() if op == "ray_backproject" else p.alloc_native()).uniform_(0.1, 1.0)
    x.view(-1)[x.numel() // 2 + 11] = float(bad)
    got = {"ray_project": p.alloc_raw, "ray_backproject": p.alloc_native}.get(op, p.alloc_lines)()
    ref = torch.empty_like(got)
    getattr(p, op)(x, got)
    s = torch.cuda.Stream()
    general.set_stream(s)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        getattr(general, op)(x, ref)
    g.replay()
    torch.cuda.synchronize()
    assert not ref.isfinite().all()
    assert torch.equal(got.isnan(), ref.isnan())
    for v in (float("inf"), float("-inf")):
        assert torch.equal(got == v, ref == v)


@pytest.mark.parametrize("nx,ny,slices,fov,x0,rotations,flip",
                         [(200, 1, 9, 400.0, 0.0, 2.3, False), (1, 200, 9, 400.0, 0.0, 2.3, True),
                          (64, 64, 2, 20.0, 140.0, 9.0, False), (64, 33, 3, 60.0, -120.0, 9.0, True),
                          (48, 48, 130, 450.0, 0.0, 12.0, False),
                          (40, 90, 130, 300.0, 40.0, 12.0, True)])
@pytest.mark.parametrize("op", ["backproject_adjoint", "matched_project"])
def test_planes_left_out(ctx, op, nx, ny, slices, fov, x0, rotations, flip):
    # Volumes that most rays miss, thin ones, and ones of several chunks of
    # slices: the gather leaves out the planes where no lane of a wave has a
    # voxel.  Against the scattering kernels, with the bound of the comparison
    # above.
    from freect_amd import wfbp
    w = S.tiny(nx=nx, n_slices=slices, n_channels=192, n_rows=17, rotations=rotations)
    rc = w.recon.replace(ny=ny, recon_fov=fov, x_origin=x0, y_origin=0.4 * x0)
    if flip:
        rc = rc.replace(start_pos=rc.end_pos, end_pos=rc.start_pos)
    p, general = wfbp.Plan(ctx, w.scan, rc), wfbp.Plan(ctx, w.scan, rc)
    gen = torch.Generator(device="cuda").manual_seed(nx)
    x = torch.rand(p.alloc_native().shape, device="cuda", generator=gen) + 0.1
    got, ref = p.alloc_lines().fill_(float("nan")), p.alloc_lines()
    getattr(p, op)(x, got)
    s = torch.cuda.Stream()
    general.set_stream(s)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        getattr(general, op)(x, ref)
    g.replay()
    torch.cuda.synchronize()
    assert ref.abs().max() > 0
    assert (got - ref).abs().max() <= 1e-5 * ref.abs().max()


@pytest.mark.parametrize("channels,rows,ffs,views",
                         [(96, 5, 0, 300), (200, 17, 0, 300), (70, 33, 0, 130), (65, 9, 2, 260),
                          (64, 16, 3, 400)])
def test_rebin_transpose_of_sparse_lines(ctx, oracle, channels, rows, ffs, views):
    # Lines that are zero but for some views (the first, the last, single ones,
    # one sample), row counts on both sides of the rows that a workgroup takes at
    # a time: against the FP64 restatement, FP32 sums of a few terms per sample
    # (at the scan's ends of half a fan's views): 1e-5 of the largest.
    import numpy as np

    from freect_amd import wfbp
    w = S.tiny(nx=8, n_slices=2, n_channels=channels, n_rows=rows, ppr=192, rotations=1.0,
               ffs_mode=ffs)
    sc = w.scan.replace(n_views=views)
    p = wfbp.Plan(ctx, sc, w.recon)
    i = p.info
    shape = (i.n_parallel_views, i.n_filtered_rows, i.channel_pitch)
    rng, nv = np.random.RandomState(views), i.n_parallel_views
    for keep in ([0], [nv - 1], [nv // 2], [nv // 3, nv // 3 + 40], [], "one"):
        g = np.zeros(shape, np.float32)
        if keep == "one":
            g[nv // 2, i.n_filtered_rows - 1, i.n_filtered_channels // 2] = 1.0
        else:
            g[keep] = rng.standard_normal((len(keep),) + shape[1:])
        out = p.alloc_raw().fill_(float("nan"))
        p.rebin_adjoint(torch.from_numpy(g).cuda(), out)
        p.synchronize()
        ref = oracle.rebin_adjoint(sc, g[..., : i.n_filtered_channels].astype(np.float64))
        assert np.abs(out.cpu().numpy() - ref).max() <= 1e-5 * np.abs(ref).max()
