"""The table-driven ray projector and its gathered transpose at the sizes
where they can go wrong: matrices that are not multiples of the 8 x 8 tiles or
of the 32 x 32 transposition, one slice more than a slab, odd row and channel
counts, a falling slice grid, coarse voxels, FFS, an off-centre field -- and
a geometry and a graph capture that take the general kernels.  Each against
the FP64 restatement; the bound is that of the FP32 sample positions (a few
ulps of a position of up to ~600 voxels, 2e-5 of the largest output), as for
the general kernels.
"""
import numpy as np
import pytest

from freect_amd import scans as S
from helpers import gpu_ctx, to_np

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return gpu_ctx()


def _setup(nx, ny, nz, rows, chans, fov, ffs=0, flip=False, rotation=1, ppr=96):
    w = S.tiny(nx=nx, n_slices=nz, n_channels=chans, n_rows=rows, ppr=ppr, rotations=1.2,
               ffs_mode=ffs)
    rc = w.recon.replace(ny=ny, recon_fov=fov, x_origin=-6.0, y_origin=4.0)
    if flip:
        rc = rc.replace(start_pos=rc.end_pos, end_pos=rc.start_pos)
    return w.scan.replace(rotation=rotation, angle0=0.4), rc


CASES = [dict(nx=33, ny=21, nz=2, rows=8, chans=96, fov=300.0),
         dict(nx=40, ny=17, nz=17, rows=11, chans=130, fov=350.0, rotation=-1),
         dict(nx=9, ny=64, nz=33, rows=16, chans=65, fov=120.0, flip=True),
         dict(nx=70, ny=70, nz=16, rows=9, chans=200, fov=400.0, ffs=1),
         dict(nx=31, ny=30, nz=12, rows=7, chans=97, fov=250.0, ffs=2, flip=True),
         # Outside the tables' rule: the volume's corners pass the focal spot.
         dict(nx=24, ny=24, nz=6, rows=8, chans=96, fov=900.0)]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_ray_pair_matches_oracle(ctx, oracle, case):
    from freect_amd import wfbp
    sc, rc = _setup(**CASES[case])
    p = wfbp.Plan(ctx, sc, rc)
    nz = p.info.n_slices_native
    gen = torch.Generator(device="cuda").manual_seed(case)
    x = torch.rand((nz, rc.ny, rc.nx), device="cuda", generator=gen)
    y = torch.rand((sc.n_views, sc.n_rows, sc.n_channels), device="cuda", generator=gen)
    px, pty = p.alloc_raw().fill_(float("nan")), p.alloc_native().fill_(float("nan"))
    for _ in range(2):   # first use builds the tables, the second reuses them
        p.ray_project(x, px)
        p.ray_backproject(y, pty)
    p.synchronize()
    ref = oracle.ray_project(sc, rc, to_np(x).astype(np.float64))
    reft = oracle.ray_backproject(sc, rc, to_np(y).astype(np.float64), nz)
    e = np.abs(to_np(px) - ref).max() / np.abs(ref).max()
    et = np.abs(to_np(pty) - reft).max() / np.abs(reft).max()
    assert e < 2e-5 and et < 2e-5, (e, et)


def test_first_call_inside_a_capture(ctx):
    # No table may be allocated inside a capture: the general kernels are
    # recorded, and later calls outside agree with the replays.
    from freect_amd import wfbp
    sc, rc = _setup(**CASES[1])
    p = wfbp.Plan(ctx, sc, rc)
    x = torch.rand((p.info.n_slices_native, rc.ny, rc.nx), device="cuda")
    px, pt = p.alloc_raw(), p.alloc_native()
    s = torch.cuda.Stream()
    p.set_stream(s)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        p.ray_project(x, px)
        p.ray_backproject(px, pt)
    for _ in range(3):
        px.zero_()
        pt.zero_()
        g.replay()
        torch.cuda.synchronize()
        a, b = px.clone(), pt.clone()
    qx, qt = p.alloc_raw(), p.alloc_native()
    p.ray_project(x, qx)
    p.ray_backproject(qx, qt)
    p.synchronize()
    assert (a - qx).abs().max() <= 2e-5 * qx.abs().max()
    assert (b - qt).abs().max() <= 2e-5 * qt.abs().max()


def test_volume_beyond_the_paired_copies(ctx):
    # A volume whose padded copies exceed 4 GiB with two slices per entry: the
    # copies hold one.  Its only nonzero slices are those of a small plan on
    # the same grid (two slices per entry).  Slice positions of up to ~1100
    # slices carry half an ulp, 1.2e-4 slices, twice (the ray's start and the
    # sample): at most 2.4e-4 of a difference of neighbouring values, a third
    # on average against a mean value of a half: 2e-4 of the largest output.
    from freect_amd import wfbp
    sc, rc = _setup(nx=512, ny=512, nz=2, rows=8, chans=96, fov=300.0, ppr=24)
    csw = sc.effective().csw
    big = wfbp.Plan(ctx, sc, rc.replace(start_pos=-1020 * csw, end_pos=1020.5 * csw))
    small = wfbp.Plan(ctx, sc, rc.replace(start_pos=-8 * csw, end_pos=7.5 * csw))
    nz, ns = big.info.n_slices_native, small.info.n_slices_native
    assert ns == 16 and (nz + 4) * 516 * 516 * 8 > 4294967000 > (nz + 4) * 516 * 516 * 4
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand((ns, 512, 512), device="cuda", generator=gen)
    xb = torch.zeros((nz, 512, 512), device="cuda")
    xb[1012:1012 + ns] = x
    a, b = small.alloc_raw().fill_(float("nan")), big.alloc_raw().fill_(float("nan"))
    small.ray_project(x, a)
    big.ray_project(xb, b)
    small.synchronize()
    big.synchronize()
    assert a.abs().max() > 0
    assert (a - b).abs().max() <= 2e-4 * a.abs().max()


def test_rays_on_the_diagonal(ctx):
    # Rays within an FP32 rounding of 45 degrees, of which the in-plane
    # direction and the direction with the row's slope round to different plane
    # axes: the projector and its transpose take the same one.  One ray at a
    # time, <P x, e> = <x, P^T e> with positive x: sums of at most 4 x 40 FP32
    # terms each way, 1e-5 of the product.
    import math

    from freect_amd import wfbp
    w = S.tiny(nx=40, n_slices=20, n_rows=16, rotations=0.1)
    sc, chan = w.scan, 30
    beta = (chan - sc.central_channel) * sc.channel_spacing / sc.dsd
    height = (np.arange(sc.n_rows) - sc.central_row) * sc.row_spacing

    def x_planes(scan, length):
        d = scan.dsd * np.array([math.cos(scan.angle0 + beta), math.sin(scan.angle0 + beta)])
        u = np.abs((d[:, None] / length).astype(np.float32))
        return u[0] >= u[1]

    tried = 0
    for off in np.linspace(-6e-8, 6e-8, 13):
        scan = sc.replace(angle0=1.25 * math.pi - beta + float(off))
        rows = np.flatnonzero(x_planes(scan, scan.dsd) != x_planes(scan, np.hypot(scan.dsd, height)))
        if rows.size == 0:
            continue
        p = wfbp.Plan(ctx, scan, w.recon)
        x = torch.rand(p.alloc_native().shape, device="cuda") + 0.1
        px, e, xt = p.alloc_raw(), p.alloc_raw().zero_(), p.alloc_native()
        p.ray_project(x, px)
        for row in rows[[0, -1]]:
            e.zero_()[0, row, chan] = 1.0
            p.ray_backproject(e, xt)
            p.synchronize()
            a, b = px[0, row, chan].item(), (x.double() * xt.double()).sum().item()
            assert a > 1.0 and abs(a - b) <= 1e-5 * a, (off, row, a, b)
            tried += 1
    assert tried > 0


def test_path_length_bits(ctx):
    # Rays that cross every plane of a volume of ones: the samples' sum is the
    # plane count exactly, and the value that count times the path length per
    # plane.  Its FP32 roundings (the step along the ray, the ray's length, two
    # products) have no bias: the mean relative error of 14 400 rays is the same
    # for x and y planes but for the step's 1800 roundings of at most 2^-24 rms /
    # 3 each: 1e-9.  (A bit of the step used otherwise shifts the two means apart
    # by an ulp, 9e-8.)
    from freect_amd import wfbp
    w = S.tiny(nx=64, n_slices=40, ppr=192, rotations=3.0)
    sc, rc = w.scan.replace(angle0=0.0123), w.recon.replace(recon_fov=300.0)
    p = wfbp.Plan(ctx, sc, rc)
    x, px = p.alloc_native().fill_(1.0), p.alloc_raw()
    p.ray_project(x, px)
    p.synchronize()
    v = np.arange(sc.n_views)[:, None, None]
    r = np.arange(sc.n_rows)[None, :, None]
    c = np.arange(sc.n_channels)[None, None, :]
    th = sc.angle0 + 2.0 * np.pi / 192 * v + (c - sc.central_channel) * sc.channel_spacing / sc.dsd
    ratio = sc.dsd / np.sqrt(sc.dsd ** 2 + ((r - sc.central_row) * sc.row_spacing) ** 2)
    inner = (np.abs(sc.z0 + v * sc.feed / 192) < 50.0) & (np.abs(c - sc.central_channel) < 12.0)
    means = []
    for u, o in ((np.cos(th), np.sin(th)), (np.sin(th), np.cos(th))):
        u, o = np.abs(u * ratio), np.abs(o * ratio)
        m = np.broadcast_to(inner & (o < 0.25 * u), px.shape)
        err = to_np(px).astype(np.float64)[m] * u[m] / 300.0 - 1.0
        assert err.size == 14400 and np.abs(err).max() < 5 * 2.0 ** -24
        means.append(err.mean())
    assert abs(means[0] - means[1]) < 1e-8, means


@pytest.mark.parametrize("case", [1, 3, 4])
def test_transpose_of_sparse_rays(ctx, oracle, case):
    # Rays that are zero but for whole views, single rays at the ends of the
    # 32-channel groups, or one row: against the FP64 restatement, with its bound
    # above; scratch left by a dense call before is not read.
    from freect_amd import wfbp
    sc, rc = _setup(**CASES[case])
    p = wfbp.Plan(ctx, sc, rc)
    nz = p.info.n_slices_native
    dense, out = p.alloc_raw().fill_(float("nan")), p.alloc_native()
    gen = torch.Generator(device="cuda").manual_seed(case)
    for keep in ("view", "channels", "row", "nothing"):
        p.ray_backproject(dense, out)
        y = torch.zeros_like(dense)
        r = torch.rand(y.shape, device="cuda", generator=gen) + 0.1
        if keep == "view":
            y[sc.n_views // 2] = r[0]
        elif keep == "channels":
            for c in (0, 31, 32, 63, 64, sc.n_channels - 1):
                y[c % 7::7, :, c] = r[c % 7::7, :, c]
        elif keep == "row":
            y[:, sc.n_rows // 2] = r[:, 0]
        p.ray_backproject(y, out)
        p.synchronize()
        ref = oracle.ray_backproject(sc, rc, to_np(y).astype(np.float64), nz)
        assert np.abs(to_np(out) - ref).max() <= 2e-5 * np.abs(ref).max()
