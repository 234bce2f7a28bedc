"""The lean backprojection's choice of a theta~'s views (a ballot over 64 of
them at a time, whole slabs first, the exact window table only near the
window's ends) and the row pairs of whole chains: feeds so small that a slab
has more than 64 views per theta~, view windows that cut into the slabs, a table
that moves down, odd row counts, every tile depth, against the direct kernel,
which tests each (voxel, view) pair on plain rows or quads.  Both add the same FP32 terms (the lean
kernel's mean through v_rcp_f32, 1 ulp), in another order of a theta~'s views:
sums over at most a few hundred theta~ differ by rounding, 2e-5 of the largest
voxel.
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


@pytest.mark.parametrize("tile_z", [4, 8, 16, 32])
@pytest.mark.parametrize("rows,feed_rows,ppr,rotations,slices,down,channels,precision",
                         [(8, 0.2, 12, 90.0, 17, False, 96, "fp32"),
                          (8, 0.2, 12, 90.0, 17, True, 96, "fp16"),
                          (16, 4.0, 48, 8.0, 40, False, 96, "fp32"),
                          (16, 6.0, 48, 6.0, 9, True, 96, "bf16"),
                          (11, 9.0, 64, 4.0, 20, True, 96, "fp32"),
                          (11, 9.0, 64, 4.0, 20, False, 300, "fp32"),
                          (12, 9.0, 64, 4.0, 20, False, 257, "fp32"),
                          (11, 9.0, 64, 4.0, 20, False, 96, "fp16"),
                          (11, 9.0, 64, 4.0, 20, False, 300, "bf16"),
                          (12, 9.0, 64, 4.0, 20, True, 257, "fp16"),
                          (12, 9.0, 32, 4.0, 20, True, 1100, "fp16")])
def test_view_choice_against_direct(ctx, tile_z, rows, feed_rows, ppr, rotations, slices, down,
                                    channels, precision):
    from freect_amd import wfbp
    w = S.tiny(nx=26, n_slices=slices, n_rows=rows, ppr=ppr, rotations=rotations, seed=5,
               n_channels=channels)
    feed = feed_rows * w.scan.effective().csw * (-1.0 if down else 1.0)
    scan = w.scan.replace(feed=feed, z0=-0.5 * (w.scan.n_views - 1) * feed / ppr)
    raw = ctx.phantom_project(scan, w.phantom, 0.0, w.seed)
    vols = []
    for variant in (1, 2):
        p = wfbp.Plan(ctx, scan, w.recon, precision=precision, tile_z=tile_z, bp_variant=variant)
        v = p.alloc_volume().fill_(float("nan"))
        p.reconstruct(raw, v)
        p.synchronize()
        vols.append(v)
    assert vols[0].abs().max() > 0
    assert (vols[1] - vols[0]).abs().max() <= 2e-5 * vols[0].abs().max()


@pytest.mark.parametrize("rows,channels", [(8, 96), (11, 300)])
def test_forward_volume_layouts(ctx, rows, channels):
    # The chain to the native volume through row pairs, through rows (no room
    # for pairs) and through the stage calls: the same arithmetic, bitwise.
    from freect_amd import wfbp
    w = S.tiny(nx=26, n_slices=20, n_rows=rows, rotations=3.0, seed=5, n_channels=channels)
    raw = ctx.phantom_project(w.scan, w.phantom, 0.0, w.seed)
    p = wfbp.Plan(ctx, w.scan, w.recon)
    ref, vol = p.alloc_native(), p.alloc_native().fill_(float("nan"))
    p.forward_native(raw, ref)
    p.forward_volume(raw, vol)
    p.synchronize()
    assert ref.abs().max() > 0 and torch.equal(vol, ref)
    n = p.info.filtered_bytes
    buf = torch.full((2 * n,), 255, dtype=torch.uint8, device="cuda")   # NaNs
    call = wfbp.load_library().fct_wfbp_gpu_forward_native
    for off, size in ((0, n), (4, 2 * n - 4)):   # rows: too small, and misaligned, for pairs
        vol.fill_(float("nan"))
        assert call(p.h, raw.data_ptr(), buf.data_ptr() + off, size, vol.data_ptr()) == 0
        p.synchronize()
        assert torch.equal(vol, ref)
    assert call(p.h, raw.data_ptr(), buf.data_ptr(), n - 1, vol.data_ptr()) == 1


@pytest.mark.parametrize("rows,nx", [(9, 60), (8, 61), (8, 8)])
def test_matched_backprojection_of_row_pairs(ctx, rows, nx):
    # Volumes large enough for the row pairs, and one that is not, against
    # the projector that is its transpose: <M x, y> = <x, M^T y>, positive x
    # and y, so that the FP32 rounding of sums of at most a few thousand terms
    # stays below 1e-5 of the product.
    from freect_amd import wfbp
    w = S.tiny(nx=nx, n_slices=19, n_rows=rows, rotations=2.5, seed=5)
    p = wfbp.Plan(ctx, w.scan, w.recon)
    gen = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.rand((p.info.n_slices_native, nx, nx), device="cuda", generator=gen)
    y = p.alloc_lines()
    y.copy_(torch.rand(y.shape, device="cuda", generator=gen))
    px, py = p.alloc_lines(), p.alloc_native().fill_(float("nan"))
    p.matched_project(x, px)
    p.matched_backproject(y, py)
    p.synchronize()
    a, b = (px.double() * y.double()).sum().item(), (x.double() * py.double()).sum().item()
    assert a > 0 and abs(a - b) <= 1e-5 * a


def test_forward_volume_with_adaptive_filtration(ctx):
    # On a plan with adaptive filtration the chain to the native volume filters
    # the raw scan as the stage calls do (the same values from the same views:
    # bitwise), and so does the forward pass of autograd.wfbp.
    from freect_amd import autograd, wfbp
    w = S.tiny(nx=26, n_slices=20, rotations=3.0, seed=5)
    raw = ctx.phantom_project(w.scan, w.phantom, 1e4, w.seed)
    recon = w.recon.replace(adaptive_filtration_s=0.3)
    p = wfbp.Plan(ctx, w.scan, recon, adaptive_filtration=True)
    plain = wfbp.Plan(ctx, w.scan, recon)
    ref, vol, other = p.alloc_native(), p.alloc_native().fill_(float("nan")), p.alloc_native()
    p.forward_native(raw, ref)
    p.forward_volume(raw, vol)
    plain.forward_volume(raw, other)
    torch.cuda.synchronize()
    assert torch.equal(vol, ref) and not torch.equal(other, ref)
    assert torch.equal(autograd.wfbp(raw, p), ref)
