"""The backprojection's theta~ segments (small volumes): view counts that the
segments do not divide, too few theta~ for several, every tile depth, and
volumes of one tile and of partial slabs, against the direct kernel, which
sweeps each voxel's theta~ in one sum.  Both add the same FP32 terms (the
lean kernel's mean through v_rcp_f32, 1 ulp), so their sums over at most a few
hundred theta~ differ by rounding: 2e-5 of the largest voxel.
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
@pytest.mark.parametrize("ppr,nx,slices,precision", [(6, 8, 1, "fp32"), (20, 9, 5, "fp32"),
                                                     (130, 30, 13, "fp16"), (354, 64, 33, "fp32"),
                                                     (96, 200, 20, "bf16")])
def test_segments_against_direct(ctx, tile_z, ppr, nx, slices, precision):
    from freect_amd import wfbp
    w = S.tiny(nx=nx, n_slices=slices, ppr=ppr, rotations=2.5, seed=3)
    raw = ctx.phantom_project(w.scan, w.phantom, 0.0, w.seed)
    vols = []
    for variant in (1, 2):
        p = wfbp.Plan(ctx, w.scan, w.recon, precision=precision, tile_z=tile_z,
                      bp_variant=variant)
        v = p.alloc_volume().fill_(float("nan"))
        p.reconstruct(raw, v)
        p.synchronize()
        vols.append(v)
    assert vols[0].abs().max() > 0
    assert (vols[1] - vols[0]).abs().max() <= 2e-5 * vols[0].abs().max()
