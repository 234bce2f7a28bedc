"""Buffers that a plan allocates on first use under captured graphs: a graph
captured after the first use holds their addresses, so they stay where they are
while the plan lives, whatever the plan is asked for later.
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


OPS = ["matched_project", "backproject_adjoint", "matched_backproject", "ray_project",
       "ray_backproject"]


def _ends(p, op):
    """Zeroed source and destination buffers of a stage call."""
    nat, raw, lines = p.alloc_native, p.alloc_raw, p.alloc_lines
    src, dst = {"matched_project": (nat, lines), "backproject_adjoint": (nat, lines),
                "matched_backproject": (lines, nat), "ray_project": (nat, raw),
                "ray_backproject": (raw, nat)}[op]
    return src().zero_(), dst().zero_()


@pytest.mark.parametrize("op", OPS)
def test_capture_between_first_uses(ctx, op):
    # Warm one call, capture it, run every other call of the plan (some need
    # more scratch than the captured one), overwrite whatever was freed, and
    # replay on new inputs.  The replay runs the eager call's kernels, whose
    # sums of at most a few thousand FP32 terms may be split among waves and
    # added in any order: 1e-5 of the largest.
    from freect_amd import wfbp
    w = S.tiny(nx=60, n_slices=19, rotations=2.5)
    p = wfbp.Plan(ctx, w.scan, w.recon)
    s = torch.cuda.Stream()
    p.set_stream(s)
    gen = torch.Generator(device="cuda").manual_seed(3)
    x, y = _ends(p, op)
    torch.cuda.synchronize()
    getattr(p, op)(x, y)
    p.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        getattr(p, op)(x, y)
    others = [(o, _ends(p, o)) for o in OPS if o != op]
    torch.cuda.synchronize()
    for o, (a, b) in others:
        getattr(p, o)(a, b)
    p.synchronize()
    junk = [torch.full((1 << k,), float("nan"), device="cuda") for k in range(10, 28)]
    for _ in range(3):
        x.uniform_(0.1, 1.0, generator=gen)
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        ref = torch.full_like(y, float("nan"))
        torch.cuda.synchronize()
        getattr(p, op)(x, ref)
        p.synchronize()
        assert ref.abs().max() > 0
        assert (y - ref).abs().max() <= 1e-5 * ref.abs().max()
    del junk


@pytest.mark.parametrize("mode", ["global", "thread_local"])
@pytest.mark.parametrize("op", OPS)
def test_first_use_beside_a_capture(ctx, op, mode):
    # The first call of a plan while another stream is being captured: the
    # capture stays valid and holds its own work only, and the call gives what
    # it gives outside (the same kernels; sums of atomics, 1e-5 of the largest).
    from freect_amd import wfbp
    w = S.tiny(nx=60, n_slices=19, rotations=2.5)
    p = wfbp.Plan(ctx, w.scan, w.recon)
    p.set_stream(torch.cuda.Stream())
    x, y = _ends(p, op)
    x.uniform_(0.1, 1.0)
    ref, a = torch.full_like(y, float("nan")), torch.zeros(64, device="cuda")
    y.fill_(float("nan"))
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=torch.cuda.Stream(), capture_error_mode=mode):
        a.add_(1.0)
        getattr(p, op)(x, y)
    torch.cuda.synchronize()
    first = y.clone()
    y.fill_(float("nan"))
    for _ in range(3):
        g.replay()
    torch.cuda.synchronize()
    assert a.eq(3.0).all() and y.isnan().all()
    getattr(p, op)(x, ref)
    p.synchronize()
    assert ref.abs().max() > 0
    assert (first - ref).abs().max() <= 1e-5 * ref.abs().max()
