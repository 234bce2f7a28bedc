"""The work a user of this framework has it do, as cases that can be timed.

listed() names the cases, draw() gives more of the same ranges, prepare() makes
what a user's program holds before the call (a scan or a volume on the GPU, or
a scan in pinned host memory, and the plan), run() is one pass through the
public entry points, work() what a pass cannot do without, and exact() the
same results in plain torch in 64 bits.

Kinds of work:
  recon    raw scan -> volume, the whole chain on the GPU (Plan.reconstruct);
  host     the same from pinned host memory to pinned host memory, streamed
           (Plan.reconstruct_host);
  batch    several uneven jobs recorded together and replayed (Batch.run);
  lines    the rebinning and ramp filter alone (Plan.rebin_filter), what the
           stage calls, the host driver and a filter comparison use;
  wfbp     the chain to the native volume and its gradient (autograd.wfbp);
  ray      the ray-driven projector and its transpose, one pass forward and
           backward (autograd.ray_project): a refinement step's work;
  matched  the voxel-driven projector pair on the parallel rows, one pass
           each way (Plan.matched_project, Plan.matched_backproject).

Sizes are those of the repository's own workloads (freect_amd/scans.py: the
888 x 64 and 736 x 16 detectors, the flying-focal-spot scan, the batch jobs,
the refinement scan) or cut down from them.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from freect_amd import autograd as A
from freect_amd import scans as S
from freect_amd import wfbp

# Every field of a case and its default.
FIELDS = dict(kind="recon", channels=736, rows=16, row_mm=0.625, ppr=1152, rotations=2.0,
              pitch=1.0, nx=256, ny=256, fov=250.0, length=20.0, thickness=1.25, spacing=1.25,
              filter="ramp", precision="fp32", ffs=0, clockwise=False, hu=False, adaptive=0.0,
              i0=0.0, jobs=1)


def _case(**kw):
    bad = set(kw) - set(FIELDS) - {"name"}
    if bad:
        raise ValueError(f"unknown fields {bad}")
    return {**FIELDS, **kw}


def listed():
    return [
        # A reconstruction of the size that smoke and unit tests use: what a
        # call costs when there is hardly any work in it.
        _case(name="recon_smoke_fp32", channels=160, rows=8, row_mm=5.0, ppr=160, rotations=3.0,
              nx=48, ny=48, fov=400.0, length=40.0, thickness=5.0, spacing=5.0),
        # The `small` workload: a 16-row scan, 256 x 256, 32 slices.
        _case(name="recon_small_fp32", rotations=2.0, length=40.0, filter="shepp-logan"),
        # A region of a 64-row scan on an odd grid, thick overlapping slices in
        # HU, a clockwise gantry, plain FP32: a routine clinical series.
        _case(name="recon_region_fp32", channels=888, rows=64, ppr=984, pitch=0.984,
              rotations=3.4, nx=500, ny=381, fov=350.0, length=55.0, thickness=3.0, spacing=1.5,
              filter="hann", clockwise=True, hu=True, i0=5e4),
        # The `full` workload on the mixed-precision path: 512 x 512 x 320
        # from ten rotations of a 64-row scan.
        _case(name="recon_full_fp16", channels=888, rows=64, ppr=984, pitch=0.984,
              rotations=10.0, nx=512, ny=512, fov=500.0, length=200.0, thickness=0.625,
              spacing=0.625, precision="fp16", i0=5e4),
        # The flying-focal-spot scan (phi + z, 1472 interleaved channels), cut
        # to three rotations.
        _case(name="recon_ffs_fp16", channels=736, rows=32, row_mm=0.6, ppr=2304, pitch=0.8,
              rotations=3.0, nx=512, ny=512, fov=500.0, length=24.0, thickness=1.0, spacing=1.0,
              filter="sharp", precision="fp16", ffs=3, i0=2.5e4),
        # A low-dose series with adaptive filtration, BF16 storage, high pitch.
        _case(name="recon_adaptive_bf16", pitch=1.375, rotations=5.0, nx=256, ny=256, fov=500.0,
              length=40.0, thickness=2.5, spacing=2.5, filter="hann", precision="bf16",
              adaptive=0.3, i0=1e4),
        # A scan that arrives in host memory and a volume that goes back there.
        _case(name="host_fp16", kind="host", channels=888, rows=64, ppr=984, pitch=0.984,
              rotations=3.5, nx=512, ny=512, fov=500.0, length=60.0, thickness=1.25,
              spacing=1.25, precision="fp16", i0=5e4),
        # Uneven jobs of a work list run together.
        _case(name="batch_fp16", kind="batch", jobs=6, precision="fp16", length=30.0, i0=5e4),
        # The rebinning and filter of a whole three-rotation 64-row scan.
        _case(name="lines_fp32", kind="lines", channels=888, rows=64, ppr=984, pitch=0.984,
              rotations=3.0, length=40.0, i0=5e4),
        # Gradients through the reconstruction (a loss on the volume).
        _case(name="wfbp_grad", kind="wfbp", ppr=984, rotations=3.0, nx=384, ny=384, fov=500.0,
              length=20.0, i0=5e4),
        # One data-consistency step's projector work on the refinement scan's
        # detector, one and a half rotations.
        _case(name="ray_grad", kind="ray", ppr=984, rotations=1.5, nx=384, ny=384, fov=500.0,
              length=20.0),
        # The voxel-driven pair, forward and back.
        _case(name="matched_grad", kind="matched", ppr=984, rotations=2.0, nx=256, ny=256,
              fov=500.0, length=20.0),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """One more case: detector, scan, matrix and options spread over the
    ranges of the listed ones, never more work than the largest of its kind."""
    kind = rng.choice(["recon", "recon", "recon", "host", "batch", "lines", "wfbp", "ray",
                       "matched"])
    limit = {"recon": 6.3e10, "host": 1.6e10, "batch": 1.2e10, "lines": 6.3e10, "wfbp": 3.6e9,
             "ray": 6.0e9, "matched": 1.6e9}[kind]
    while True:
        ffs = rng.choice([1, 2, 3]) if kind == "recon" and rng.random() < 0.2 else 0
        channels = int(_log(rng, 96, 888))
        rows = rng.choice([8, 11, 16, 23, 32, 64])
        if ffs:
            channels, rows = min(channels, 736), min(rows, 32)
        ppr = 8 * int(_log(rng, 20, 144)) * (2 if ffs == 3 else 1)
        row_mm = rng.choice([0.5, 0.625, 1.25]) if rows > 8 else rng.choice([1.25, 2.5, 5.0])
        pitch = rng.choice([0.516, 0.8, 0.984, 1.0, 1.375])
        feed = pitch * rows * row_mm
        length = min(_log(rng, 4, 200) * row_mm, 200.0, 18 * feed)
        length = max(length, 4 * row_mm)
        nx = int(_log(rng, 32, 512))
        ny = nx if rng.random() < 0.6 else int(_log(rng, 32, 512))
        thick = rng.choice([1.0, 2.0, 3.7]) * row_mm
        c = _case(kind=kind, channels=channels, rows=rows, row_mm=row_mm, ppr=ppr,
                  rotations=round(length / feed + rng.uniform(1.2, 2.4), 2), pitch=pitch, nx=nx,
                  ny=ny, fov=rng.choice([200.0, 350.0, 500.0]), length=round(length, 3),
                  thickness=thick, spacing=thick * rng.choice([0.5, 1.0]),
                  filter=rng.choice(["ramp", "shepp-logan", "hann", "medium"]), ffs=ffs,
                  clockwise=rng.random() < 0.3, hu=kind in ("recon", "host") and
                  rng.random() < 0.3, i0=rng.choice([0.0, 1e4, 5e4]))
        if kind in ("recon", "host", "batch"):
            c["precision"] = rng.choice(["fp32", "fp32", "fp16", "fp16", "bf16"])
        if kind == "recon" and rng.random() < 0.2:
            c["adaptive"] = rng.choice([0.2, 0.5])
        if kind == "batch":
            c["jobs"] = rng.randint(2, 8)
            c["nx"] = c["ny"] = min(nx, 256)
        if kind == "lines":
            c["precision"] = "fp32"
        if _units(c) <= limit and _rays(c) <= 5.7e8:
            return c


# --------------------------------------------------------------------------
# Geometry of a case.
# --------------------------------------------------------------------------
def _scan(c):
    r, dsd = (595.0, 1085.6) if c["ffs"] else (541.0, 949.0)
    n = c["channels"]
    dgamma = 2.0 * math.asin(250.0 / r) / (n - 1)
    det = dict(n_channels=n, n_rows=c["rows"], views_per_rotation=c["ppr"],
               channel_spacing=dgamma * dsd, row_spacing=c["row_mm"] * dsd / r, dsd=dsd, r=r,
               central_channel=0.5 * (n - 1) + 0.25, central_row=0.5 * (c["rows"] - 1))
    scan = S.helical(det, pitch=c["pitch"], rotations=c["rotations"], angle0=0.1)
    if c["ffs"]:
        scan = scan.replace(ffs_mode=c["ffs"], anode_angle=0.1222)
    if c["clockwise"]:
        scan = scan.replace(rotation=-1)
    return scan


def _recon(c):
    return S.ReconConfig(start_pos=-0.5 * c["length"], end_pos=0.5 * c["length"],
                         recon_fov=c["fov"], slice_thickness=c["thickness"],
                         slice_pitch=c["spacing"], nx=c["nx"], ny=c["ny"], filter=c["filter"],
                         adaptive_filtration_s=c["adaptive"])


def _jobs(c):
    """The jobs of a batch: scan lengths, pitches, matrices, slice widths and
    filters differ from job to job, by a rule on the job's number."""
    jobs = []
    for j in range(c["jobs"]):
        f = (0.6, 1.0, 1.5, 0.8, 1.9, 0.7, 1.2, 0.9)[j % 8]
        pitch = (0.516, 0.984, 1.375)[j % 3]
        length = c["length"] * f
        n = int(c["nx"] * (1.0, 1.5, 0.75)[j % 3])
        jobs.append({**c, "kind": "recon", "pitch": pitch, "length": length, "nx": n, "ny": n,
                     "rotations": round(length / (pitch * c["rows"] * c["row_mm"]) + 2.0, 2),
                     "filter": ("ramp", "shepp-logan", "hann")[j % 3]})
    return jobs


def _native(c):
    """Native slices (spacing: the effective detector row at the isocentre)."""
    step = c["row_mm"] / (2 if c["ffs"] & 2 else 1)
    return max(1, math.ceil(c["length"] / step - 1e-9))


def _rays(c):
    return int(round(c["rotations"] * c["ppr"])) * c["rows"] * c["channels"]


def _voxel_views(c):
    """(voxel in the FOV, view that sees it) pairs, as the geometry gives them
    for a volume inside the scan."""
    if c["kind"] == "batch":
        return sum(_voxel_views(j) for j in _jobs(c))
    dx, dy = c["fov"] / c["nx"], c["fov"] / c["ny"]
    cols = min(c["nx"] * c["ny"], math.pi * 250.0 ** 2 / (dx * dy))
    ppr = c["ppr"] / {0: 1, 1: 2, 2: 2, 3: 4}[c["ffs"]]
    return cols * _native(c) * ppr * min(1.0 / c["pitch"], c["rotations"])


def _units(c):
    """What bounds a kind's work: voxel-views, rays times planes, or rays."""
    if c["kind"] == "ray":
        return _rays(c) * 0.5 * (c["nx"] + c["ny"])
    if c["kind"] == "lines":
        return _rays(c) * 100.0
    return _voxel_views(c)


# --------------------------------------------------------------------------
# The calls.
# --------------------------------------------------------------------------
def _raw(ctx, c, scan, seed):
    ph = S.make_phantom(seed, -0.5 * c["length"], 0.5 * c["length"])
    return ctx.phantom_project(scan, ph, c["i0"], seed)


def _volume(plan, c, seed):
    """A reconstructed volume: water cylinder, inserts and noise, 1/mm."""
    z, y, x = plan.info.n_slices_native, c["ny"], c["nx"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    fy = (torch.arange(y, device="cuda") - 0.5 * (y - 1)) * (c["fov"] / y)
    fx = (torch.arange(x, device="cuda") - 0.5 * (x - 1)) * (c["fov"] / x)
    r2 = fy[:, None] ** 2 + fx[None, :] ** 2
    plane = torch.where(r2 < 150.0 ** 2, S.MU_WATER, 0.0)
    rs = np.random.RandomState(seed % (1 << 31))
    for _ in range(6):
        cx, cy, rad = rs.uniform(-100, 100), rs.uniform(-100, 100), rs.uniform(8, 40)
        hit = (fy[:, None] - cy) ** 2 + (fx[None, :] - cx) ** 2 < rad * rad
        plane = plane + torch.where(hit, S.MU_WATER * rs.uniform(-0.9, 1.0), 0.0)
    noise = torch.randn((z, y, x), device="cuda", generator=g) * (0.03 * S.MU_WATER)
    return (plane[None] + noise).float().contiguous()


def _randn(shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, device="cuda", generator=g)


def _inputs(ctx, plan, c, scan, seed):
    """Inputs of a gradient kind: what goes in and the gradient that comes
    back to its output."""
    nat = (plan.info.n_slices_native, c["ny"], c["nx"])
    raw = (scan.n_views, scan.n_rows, scan.n_channels)
    if c["kind"] == "wfbp":
        return _raw(ctx, c, scan, seed), _randn(nat, seed + 1) * 1e-3
    if c["kind"] == "matched":
        g = _randn(raw, seed + 1) * 0.05
        return _volume(plan, c, seed), torch.nn.functional.pad(
            g, (0, plan.info.channel_pitch - scan.n_channels))
    return _volume(plan, c, seed), _randn(raw, seed + 1) * 0.05


def prepare(case, seed):
    c = {**FIELDS, **case}
    ctx = wfbp.Context(0)
    st = {"case": c, "ctx": ctx}
    if c["kind"] == "batch":
        jobs = _jobs(c)
        st["batch"] = wfbp.Batch(ctx, [(_scan(j), _recon(j)) for j in jobs],
                                 precision=c["precision"])
        st["raw"] = [_raw(ctx, j, _scan(j), seed + k) for k, j in enumerate(jobs)]
        st["vol"] = [p.alloc_volume() for p in st["batch"].plans]
        for k, (r, v) in enumerate(zip(st["raw"], st["vol"])):
            st["batch"].submit(k, r, v)
        return st
    scan = _scan(c)
    plan = st["plan"] = wfbp.Plan(ctx, scan, _recon(c), precision=c["precision"],
                                  adaptive_filtration=c["adaptive"] > 0.0)
    if c["hu"]:
        plan.set_output_units("hu")
    if c["kind"] in ("wfbp", "ray", "matched"):
        st["x"], st["g"] = _inputs(ctx, plan, c, scan, seed)
        if c["kind"] == "matched":
            st["lines"], st["native"] = plan.alloc_lines(), plan.alloc_native()
        return st
    st["raw"] = _raw(ctx, c, scan, seed)
    if c["kind"] == "lines":
        st["out"], _ = plan.alloc_filtered()
    elif c["kind"] == "host":
        st["raw"] = torch.empty(st["raw"].shape, pin_memory=True).copy_(st["raw"])
        shape = (plan.info.n_slices_requested, c["ny"], c["nx"])
        st["out"] = torch.empty(shape, pin_memory=True).numpy()
    else:
        st["vol"] = plan.alloc_volume()
    return st


def run(st):
    kind = st["case"]["kind"]
    if kind == "recon":
        st["plan"].reconstruct(st["raw"], st["vol"])
        return st["vol"]
    if kind == "host":
        return st["plan"].reconstruct_host(st["raw"], out=st["out"])
    if kind == "batch":
        st["batch"].run()
        return st["vol"]
    if kind == "lines":
        st["plan"].rebin_filter(st["raw"], st["out"])
        return st["plan"].filtered_view(st["out"])
    if kind == "matched":
        st["plan"].matched_project(st["x"], st["lines"])
        st["plan"].matched_backproject(st["g"], st["native"])
        return {"out": st["lines"], "grad": st["native"]}
    op = {"wfbp": A.wfbp, "ray": A.ray_project}[kind]
    x = st["x"].detach().requires_grad_()
    y = op(x, st["plan"])
    y.backward(st["g"])
    return {"out": y.detach(), "grad": x.grad}


def work(case):
    c = {**FIELDS, **case}
    if c["kind"] == "batch":
        w = [work({**j, "name": ""}) for j in _jobs(c)]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    phi, zf = (2 if c["ffs"] & 1 else 1), (2 if c["ffs"] & 2 else 1)
    states = {0: 1, 1: 2, 2: 2, 3: 4}[c["ffs"]]
    vox = _native(c) * c["ny"] * c["nx"]
    views = int(round(c["rotations"] * c["ppr"])) // states
    # Views within a rotation of the volume: the only ones a whole chain reads.
    feed = c["pitch"] * c["rows"] * c["row_mm"]
    part = min(1.0, (c["length"] / feed + 2.0) / c["rotations"])
    if c["kind"] in ("lines", "wfbp", "matched", "ray"):
        part = 1.0
    lines, ncols = views * part * c["rows"] * zf, c["channels"] * phi
    n = 2 ** math.ceil(math.log2(2 * ncols))
    filt = lines * (5.0 * n * math.log2(n) + 12.0 * ncols)
    raw, vv = 4.0 * _rays(c), _voxel_views(c)
    out = 4.0 * math.ceil(c["length"] / c["spacing"] - 1e-9) * c["ny"] * c["nx"]
    if c["kind"] == "lines":
        return {"bytes": raw + 4.0 * lines * ncols, "flops": filt}
    if c["kind"] == "wfbp":      # both directions, each reading and writing scan and volume
        return {"bytes": 2 * (raw + 4.0 * vox), "flops": 2 * filt + 2 * 24.0 * vv}
    if c["kind"] == "matched":
        return {"bytes": 2 * (raw + 4.0 * vox), "flops": 2 * 12.0 * vv}
    if c["kind"] == "ray":
        # Planes a ray crosses inside the slab: the cone leaves it early.
        return {"bytes": 2 * (raw + 4.0 * vox), "flops": 2 * 12.0 * 0.7 * _units(c)}
    return {"bytes": part * raw + out, "flops": filt + 24.0 * vv}


# --------------------------------------------------------------------------
# The same results in 64 bits, from the definitions, in plain torch.
# --------------------------------------------------------------------------
_F = torch.float64


class _Geo:
    """Geometry of a case without flying focal spot, in 64 bits."""

    def __init__(self, c):
        s, self.c = _scan(c), c
        self.s = s
        self.dgamma = s.channel_spacing / s.dsd
        self.ds = self.dgamma * s.r
        self.csw = s.r * s.row_spacing / s.dsd
        self.dth = 2.0 * math.pi / s.views_per_rotation
        self.dz = s.feed / s.views_per_rotation
        self.H = s.views_per_rotation // 2
        self.hr = 0.5 * (s.n_rows - 1)
        self.tanc = self.hr * self.csw / s.r
        self.scale = self.dth
        n = self.n_native = max(1, math.ceil(c["length"] / self.csw - 1e-9))
        self.z = -0.5 * c["length"] + self.csw * torch.arange(n, dtype=_F, device="cuda")
        # A clockwise scan is the mirror image of the counter-clockwise one.
        self.mirror = -1.0 if c["clockwise"] else 1.0
        self.angle0 = self.mirror * s.angle0
        ax = [(torch.arange(m, dtype=_F, device="cuda") - 0.5 * (m - 1)) * (c["fov"] / m)
              for m in (c["ny"], c["nx"])]
        yy, xx = torch.meshgrid(self.mirror * ax[0], ax[1], indexing="ij")
        acq = 2.0 * s.r * math.sin(0.5 * (s.n_channels - 1) * self.dgamma)
        self.fov = ((xx ** 2 + yy ** 2) <= 0.25 * acq * acq).reshape(-1).nonzero()[:, 0]
        self.x, self.y = xx.reshape(-1)[self.fov], yy.reshape(-1)[self.fov]

    # Fan -> parallel: (view offset, view fraction, channels, fraction, valid).
    def rebin_table(self):
        s = self.s
        c = torch.arange(s.n_channels, dtype=_F, device="cuda")
        sb = (c - s.central_channel) * self.dgamma
        beta = torch.asin(sb.clamp(-1, 1))
        b = beta / self.dgamma + s.central_channel
        ok = (sb.abs() <= 1) & (b >= 0) & (b < s.n_channels)
        b0 = b.floor().clamp(0, s.n_channels - 1)
        nd = -beta / self.dth
        return (nd.floor().long(), nd - nd.floor(), b0.long(),
                (b0 + 1).clamp(max=s.n_channels - 1).long(), (b - b0) * ok, ok.to(_F))

    def rebin_taps(self, j):
        """For parallel views j: [len(j), channels] raw views, channels, weights."""
        aoff, fa, b0, b1, fb, ok = self.rebin_table()
        last = self.s.n_views - 1
        va = (j[:, None] + aoff).clamp(0, last)
        vb = (j[:, None] + aoff + 1).clamp(0, last)
        e = torch.ones_like(va)
        return [(va, e * b0, (1 - fa) * (1 - fb) * ok), (vb, e * b0, fa * (1 - fb) * ok),
                (va, e * b1, (1 - fa) * fb * ok), (vb, e * b1, fa * fb * ok)]

    def rebin(self, raw):
        s, out = self.s, torch.zeros((self.s.n_views, self.s.n_rows, self.s.n_channels),
                                     dtype=_F, device="cuda")
        for v0 in range(0, s.n_views, 64):
            j = torch.arange(v0, min(v0 + 64, s.n_views), device="cuda")
            for v, b, w in self.rebin_taps(j):
                out[j] += (raw[v, :, b].to(_F) * w[..., None]).permute(0, 2, 1)
        return out

    def rebin_t(self, lines):
        s = self.s
        out = torch.zeros((s.n_views * s.n_channels, s.n_rows), dtype=_F, device="cuda")
        for v0 in range(0, s.n_views, 64):
            j = torch.arange(v0, min(v0 + 64, s.n_views), device="cuda")
            val = lines[j].permute(0, 2, 1)
            for v, b, w in self.rebin_taps(j):
                out.index_add_(0, (v * s.n_channels + b).reshape(-1),
                               (val * w[..., None]).reshape(-1, s.n_rows))
        return out.view(s.n_views, s.n_channels, s.n_rows).permute(0, 2, 1).contiguous()

    def filter(self, lines):
        n = self.s.n_channels
        kind, cut, a = S.FILTERS[self.c["filter"]]
        i = np.arange(-(n - 1), n, dtype=np.float64)
        if kind == 1:
            h = 2.0 / (math.pi ** 2 * self.ds * (1.0 - 4.0 * i * i))
        else:
            def r(t):
                z = t == 0.0
                u = np.where(z, 1.0, t)
                return np.where(z, 0.5, np.sin(u) / u + (np.cos(u) - 1.0) / (u * u))
            h = cut * cut / (2.0 * self.ds) * (
                a * r(cut * math.pi * i) + 0.5 * (1 - a) * (r(math.pi * cut * i + math.pi) +
                                                           r(math.pi * cut * i - math.pi)))
        m = 4 * n
        k = torch.zeros(m, dtype=_F, device="cuda")
        k[torch.as_tensor(i.astype(np.int64) % m, device="cuda")] = \
            torch.as_tensor(h, device="cuda")
        fk = torch.fft.rfft(k)
        out = torch.empty_like(lines)
        for v0 in range(0, lines.shape[0], 256):
            x = torch.fft.rfft(lines[v0:v0 + 256], n=m) * fk
            out[v0:v0 + 256] = torch.fft.irfft(x, n=m)[..., :n]
        return out

    def theta(self, t, plain):
        """The views t + k H that see some voxel column: (view, slices lo..hi,
        selected, weight, row, row fraction, channel, channel fraction);
        plain: the R / l weight of every view instead of the window and W."""
        s = self.s
        co, si = math.cos(self.angle0 + t * self.dth), math.sin(self.angle0 + t * self.dth)
        p, f = self.x * si - self.y * co, self.x * co + self.y * si
        sq = torch.sqrt(s.r ** 2 - p * p)
        kb = s.feed / (2 * math.pi) * torch.asin(p / s.r)
        zl = self.z.tolist()
        reach = (s.r + 300.0) * self.tanc + abs(s.feed)
        for k in range((s.n_views - t + self.H - 1) // self.H):
            v, sg = t + k * self.H, -1.0 if k & 1 else 1.0
            zt = s.z0 + self.dz * v
            half = reach if plain else abs(s.feed)
            inside = [i for i, z in enumerate(zl) if abs(z - zt) <= half]
            if not inside:
                continue
            lo, hi = inside[0], inside[-1] + 1
            l = sq - sg * f
            pi = sg * p / self.ds + s.central_channel
            q = (self.z[lo:hi, None] - zt + sg * kb) / (l * self.tanc)
            qi = q * self.hr + s.central_row
            ip, iq = pi.floor(), qi.floor()
            sel = ((q.abs() <= 1) & (iq >= 0) & (iq <= s.n_rows - 2) &
                   (ip >= 0) & (ip <= s.n_channels - 2))
            if plain:
                w = sel * (s.r / l)
            else:
                u = ((1 - q.abs()) / 0.4).clamp(0, 1)
                w = sel * torch.sin(0.5 * math.pi * u) ** 2
            yield (v, lo, hi, w, iq.clamp(0, s.n_rows - 2).long(), qi - iq,
                   ip.clamp(0, s.n_channels - 2).long(), pi - ip)

    @staticmethod
    def taps(iq, wq, ip, wp, n):
        o = iq * n + ip
        return [(o, (1 - wq) * (1 - wp)), (o + 1, (1 - wq) * wp), (o + n, wq * (1 - wp)),
                (o + n + 1, wq * wp)]

    def backproject(self, lines, plain=False):
        n = self.s.n_channels
        acc = torch.zeros((self.n_native, len(self.x)), dtype=_F, device="cuda")
        for t in range(self.H):
            num, den = torch.zeros_like(acc), torch.zeros_like(acc)
            for v, lo, hi, w, iq, wq, ip, wp in self.theta(t, plain):
                row = lines[v].reshape(-1)
                val = sum(row[o] * tw for o, tw in self.taps(iq, wq, ip, wp, n))
                num[lo:hi] += w * val
                den[lo:hi] += w
            acc += num if plain else torch.where(den > 0, num / den.clamp(min=1e-300), 0.0)
        out = torch.zeros((self.n_native, self.c["ny"] * self.c["nx"]), dtype=_F, device="cuda")
        out[:, self.fov] = acc * self.scale
        return out.view(self.n_native, self.c["ny"], self.c["nx"])

    def backproject_t(self, vol, plain=False):
        s = self.s
        n = s.n_channels
        x = vol.to(_F).reshape(self.n_native, -1)[:, self.fov] * self.scale
        lines = torch.zeros((s.n_views, s.n_rows * n), dtype=_F, device="cuda")
        for t in range(self.H):
            seen = list(self.theta(t, plain))
            c = x
            if not plain:
                den = torch.zeros_like(x)
                for v, lo, hi, w, *_ in seen:
                    den[lo:hi] += w
                c = torch.where(den > 0, x / den.clamp(min=1e-300), 0.0)
            for v, lo, hi, w, iq, wq, ip, wp in seen:
                cw = w * c[lo:hi]
                for o, tw in self.taps(iq, wq, ip, wp, n):
                    lines[v].index_add_(0, o.reshape(-1), (cw * tw).reshape(-1))
        return lines.view(s.n_views, s.n_rows, n)

    def thicken(self, native):
        c = self.c
        m = max(1, math.ceil(c["length"] / c["spacing"] - 1e-9))
        zr = -0.5 * c["length"] + c["spacing"] * torch.arange(m, dtype=_F, device="cuda")
        w = (1 - (self.z[None] - zr[:, None]).abs() / c["thickness"]).clamp(min=0)
        out = torch.tensordot(w / w.sum(1, keepdim=True), native, dims=1)
        return 1000.0 * out / S.MU_WATER - 1000.0 if c["hu"] else out

    def adaptive(self, raw):
        a = self.c["adaptive"]
        x = raw.to(_F)
        m = x.abs().amax((1, 2), keepdim=True)
        lam = ((x - (1 - a) * m) / (a * m)).clamp(0, 1)
        mean = torch.nn.functional.avg_pool2d(x[:, None], 3, 1, 1, count_include_pad=False)[:, 0]
        return x + lam * (mean - x)

    def reconstruct(self, raw):
        if self.c["adaptive"] > 0:
            raw = self.adaptive(raw)
        return self.thicken(self.backproject(self.filter(self.rebin(raw))))

    def ray(self, vol, back=None):
        """Joseph's method: line integrals of vol along the raw rays, or with
        `back` (a scan) the transpose."""
        s, c, nz = self.s, self.c, self.n_native
        ny, nx = c["ny"], c["nx"]
        dx, dy = c["fov"] / nx, self.mirror * c["fov"] / ny
        x0, y0 = -0.5 * (nx - 1) * dx, -0.5 * (ny - 1) * dy
        beta = (torch.arange(s.n_channels, dtype=_F, device="cuda") - s.central_channel) * \
            self.dgamma
        w = (torch.arange(s.n_rows, dtype=_F, device="cuda") - s.central_row) * s.row_spacing
        flat = vol.to(_F).reshape(-1) if back is None else None
        out = torch.zeros((s.n_views, s.n_rows, s.n_channels) if back is None else
                          nz * ny * nx, dtype=_F, device="cuda")
        for v in range(s.n_views):
            a = self.angle0 + v * self.dth
            sx, sy, sz = s.r * math.cos(a), s.r * math.sin(a), s.z0 + v * self.dz
            ux, uy = -s.dsd * torch.cos(a + beta), -s.dsd * torch.sin(a + beta)
            xm = ux.abs() >= uy.abs()
            for major in (True, False):
                ch = (xm if major else ~xm).nonzero()[:, 0]
                if not len(ch):
                    continue
                p0, dp, q0, dq = (x0, dx, y0, dy) if major else (y0, dy, x0, dx)
                sp, sq = (sx, sy) if major else (sy, sx)
                up, uq = (ux[ch], uy[ch]) if major else (uy[ch], ux[ch])
                npl, nq = (nx, ny) if major else (ny, nx)
                i = torch.arange(npl, dtype=_F, device="cuda")[:, None]
                t = (p0 + i * dp - sp) / up                      # [plane, channel]
                fq = (sq + t * uq - q0) / dq
                jq = fq.floor()
                fz = (sz + t[None] * w[:, None, None] + 0.5 * c["length"]) / self.csw
                kz = fz.floor()                                  # [row, plane, channel]
                length = (dp / up).abs() * torch.sqrt(up ** 2 + uq ** 2 + w[:, None] ** 2)
                val = 0.0 if back is None else (back[v][:, ch].to(_F) * length)[:, None, :]
                for dk in (0, 1):
                    for dj in (0, 1):
                        j, k = (jq + dj).long(), (kz + dk).long()
                        wj = (fq - jq) if dj else 1 - (fq - jq)
                        wk = (fz - kz) if dk else 1 - (fz - kz)
                        m = (j >= 0) & (j < nq) & (k >= 0) & (k < nz)
                        ii = i.long()
                        o = k * (ny * nx) + (j * nx + ii if major else ii * nx + j)
                        o = torch.where(m, o, 0)
                        wt = wj * wk * m
                        if back is None:
                            val = val + (flat[o] * wt).sum(1)
                        else:
                            out.index_add_(0, o.reshape(-1), (wt * val).reshape(-1))
                if back is None:
                    out[v][:, ch] = val * length
        return out if back is None else out.view(nz, ny, nx)


def exact(case, seed):
    c = {**FIELDS, **case}
    if c["kind"] == "batch":
        if _voxel_views(c) > 8e9 or any(j["ffs"] for j in _jobs(c)):
            return None
        raws = prepare(case, seed)["raw"]
        return [_Geo(j).reconstruct(r) for j, r in zip(_jobs(c), raws)]
    if c["ffs"]:
        return None
    if c["kind"] in ("recon", "host") and _voxel_views(c) > 1.2e10:
        return None
    if c["kind"] == "lines" and _rays(c) > 2e8:
        return None
    st, g = prepare(case, seed), _Geo(c)
    if c["kind"] in ("recon", "host"):
        return g.reconstruct(st["raw"].cuda())
    if c["kind"] == "lines":
        y = g.filter(g.rebin(st["raw"]))
        return torch.nn.functional.pad(y, (0, st["plan"].info.channel_pitch - y.shape[-1]))
    x, cot = st["x"], st["g"]
    if c["kind"] == "wfbp":
        return {"out": g.backproject(g.filter(g.rebin(x))),
                "grad": g.rebin_t(g.filter(g.backproject_t(cot)))}
    if c["kind"] == "matched":
        n = c["channels"]
        return {"out": torch.nn.functional.pad(g.backproject_t(x, plain=True),
                                               (0, cot.shape[-1] - n)),
                "grad": g.backproject(cot[..., :n].to(_F).contiguous(), plain=True)}
    return {"out": g.ray(x), "grad": g.ray(None, back=cot)}
