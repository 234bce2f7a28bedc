// adjoint.hip -- exact transpose of the FP32 WFBP chain (a matched helical
// forward projector): native volume -> filtered parallel rows -> raw fan data.
//
// The forward chain (rebin, filter, W-weighted backprojection,
// cuda_kernels.cuh:11-93, 198-287) is linear in the raw data for a fixed
// geometry: W(q) and its per-theta~ sum depend on geometry only.  Transposes:
//   backprojection^T: per voxel and theta~, the weight sum over the selected
//     views is formed first, then every selected sample adds
//     scale * xbar * W / sum W times its four bilinear weights -- gathered per
//     detector sample, or (where the gather has no scratch: a graph capture
//     before its first use) scattered by FP32 hardware atomics;
//   filter^T: the filter (symmetric Toeplitz), run by rebin_filter.hip's
//     filter-only mode;
//   rebin^T: every fan sample collects from the parallel samples that read it.
// Selection and the FP32 weights are computed by the same code as the forward
// kernels, so the transpose is exact up to FP32 summation order.
#include <algorithm>
#include <cmath>

#include "wave_ops.h"
#include "wfbp_internal.h"

namespace fct {
namespace {

// MATCHED: the transpose of backproject_v1.hip's matched mode instead --
// every view that sees the voxel, weight scale * R / l, no W normalisation
// and no view window: a voxel-driven helical projector of the native volume
// onto the parallel rows (with the rebinning transpose, onto the fan data).
template <int TZ, bool CENTERED, bool MATCHED>
__global__ __launch_bounds__(64) void bp_adjoint_kernel(BpAdjArgs a) {
  const BpArgs& b = a.bp;
  const int lane = threadIdx.x;
  const int tiles = b.tiles_x * b.tiles_y;
  const int slab = blockIdx.x / tiles;
  const int tile = blockIdx.x - slab * tiles;
  const int tx = tile % b.tiles_x, ty = tile / b.tiles_x;
  const int ix = tx * 8 + (lane & 7), iy = ty * 8 + (lane >> 3);
  const bool inb = ix < b.nx && iy < b.ny;
  const float x = inb ? b.xs[ix] : 0.0f;
  const float y = inb ? b.ys[iy] : 0.0f;
  const FctBpConsts& g = b.g;
  const bool active = inb && fct_in_fov(x, y, g);
  if (!__any(active)) return;
  const int s0 = slab * TZ;
  const int nz = min(TZ, b.n_native - s0);
  const int chunk = s0 / fct_tables::kSliceChunk;
  float zs[TZ], xb[TZ];
#pragma unroll
  for (int i = 0; i < TZ; ++i) {
    zs[i] = i < nz ? b.zs[s0 + i] : 0.0f;
    xb[i] = (i < nz && active) ? a.xbar[((size_t)(s0 + i) * b.ny + iy) * b.nx + ix] * b.scale
                               : 0.0f;
  }
  const float* ztc = b.zt + (size_t)chunk * b.nviews;
  const int2 vr = b.slab_vrange[slab];
  const int H = b.H;
  const size_t vstride = (size_t)g.nrows * b.cpitch;

  for (int t = 0; t < H; ++t) {
    const int kmin = vr.x <= t ? 0 : (vr.x - t + H - 1) / H;
    const int kmax = vr.y <= t ? 0 : (vr.y - t + H - 1) / H;
    if (kmin >= kmax) continue;
    const float2 cs = b.cs[t];
    const float p = fmaf(x, cs.y, -(y * cs.x));
    const float sq = sqrtf(fmaf(-p, p, g.R2));
    const float f = fmaf(x, cs.x, y * cs.y);
    const float kb = g.kappa * fct_asinf(p * g.invR);
    const float pidx_e = fmaf(p, g.inv_ds, g.cc), pidx_o = fmaf(-p, g.inv_ds, g.cc);
    const float invL_e = g.hr / ((sq - f) * g.tanc), invL_o = g.hr / ((sq + f) * g.tanc);
    const float fR_e = g.tanc / ((sq - f) * g.tanc * g.invR);   // R / l (matched mode)
    const float fR_o = g.tanc / ((sq + f) * g.tanc * g.invR);
    float den[TZ];
#pragma unroll
    for (int i = 0; i < TZ; ++i) den[i] = 0.0f;
    // Pass 0: weight sums; pass 1: scatter.
    for (int pass = MATCHED ? 1 : 0; pass < 2; ++pass) {
      float rden[TZ];
      if (pass == 1) {
#pragma unroll
        for (int i = 0; i < TZ; ++i) rden[i] = den[i] > 0.0f ? xb[i] / den[i] : 0.0f;
      }
      for (int k = kmin; k < kmax; ++k) {
        const int v = t + k * H;
        const bool odd = k & 1;
        const float pidx = odd ? pidx_o : pidx_e;
        const float invL = odd ? invL_o : invL_e;
        const float ztv = ztc[v];
        const float row0 = fmaf((odd ? -kb : kb) - ztv, invL, g.cr);   // fct_bp_row0
        const float pfl = floorf(pidx);
        const bool chan_ok = active && pfl >= 0.0f && pfl <= (float)(g.ncols - 2);
        const int pf = chan_ok ? (int)pfl : 0;
        const float wp = pidx - pfl;
        float* vb = a.gbar + (size_t)v * vstride + pf;
#pragma unroll
        for (int i = 0; i < TZ; ++i) {
          if (i >= nz || (!MATCHED && !fct_bp_in_window(ztv, zs[i], g))) continue;
          const float qi = fmaf(zs[i], invL, row0);   // fct_bp_row
          const float qfl = floorf(qi);
          bool sel;
          if (CENTERED)
            sel = chan_ok && (uint32_t)(int)qfl <= (uint32_t)(g.nrows - 2);
          else
            sel = chan_ok && !(fabsf(qi - g.cr) > g.hr) && qfl >= 0.0f &&
                  qfl <= (float)(g.nrows - 2);
          if (!sel) continue;
          if (MATCHED) {
            const float c = xb[i] * (odd ? fR_o : fR_e);
            const float wq = qi - qfl;
            float* r0 = vb + (size_t)(int)qfl * b.cpitch;
            float* r1 = r0 + b.cpitch;
            unsafeAtomicAdd(r0, c * (1.0f - wq) * (1.0f - wp));
            unsafeAtomicAdd(r0 + 1, c * (1.0f - wq) * wp);
            unsafeAtomicAdd(r1, c * wq * (1.0f - wp));
            unsafeAtomicAdd(r1 + 1, c * wq * wp);
            continue;
          }
          const float W = fct_w_of_row(qi, g);
          if (pass == 0) {
            den[i] += W;
            continue;
          }
          const float c = W * rden[i];
          if (c == 0.0f) continue;
          const float wq = qi - qfl;
          float* r0 = vb + (size_t)(int)qfl * b.cpitch;
          float* r1 = r0 + b.cpitch;
          unsafeAtomicAdd(r0, c * (1.0f - wq) * (1.0f - wp));
          unsafeAtomicAdd(r0 + 1, c * (1.0f - wq) * wp);
          unsafeAtomicAdd(r1, c * wq * (1.0f - wp));
          unsafeAtomicAdd(r1 + 1, c * wq * wp);
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Gathered form: every detector sample collects from the voxels that read it.
// ---------------------------------------------------------------------------
// Volume order of a theta~: planes of the axis its parallel rays run along
// (the primary axis: x where |cos| >= |sin|, else y), slices, then the other
// in-plane axis, so that the 64 neighbouring channels of a wave read
// neighbouring addresses.

// What the other kernels need of every voxel column for the theta~ [t0, t0 +
// nt): (rows per mm of z for the even and the odd views, kappa asin(p / R),
// p), the forward kernels' FP32 values; p = 1e30 outside the FOV, which no
// channel matches.
__global__ __launch_bounds__(256) void bp_adjoint_column_kernel(BpAdjArgs a, AdjGather q) {
  const BpArgs& b = a.bp;
  const FctBpConsts& g = b.g;
  const int ns = q.swap ? b.ny : b.nx;
  const int i = blockIdx.x * 256 + threadIdx.x, n = b.nx * b.ny;
  if (i >= n) return;
  const int prim = i / ns, sec = i - prim * ns;
  const float x = b.xs[q.swap ? prim : sec], y = b.ys[q.swap ? sec : prim];
  const bool active = fct_in_fov(x, y, g);
  for (int ti = blockIdx.y; ti < q.nt; ti += gridDim.y) {
    const float* csp = reinterpret_cast<const float*>(b.cs + q.t0 + ti);
    const float c = ld_uniform(csp), sn = ld_uniform(csp + 1);
    const float p = fmaf(x, sn, -(y * c));
    const float sq = sqrt_rn_large(fmaf(-p, p, g.R2));
    const float f = fmaf(x, c, y * sn);
    const float4 e = make_float4(div_rn_normal(g.hr, (sq - f) * g.tanc),
                                 div_rn_normal(g.hr, (sq + f) * g.tanc),
                                 g.kappa * fct_asinf(p * g.invR), p);
    q.col[(size_t)ti * n + i] = active ? e : make_float4(0.0f, 0.0f, 0.0f, 1e30f);
  }
}

// xbar * scale / sum W of every voxel for the theta~ [t0, t0 + nt) (0 where no
// view selects the voxel), in that order: one wave per 64 voxels along the
// secondary axis and eight slices.  9.3 GB of writes for 384 x 384 x 32 voxels x
// 492 theta~ at 2.2 TB/s, VALU issue 66 % of its cycles: 4.5 -> 4.3 ms with the
// mask-free weight.  The division is correctly rounded, as in the scattering
// kernel; v_rcp_f32 in its place saves 0.5 ms and is a bit less precise.
constexpr int kAdjSlices = 8;
template <bool CENTERED>
__global__ __launch_bounds__(64) void bp_adjoint_weights_kernel(BpAdjArgs a, AdjGather q) {
  const BpArgs& b = a.bp;
  const FctBpConsts& g = b.g;
  const int ns = q.swap ? b.ny : b.nx, np = q.swap ? b.nx : b.ny;
  const int groups = (ns + 63) >> 6, nsl = (b.n_native + kAdjSlices - 1) / kAdjSlices;
  const int id = xcd_block(blockIdx.x, gridDim.x);
  const int slab = id / (groups * np), rest = id - slab * groups * np;
  const int prim = rest / groups, sec = (rest - prim * groups) * 64 + threadIdx.x;
  const int ix = q.swap ? prim : sec, iy = q.swap ? sec : prim;
  const bool inb = sec < ns;
  const bool active = inb && fct_in_fov(b.xs[min(ix, b.nx - 1)], b.ys[min(iy, b.ny - 1)], g);
  const int s0 = slab * kAdjSlices, nz = min(kAdjSlices, b.n_native - s0);
  const int chunk = s0 / fct_tables::kSliceChunk;
  float zs[kAdjSlices], xb[kAdjSlices];
#pragma unroll
  for (int i = 0; i < kAdjSlices; ++i) {
    zs[i] = b.zs[s0 + min(i, nz - 1)];
    xb[i] = (i < nz && active) ? a.xbar[((size_t)(s0 + i) * b.ny + iy) * b.nx + ix] * b.scale
                               : 0.0f;
  }
  const bool some = __any(active);
  const float* ztc = b.zt + (size_t)chunk * b.nviews;
  const int* wrc = reinterpret_cast<const int*>(b.wrange + (size_t)chunk * b.nviews);
  const size_t plane = (size_t)b.nx * b.ny;
  const int ti0 = (int)((long long)q.nt * blockIdx.y / gridDim.y);
  const int ti1 = (int)((long long)q.nt * (blockIdx.y + 1) / gridDim.y);
  float* out = q.wgt + ti0 * plane * b.n_native + ((size_t)prim * b.n_native + s0) * ns + sec;
  for (int ti = ti0; ti < ti1; ++ti, out += plane * b.n_native) {
    const int t = q.t0 + ti;
    float den[kAdjSlices];
#pragma unroll
    for (int i = 0; i < kAdjSlices; ++i) den[i] = 0.0f;
    if (some) {
      const float4 col = q.col[(size_t)ti * plane + (size_t)prim * ns + min(sec, ns - 1)];
      const float p = col.w, kb = col.z;
#pragma unroll
      for (int par = 0; par < 2; ++par) {
        const float pidx = par ? fmaf(-p, g.inv_ds, g.cc) : fmaf(p, g.inv_ds, g.cc);
        const float pfl = floorf(pidx);
        const bool ok = active && pfl >= 0.0f && pfl <= (float)(g.ncols - 2);
        const float invL = ok ? (par ? col.y : col.x) : 0.0f;
        for (int v = t + par * b.H; v < b.nviews; v += 2 * b.H) {
          const int wx = ld_uniform(wrc + 2 * v), wy = ld_uniform(wrc + 2 * v + 1);
          if (wx > s0 + nz - 1 || wy < s0) continue;
          const float row0 = ok ? fmaf((par ? -kb : kb) - ld_uniform(ztc + v), invL, g.cr) : -1e30f;
          const float qa = fmaf(zs[0], invL, row0), qb = fmaf(zs[kAdjSlices - 1], invL, row0);
          if (!__any(fmaxf(qa, qb) >= 0.0f && fminf(qa, qb) < (float)(g.nrows - 1))) continue;
#pragma unroll
          for (int i = 0; i < kAdjSlices; ++i) {
            if (s0 + i < wx || s0 + i > wy) continue;
            const float qi = fmaf(zs[i], invL, row0);
            if (CENTERED) {
              // W = 0 exactly on every row outside the detector and in the
              // lanes at row -1e30 (t clamped to [0, 1]): no mask.
              den[i] += fct_w_of_t(
                  __builtin_amdgcn_fmed3f(fmaf(-fabsf(qi - g.cr), g.wk, FCT_WC), 0.0f, 1.0f));
              continue;
            }
            const int iq = floor_int(qi);
            const bool sel = ok && (uint32_t)iq <= (uint32_t)(g.nrows - 2) &&
                             !(fabsf(qi - g.cr) > g.hr);
            const float W = fct_w_of_row(qi, g);
            den[i] += sel ? W : 0.0f;
          }
        }
      }
    }
    if (inb)
#pragma unroll
      for (int i = 0; i < kAdjSlices; ++i)
        if (i < nz) out[(size_t)i * ns] = den[i] > 0.0f ? xb[i] / den[i] : 0.0f;
  }
}

// The matched pair's volume in the swapped order [x][slice][y].
__global__ __launch_bounds__(256) void swap_volume_kernel(const float* __restrict__ in,
                                                          float* __restrict__ out, int nx, int ny,
                                                          int nz) {
  __shared__ float tile[32][33];
  const int bx = blockIdx.x * 32, by = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int z = blockIdx.z; z < nz; z += gridDim.z) {
    for (int r = ty; r < 32; r += 8)
      if (bx + tx < nx && by + r < ny) tile[r][tx] = in[((size_t)z * ny + by + r) * nx + bx + tx];
    __syncthreads();
    for (int r = ty; r < 32; r += 8)
      if (bx + r < nx && by + tx < ny) out[((size_t)(bx + r) * nz + z) * ny + by + tx] = tile[tx][r];
    __syncthreads();
  }
}

// One wave per (view, 64 channels, RC detector rows), a lane per channel with
// its rows in LDS.  Plane by plane along the primary axis, the voxel columns
// whose channel position lies within one channel of the lane's (a fixed
// small number of candidates around the ray, tested with the forward
// kernels' FP32 position) add their slices into the lane's rows (one LDS read
// and write of two rows per slice, conflict-free).  23 VALU instructions per slice
// of a candidate, 14 in the matched projector; counters (2952 views x 16 x 736,
// 384 x 384 x 32 voxels): VALU issue 92 % of the kernel's cycles with 39 of 64 lanes
// active (half to three quarters of the lanes hold a column), address unit 47 %;
// matched (2304 views, 256 x 256 x 32) 76 % with 49 lanes, 56 %.  287 ms with four
// global atomics per sample -> 4.3 (weights) + 11.1 ms.  Planes on which no lane
// has a voxel in its rows are left out (9840 views x 64 x 888, 32 x 32 x 4 of 40 mm:
// 5.2 -> 2.4 ms, where the atomics take 2.6; 2304 views x 16 x 736, 512 x 1 x 16: 2.7
// -> 1.0 ms, atomics 1.8).  RC rows per wave: 16 or 32, so that the rows in LDS
// leave at least 16 waves per CU.
template <int RC, bool CENTERED, bool MATCHED>
__global__ __launch_bounds__(64) void bp_adjoint_gather_kernel(BpAdjArgs a, AdjGather q) {
  // Detector rows rlo .. rlo + rspan + 1 (below): this wave's and the
  // neighbouring waves' rows next to them, which are dropped.
  __shared__ float acc[(RC + 2) * 64];
  const BpArgs& b = a.bp;
  const FctBpConsts& g = b.g;
  const int lane = threadIdx.x, H = b.H;
  const int cg = b.cpitch >> 6, nrc = (g.nrows + RC - 1) / RC;
  const int kv = (b.nviews + H - 1) / H;
  int id = xcd_block(blockIdx.x, gridDim.x);
  const int ch = (id % cg) * 64 + lane;
  id /= cg;
  const int split = id % q.nsplit;
  id /= q.nsplit;
  const int R0 = (id % nrc) * RC;
  id /= nrc;
  const int kk = id % kv, ti = id / kv;
  const int t = q.t0 + ti, v = t + kk * H;
  if (v >= b.nviews) return;
  const bool odd = kk & 1;
  const float* csp = reinterpret_cast<const float*>(b.cs + t);
  const int ns = q.swap ? b.ny : b.nx, np = q.swap ? b.nx : b.ny;
  const int i0 = (int)((long long)np * split / q.nsplit);
  const int i1 = (int)((long long)np * (split + 1) / q.nsplit);
#pragma unroll
  for (int r = 0; r < RC + 2; ++r) acc[r * 64 + lane] = 0.0f;
  // Footprints of rows [rlo, rlo + rspan] reach this wave's rows.
  const int rlo = max(0, R0 - 1), rspan = min(g.nrows - 2, R0 + RC - 1) - rlo;
  float* lrow = acc + lane;   // row rlo

  // Along the channel's ray, linear in the plane index i: the secondary
  // position J0 + i J1 (columns within hw of it are within one channel) and
  // the distance from the focal spot to the column, L0 + i L1.
  float J0, J1, hw, L0, L1, kb0, zmargin;
  {
    const double ds = 1.0 / (double)g.inv_ds, c = ld_uniform(csp), s = ld_uniform(csp + 1);
    const double pe = ((double)min(ch, g.ncols - 1) - (double)g.cc) * ds, p = odd ? -pe : pe;
    const double x0 = q.gx0, y0 = q.gy0, dx = q.gdx, dy = q.gdy;
    const double sqr = sqrt(fmax((double)g.R2 - p * p, 1.0));
    double f0, f1;
    if (q.swap) {   // x planes: y = (x s - p) / c
      J0 = (float)(((x0 * s - p) / c - y0) / dy);
      J1 = (float)(dx * s / c / dy);
      hw = (float)fabs(ds / (c * dy));
      f0 = x0 * c + (x0 * s - p) / c * s;
      f1 = dx * c + dx * s / c * s;
    } else {        // y planes: x = (p + y c) / s
      J0 = (float)(((p + y0 * c) / s - x0) / dx);
      J1 = (float)(dy * c / s / dx);
      hw = (float)fabs(ds / (s * dx));
      f0 = (p + y0 * c) / s * c + y0 * s;
      f1 = dy * c / s * c + dy * s;
    }
    hw = fmaf(hw, 1.001f, 0.01f);   // rounding of the positions
    L0 = (float)(odd ? sqr + f0 : sqr - f0);
    L1 = (float)(odd ? f1 : -f1);
    const float kb = g.kappa * fct_asinf((float)p * g.invR);
    kb0 = odd ? -kb : kb;
    // A candidate's column lies within one channel of the ray, and within
    // hw of it along the secondary axis (sqrt 2 channels at most).
    zmargin = (float)(1.5 * ds / sqr) * fabsf(g.kappa) + 4.0f * (float)ds * g.tanc *
              (1.0f + 2.0f / g.hr);
  }
  const int nj = __builtin_amdgcn_readfirstlane((int)(2.0f * hw) + 1);
  const float inv_dz = (float)(1.0 / q.dz);
  const float ra = ((float)rlo - g.cr) / g.hr * g.tanc;
  const float rb = ((float)(rlo + rspan + 1) - g.cr) / g.hr * g.tanc;
  const int nchunks = (b.n_native + fct_tables::kSliceChunk - 1) / fct_tables::kSliceChunk;
  const float* vol = MATCHED ? (q.swap ? q.wgt : a.xbar)
                             : q.wgt + (size_t)ti * b.nx * b.ny * b.n_native;
  const float4* cols = q.col + (size_t)ti * b.nx * b.ny;
  // (The matched projector reads the volume itself for y planes.)
  const size_t pstride = MATCHED && !q.swap ? (size_t)b.nx : (size_t)b.n_native * ns;
  const size_t sstride = MATCHED && !q.swap ? (size_t)b.nx * b.ny : (size_t)ns;

  bool touched = false;   // (wave-uniform)
  for (int chunk = 0; rspan >= 0 && chunk < nchunks; ++chunk) {
    const int a0 = chunk * fct_tables::kSliceChunk;
    const int na = min(fct_tables::kSliceChunk, b.n_native - a0);
    int k0 = 0, k1 = na - 1;   // slices a0 + [k0, k1] of this chunk the view may select
    if (MATCHED) {
      // Every slab whose view range holds the view (as the backprojection).
      int first = na, last = -1;
      for (int s = 0; s < na; s += q.tile_z) {
        const int* vr = reinterpret_cast<const int*>(b.slab_vrange + (a0 + s) / q.tile_z);
        if (ld_uniform(vr) <= v && v < ld_uniform(vr + 1)) {
          first = min(first, s);
          last = min(s + q.tile_z, na) - 1;
        }
      }
      k0 = first;
      k1 = last;
    } else {
      const int* wr = reinterpret_cast<const int*>(b.wrange + (size_t)chunk * b.nviews + v);
      k0 = max(k0, ld_uniform(wr) - a0);
      k1 = min(k1, ld_uniform(wr + 1) - a0);
    }
    if (k0 > k1) continue;
    const float zsl = b.zs[a0 + min(lane, na - 1)];   // slice z, one per lane
    const float zfirst = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(zsl), 0));
    const float ztv = ld_uniform(b.zt + (size_t)chunk * b.nviews + v);
    // Slice positions at which the rows rlo and rlo + rspan + 1 cross the ray.
    const float zc = ztv - kb0 - zfirst, sm = fmaf(zmargin, fabsf(inv_dz), 0.05f);
    const float A0 = fmaf(ra, L0, zc) * inv_dz, A1 = ra * L1 * inv_dz;
    const float B0 = fmaf(rb, L0, zc) * inv_dz, B1 = rb * L1 * inv_dz;
    // Planes on which the ray lies in the grid and these slices between the two
    // rows (their crossings keep their order along the ray): for every lane an
    // interval, as all of this is linear in the plane index.  A tenth of a column
    // or slice covers the rounding of the positions, a plane that of the ends.
    float lo = (float)i0, hi = (float)(i1 - 1);
    auto at_least = [&](float a, float b, float c) {   // a + b i >= c
      const float t = (c - a) / b;
      if (b > 0.0f) lo = fmaxf(lo, t);
      if (b < 0.0f) hi = fminf(hi, t);
      if (b == 0.0f && a < c) hi = -1.0f;
    };
    const bool up = inv_dz > 0.0f;
    at_least(J0, J1, -hw - 0.1f);
    at_least(-J0, -J1, (float)(1 - ns) - hw - 0.1f);
    at_least(up ? B0 : A0, up ? B1 : A1, (float)k0 - sm - 0.1f);
    at_least(up ? -A0 : -B0, up ? -A1 : -B1, -(float)k1 - sm - 0.1f);
    const bool meets = ch < g.ncols && lo <= hi;
    const int ia = max(i0, wave_min_i(meets ? (int)floorf(lo) - 1 : INT32_MAX));
    const int ib = min(i1 - 1, wave_max_i(meets ? (int)ceilf(hi) + 1 : -1));
    for (int i = ia; i <= ib; ++i) {
      const float fi = (float)i, sa = fmaf(fi, A1, A0), sb = fmaf(fi, B1, B0);
      const int j0 = (int)ceilf(fmaf(fi, J1, J0) - hw);
      const bool some = ch < g.ncols && j0 < ns && j0 + nj > 0;
      const int sl = max(wave_min_i(some ? (int)ceilf(fminf(sa, sb) - sm) : INT32_MAX), k0);
      const int sh = min(wave_max_i(some ? (int)floorf(fmaxf(sa, sb) + sm) : -1), k1);
      if (sl > sh) continue;
      touched = true;
      const float* vplane = vol + (size_t)i * pstride + (size_t)(a0 + sl) * sstride;
      for (int m = 0; m < nj; ++m) {
        const int j = j0 + m, jc = min(max(j, 0), ns - 1);
        const float4 col = cols[(size_t)i * ns + jc];
        const float pidx = odd ? fmaf(-col.w, g.inv_ds, g.cc) : fmaf(col.w, g.inv_ds, g.cc);
        const float pfl = floorf(pidx);
        const int d = ch - (int)pfl;
        const bool ok = j == jc && pfl >= 0.0f && pfl <= (float)(g.ncols - 2) && (uint32_t)d <= 1u;
        if (!ok) continue;
        const float wp = pidx - pfl;
        float wc = d ? wp : 1.0f - wp;
        const float invL = odd ? col.y : col.x;
        const float row0 = fmaf((odd ? -col.z : col.z) - ztv, invL, g.cr);   // fct_bp_row0
        // R / l = tanc / (lt / R) with lt = hr / invL.
        if (MATCHED) wc *= b.scale * (g.tanc / (g.hr * g.invR)) * invL;
        auto add = [&](int s, float xv) {
          const float z = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(zsl), s));
          const float qi = fmaf(z, invL, row0);   // fct_bp_row
          const uint32_t l = (uint32_t)(floor_int(qi) - rlo);
          bool sel = l <= (uint32_t)rspan;
          if (!CENTERED) sel = sel && !(fabsf(qi - g.cr) > g.hr);
          float val = xv * wc;
          if (!MATCHED)
            val *= fct_w_of_t(
                __builtin_amdgcn_fmed3f(fmaf(-fabsf(qi - g.cr), g.wk, FCT_WC), 0.0f, 1.0f));
          val = sel ? val : 0.0f;
          const float wq = __builtin_amdgcn_fractf(qi);
          float* r = lrow + min(l, (uint32_t)rspan) * 64;
          const float r0 = r[0], r1 = r[64];
          r[0] = fmaf(val, 1.0f - wq, r0);   // (finite weights: val may be infinite)
          r[64] = fmaf(val, wq, r1);
        };
        const float* xp = vplane;
        int s = sl;
        for (; s + 3 <= sh; s += 4, xp += 4 * sstride) {
          float xv[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) xv[u] = xp[u * sstride + (uint32_t)jc];
#pragma unroll
          for (int u = 0; u < 4; ++u) add(s + u, xv[u]);
        }
        for (; s <= sh; ++s, xp += sstride) add(s, xp[(uint32_t)jc]);
      }
    }
  }
  if (q.nsplit > 1 && !touched) return;   // (gbar was cleared)
#pragma unroll
  for (int r = 0; r < RC; ++r)
    if (R0 + r < g.nrows) {
      float* o = a.gbar + ((size_t)v * g.nrows + R0 + r) * b.cpitch + ch;
      const float s = lrow[(R0 + r - rlo) * 64];
      if (q.nsplit > 1)
        unsafeAtomicAdd(o, s);
      else
        *o = s;
    }
}

// Transpose of the rebinning as a gather: a raw sample (view v = m S + rho,
// row, channel b) collects from the parallel samples whose table entry reads
// it.  The entries of (rho, b) are listed per channel (two or three); entry
// (c, aoff, fa, weight of b) reads projection m from the views j with j +
// aoff = m (weight 1 - fa) and j + aoff + 1 = m (weight fa) -- every j below
// (above) that where m is the first (last) projection, to which the forward
// gather clamps.  Every raw sample is written once, no atomics: 2952 views x
// 16 x 736 2.03 ms (four atomics per sample) -> 0.23 ms, bound by the scattered
// reads (a wave of 64 channels spans about 11 views).  Views without a value
// (outside a short volume's reach) are found first, by a pass that ends at a
// view's first value, and waves that span no other write zeros: with one view in
// sixteen 0.25 -> 0.19 ms (the scatter, which skipped zeros, 0.22), 9840 x 64 x 888
// 4.15 -> 2.5 (3.2), all zero 0.25 -> 0.12 (0.09).
__global__ __launch_bounds__(256) void view_flags_kernel(const float* __restrict__ lines, size_t n,
                                                         uint32_t* __restrict__ flags) {
  const float* p = lines + blockIdx.x * n;
  bool some = false;
  for (size_t i = 0; i < n && !some; i += 2048) {
    bool mine = false;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const size_t k = i + u * 256 + threadIdx.x;
      mine = mine || (k < n && p[k] != 0.0f);
    }
    some = __syncthreads_or(mine);
  }
  if (threadIdx.x == 0) flags[blockIdx.x] = some;
}

// A workgroup takes 64 channels of a view, each of its waves every fourth
// detector row, four of them at a time: the entries and flags are read once for
// all rows (a wave per row: 0.34 ms; one, two and four rows at a time 0.27, 0.24
// and 0.23, of 64 rows 4.0, 3.6 and 3.3).
constexpr int kRebinWaves = 4, kRebinRows = 4;
__global__ __launch_bounds__(64 * kRebinWaves) void rebin_adjoint_kernel(RebinAdjArgs a) {
  const int cg = (a.raw_ncols + 63) >> 6;
  const int id = xcd_block(blockIdx.x, gridDim.x);
  const int v = id / cg, lane = threadIdx.x & 63, b = (id - v * cg) * 64 + lane;
  const bool in = b < a.raw_ncols;
  const int m = v / a.states, rho = v - m * a.states;
  const int e0 = in ? a.off[rho * a.raw_ncols + b] : 0;
  const int e1 = in ? a.off[rho * a.raw_ncols + b + 1] : 0;
  const int mmax = (a.raw_nviews - rho + a.states - 1) / a.states - 1;
  const size_t vstride = (size_t)a.nrows * a.cpitch;
  // The wave's views: one with a value among them (the scan's ends read more)?
  int jlo = INT32_MAX, jhi = -1;
  for (int k = e0; k < e1; ++k) {
    const int j = m - a.ent[k].aoff;
    jlo = min(jlo, j - 1);
    jhi = max(jhi, j);
  }
  jlo = max(wave_min_i(jlo), 0);
  jhi = min(wave_max_i(jhi), a.nviews - 1);
  const bool end = m == 0 || m == mmax;
  bool some = end;
  for (int j = jlo; !some && j <= jhi; j += 64)
    some = __any(j + lane <= jhi && a.flags[min(j + lane, jhi)] != 0);
  if (!in) return;
  for (int r0 = threadIdx.x >> 6; r0 < a.raw_nrows; r0 += kRebinWaves * kRebinRows) {
    float sum[kRebinRows] = {};
    for (int k = e0; some && k < e1; ++k) {
      const RebinTDev e = a.ent[k];
      const float* g = a.gbar + (size_t)(e.c >> 16) * a.cpitch + (e.c & 0xffff);
      const int j = m - e.aoff;   // s0: views with j + aoff at m, s1: with j + aoff + 1
      float g0[kRebinRows], g1[kRebinRows];
      size_t o[kRebinRows];
#pragma unroll
      for (int u = 0; u < kRebinRows; ++u) {
        o[u] = (size_t)(min(r0 + u * kRebinWaves, a.raw_nrows - 1) << a.zshift) * a.cpitch;
        g0[u] = j >= 0 && j < a.nviews ? g[o[u] + (size_t)j * vstride] : 0.0f;
        g1[u] = j >= 1 && j <= a.nviews ? g[o[u] + (size_t)(j - 1) * vstride] : 0.0f;
      }
      float beyond[kRebinRows] = {};
      if (end) {   // the views beyond the pair, which the clamp adds to both
        const int lo_end = m == 0 ? min(j - 1, a.nviews) : 0;        // views [0, lo_end)
        const int hi_first = m == mmax ? max(j + 1, 0) : a.nviews;   // views [hi_first, nviews)
        auto add = [&](int j0, int j1) {
#pragma unroll 4
          for (int jj = j0; jj < j1; ++jj)
#pragma unroll
            for (int u = 0; u < kRebinRows; ++u) beyond[u] += g[o[u] + (size_t)jj * vstride];
        };
        add(0, lo_end);
        add(hi_first, a.nviews);
      }
#pragma unroll
      for (int u = 0; u < kRebinRows; ++u) {
        const float s0 = g0[u] + (beyond[u] + (m == 0 ? g1[u] : 0.0f));
        const float s1 = g1[u] + (beyond[u] + (m == mmax ? g0[u] : 0.0f));
        sum[u] = fmaf(e.wb, fmaf(e.fa, s1, (1.0f - e.fa) * s0), sum[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < kRebinRows; ++u)
      if (r0 + u * kRebinWaves < a.raw_nrows)
        a.pbar[((size_t)v * a.raw_nrows + r0 + u * kRebinWaves) * a.raw_ncols + b] = sum[u];
  }
}

__global__ __launch_bounds__(256) void fill_kernel(float* p, size_t n, float v) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
    p[i] = v;
}

template <int TZ>
hipError_t launch_tz(const BpAdjArgs& a, hipStream_t s, bool matched) {
  const int blocks = a.bp.tiles_x * a.bp.tiles_y * a.bp.nslabs;
  const bool c = a.bp.g.cr == a.bp.g.hr;
  if (matched) {
    if (c)
      hipLaunchKernelGGL((bp_adjoint_kernel<TZ, true, true>), dim3(blocks), dim3(64), 0, s, a);
    else
      hipLaunchKernelGGL((bp_adjoint_kernel<TZ, false, true>), dim3(blocks), dim3(64), 0, s, a);
  } else if (c) {
    hipLaunchKernelGGL((bp_adjoint_kernel<TZ, true, false>), dim3(blocks), dim3(64), 0, s, a);
  } else {
    hipLaunchKernelGGL((bp_adjoint_kernel<TZ, false, false>), dim3(blocks), dim3(64), 0, s, a);
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_backproject_adjoint(const BpAdjArgs& a, int tile_z, hipStream_t s,
                                      bool matched) {
  switch (tile_z) {
    case 4: return launch_tz<4>(a, s, matched);
    case 8: return launch_tz<8>(a, s, matched);
    case 16: return launch_tz<16>(a, s, matched);
    case 32: return launch_tz<32>(a, s, matched);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_adjoint_columns(const BpAdjArgs& a, const AdjGather& q, hipStream_t s) {
  hipLaunchKernelGGL(bp_adjoint_column_kernel,
                     dim3((a.bp.nx * a.bp.ny + 255) / 256, std::min(q.nt, 65535)), dim3(256), 0, s,
                     a, q);
  return hipGetLastError();
}

hipError_t launch_adjoint_weights(const BpAdjArgs& a, const AdjGather& q, hipStream_t s) {
  const int ns = q.swap ? a.bp.ny : a.bp.nx, np = q.swap ? a.bp.nx : a.bp.ny;
  // Small volumes: the theta~ shared by several waves, towards 8192 (2304
  // views x 16 x 736, 8 x 8 x 2 voxels, the whole call: 1.06 -> 0.19 ms).
  const int waves = (ns + 63) / 64 * np * ((a.bp.n_native + kAdjSlices - 1) / kAdjSlices);
  const dim3 grid((unsigned)waves, (unsigned)std::max(1, std::min(q.nt, 8192 / waves)));
  if (a.bp.g.cr == a.bp.g.hr)
    hipLaunchKernelGGL(bp_adjoint_weights_kernel<true>, grid, dim3(64), 0, s, a, q);
  else
    hipLaunchKernelGGL(bp_adjoint_weights_kernel<false>, grid, dim3(64), 0, s, a, q);
  return hipGetLastError();
}

hipError_t launch_swap_volume(const float* in, float* out, int nx, int ny, int nz, hipStream_t s) {
  hipLaunchKernelGGL(swap_volume_kernel,
                     dim3((nx + 31) / 32, (ny + 31) / 32, std::min(nz, 65535)), dim3(256), 0, s,
                     in, out, nx, ny, nz);
  return hipGetLastError();
}

int adjoint_gather_waves(const BpArgs& b) {   // waves per theta~
  const int rc = b.g.nrows <= 16 ? 16 : 32;
  return (b.cpitch / 64) * ((b.g.nrows + rc - 1) / rc) * ((b.nviews + b.H - 1) / b.H);
}

template <int RC, bool C>
hipError_t launch_gather_rc(const BpAdjArgs& a, const AdjGather& q, bool matched, hipStream_t s) {
  const dim3 grid((unsigned)(adjoint_gather_waves(a.bp) * q.nt * q.nsplit));
  if (matched)
    hipLaunchKernelGGL((bp_adjoint_gather_kernel<RC, C, true>), grid, dim3(64), 0, s, a, q);
  else
    hipLaunchKernelGGL((bp_adjoint_gather_kernel<RC, C, false>), grid, dim3(64), 0, s, a, q);
  return hipGetLastError();
}

hipError_t launch_adjoint_gather(const BpAdjArgs& a, const AdjGather& q, bool matched,
                                 hipStream_t s) {
  const bool c = a.bp.g.cr == a.bp.g.hr;
  if (a.bp.g.nrows <= 16)
    return c ? launch_gather_rc<16, true>(a, q, matched, s)
             : launch_gather_rc<16, false>(a, q, matched, s);
  return c ? launch_gather_rc<32, true>(a, q, matched, s)
           : launch_gather_rc<32, false>(a, q, matched, s);
}

hipError_t launch_rebin_adjoint(const RebinAdjArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(view_flags_kernel, dim3(a.nviews), dim3(256), 0, s, a.gbar,
                     (size_t)a.nrows * a.cpitch, a.flags);
  const int blocks = a.raw_nviews * ((a.raw_ncols + 63) / 64);
  hipLaunchKernelGGL(rebin_adjoint_kernel, dim3(blocks), dim3(64 * kRebinWaves), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_fill(float* p, size_t n, float v, hipStream_t s) {
  const size_t blocks = std::min<size_t>((n + 255) / 256, 65536);
  hipLaunchKernelGGL(fill_kernel, dim3((unsigned)std::max<size_t>(blocks, 1)), dim3(256), 0, s, p,
                     n, v);
  return hipGetLastError();
}

}  // namespace fct
