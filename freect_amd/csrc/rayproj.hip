// rayproj.hip -- ray-driven helical projector of the native volume onto the
// raw fan data (Joseph's method) and its exact transpose.  No counterpart in
// the reference: the data-consistency refinement needs a forward model of
// the measured line integrals, and the WFBP chain's own transpose (a filtered
// sinogram) or the voxel-driven matched projector (which leaves channels
// between the footprints of voxels larger than a channel empty) are not one.
//
// A ray is that of the synthetic scan generator (aux_kernels.hip): the
// (deflected) focal spot of raw projection v to its detector cell, in the
// plan's frame (a clockwise scan as its mirror image, like the voxel
// tables).  Joseph's method (P. M. Joseph, "An improved algorithm for
// reprojecting rays through pixel images", IEEE TMI 1 (1982) 192): along the
// in-plane axis the ray is most aligned with, at every voxel plane of that
// axis, the volume is interpolated bilinearly in the other in-plane axis and
// z (zero outside the volume) and the samples are summed times the path
// length per plane, |step / u_axis|.  The transpose scatters each ray's
// value with the same weights.
//
// Two forms of each: the general kernels (a ray per thread, FP64 set-up, the
// transpose by FP32 atomics on the volume) take any geometry, a graph capture
// that starts before the plan has its tables, and plans without memory for
// them; the table-driven ones
// below them take everything else.
#include <algorithm>
#include <cmath>

#include "wave_ops.h"
#include "wfbp_internal.h"

namespace fct {
namespace {

struct Ray {
  float sx, sy, sz, ux, uy, uz;
};

// FP64 ray of (view, row, channel), then FP32 for the march (positions of a
// few hundred mm: 3e-5 mm resolution); the part that no row changes apart.
struct RayDir {
  double sx, sy, sz, dx, dy, oz;
};
__device__ __forceinline__ RayDir ray_dir(const RayProjArgs& a, int v, int c) {
  const double ang = a.angle0 + a.dtheta * (double)v;
  const double ca = cos(ang), sa = sin(ang);
  const double beta = ((double)c - a.cc) * a.dgamma;
  RayDir d{a.r * ca, a.r * sa, a.z0 + a.dz * (double)v, -a.dsd * cos(ang + beta),
           -a.dsd * sin(ang + beta), 0.0};
  if (a.states > 1) {
    const double* o = a.ffs_off[v % a.states];
    const double ox = o[0] * ca - o[1] * sa, oy = o[0] * sa + o[1] * ca;
    d.sx += ox;
    d.sy += oy;
    d.sz += o[2];
    d.dx -= ox;
    d.dy -= oy;
    d.oz = o[2];
  }
  return d;
}
__device__ __forceinline__ Ray ray_of(const RayProjArgs& a, const RayDir& d, int row) {
  const double dz = ((double)row - a.cr) * a.drow - d.oz;
  const double len = sqrt(d.dx * d.dx + d.dy * d.dy + dz * dz);
  return Ray{(float)d.sx, (float)d.sy, (float)d.sz, (float)(d.dx / len), (float)(d.dy / len),
             (float)(dz / len)};
}
__device__ __forceinline__ Ray make_ray(const RayProjArgs& a, int v, int row, int c) {
  return ray_of(a, ray_dir(a, v, c), row);
}

// Index range [lo, hi] of the planes whose sample f = A + i B lies in
// (-1, n) (the bilinear footprint touches the volume).
__device__ __forceinline__ void plane_range(float A, float B, int n, int* lo, int* hi) {
  if (B == 0.0f) {
    if (!(A > -1.0f && A < (float)n)) *lo = 1, *hi = 0;
    return;
  }
  float t0 = (-1.0f - A) / B, t1 = ((float)n - A) / B;
  if (t0 > t1) {
    const float t = t0;
    t0 = t1;
    t1 = t;
  }
  *lo = max(*lo, (int)floorf(t0));
  *hi = min(*hi, (int)ceilf(t1));
}

// Walk of a ray: calls f(i_primary, j, k, weight) for every volume voxel a
// plane's bilinear sample touches (the weight without the path length).
template <class F>
__device__ __forceinline__ float walk(const RayProjArgs& a, const Ray& r, F&& f) {
  const bool xmajor = fabsf(r.ux) >= fabsf(r.uy);
  // Primary axis p (planes), secondary s (in-plane), and z.
  const float p0 = xmajor ? a.gx0 : a.gy0, dp = xmajor ? a.gdx : a.gdy;
  const float q0 = xmajor ? a.gy0 : a.gx0, dq = xmajor ? a.gdy : a.gdx;
  const float sp = xmajor ? r.sx : r.sy, sq = xmajor ? r.sy : r.sx;
  const float up = xmajor ? r.ux : r.uy, uq = xmajor ? r.uy : r.ux;
  const int np = xmajor ? a.nx : a.ny, nq = xmajor ? a.ny : a.nx;
  // t at plane i: (p0 + i dp - sp) / up; sample positions linear in i.
  const float t0 = (p0 - sp) / up, dt = dp / up;
  const float Aq = (sq + t0 * uq - q0) / dq, Bq = dt * uq / dq;
  const float Az = (r.sz + t0 * r.uz - a.gz0) / a.gdz, Bz = dt * r.uz / a.gdz;
  int lo = 0, hi = np - 1;
  plane_range(Aq, Bq, nq, &lo, &hi);
  plane_range(Az, Bz, a.nz, &lo, &hi);
  for (int i = lo; i <= hi; ++i) {
    const float fq = fmaf((float)i, Bq, Aq), fz = fmaf((float)i, Bz, Az);
    const float jq = floorf(fq), kz = floorf(fz);
    const float wq = fq - jq, wz = fz - kz;
    const int j = (int)jq, k = (int)kz;
#pragma unroll
    for (int dk = 0; dk < 2; ++dk)
#pragma unroll
      for (int dj = 0; dj < 2; ++dj) {
        const int jj = j + dj, kk = k + dk;
        if (jj < 0 || jj >= nq || kk < 0 || kk >= a.nz) continue;
        const float wgt = (dj ? wq : 1.0f - wq) * (dk ? wz : 1.0f - wz);
        const int ix = xmajor ? i : jj, iy = xmajor ? jj : i;
        f(((size_t)kk * a.ny + iy) * a.nx + ix, wgt);
      }
  }
  return fabsf(dt);   // path length per plane (u is a unit vector)
}

__global__ __launch_bounds__(256) void ray_project_kernel(RayProjArgs a) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  const int row = blockIdx.y, v = a.v0 + blockIdx.z;
  if (c >= a.ncols) return;
  const Ray r = make_ray(a, v, row, c);
  float acc = 0.0f;
  const float len = walk(a, r, [&](size_t o, float w) { acc = fmaf(w, a.vol_in[o], acc); });
  a.raw_out[((size_t)(v - a.v0) * a.nrows + row) * a.ncols + c] = acc * len;
}

__global__ __launch_bounds__(256) void ray_backproject_kernel(RayProjArgs a) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  const int row = blockIdx.y, v = a.v0 + blockIdx.z;
  if (c >= a.ncols) return;
  const float val = a.raw_in[((size_t)(v - a.v0) * a.nrows + row) * a.ncols + c];
  if (val == 0.0f) return;
  const Ray r = make_ray(a, v, row, c);
  // The path length is known before the walk: |dp / u_primary|.
  const bool xmajor = fabsf(r.ux) >= fabsf(r.uy);
  const float len = fabsf((xmajor ? a.gdx : a.gdy) / (xmajor ? r.ux : r.uy));
  const float s = val * len;
  walk(a, r, [&](size_t o, float w) { atomicAdd(a.vol_out + o, w * s); });
}


// ---------------------------------------------------------------------------
// Table-driven forms.  Within one raw view the in-plane path of a ray depends
// on its channel only: fq = A + i B (sample position at plane i), the
// fraction of the way from the focal spot to the detector T = T0 + i DT, and
// fz = zoff + T (w_row - oz) / gdz.  ray_table_kernel writes (A, B, T0, DT)
// per (view, channel) from FP64, and a bit that says whether the planes are x
// planes.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void ray_table_kernel(RayProjArgs a, RayTables t) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  const int v = blockIdx.y + gridDim.y * blockIdx.z;
  if (v >= a.v1) return;
  const double ang = a.angle0 + a.dtheta * (double)v;
  const double ca = cos(ang), sa = sin(ang);
  const int rho = v % a.states;
  const double o0 = a.ffs_off[rho][0], o1 = a.ffs_off[rho][1], oz = a.ffs_off[rho][2];
  const double sx = (a.r + o0) * ca - o1 * sa, sy = (a.r + o0) * sa + o1 * ca;
  if (c == 0) {
    t.view[2 * v] = make_float4((float)ca, (float)sa, (float)(a.r + o0), (float)o1);
    t.view[2 * v + 1] = make_float4((float)((-a.cr * a.drow - oz) / a.ddz), (float)o0, 0.0f, 0.0f);
    t.zoff[v] = (a.z0 + a.dz * (double)v + oz - a.dz0) / a.ddz;
  }
  if (c >= a.ncols) return;
  const double beta = ((double)c - a.cc) * a.dgamma;
  const double ux = -a.dsd * cos(ang + beta) - (o0 * ca - o1 * sa);
  const double uy = -a.dsd * sin(ang + beta) - (o0 * sa + o1 * ca);
  const double len = sqrt(ux * ux + uy * uy);
  const bool xmajor = fabsf((float)(ux / len)) >= fabsf((float)(uy / len));
  const double p0 = xmajor ? a.dx0 : a.dy0, dp = xmajor ? a.ddx : a.ddy;
  const double q0 = xmajor ? a.dy0 : a.dx0, dq = xmajor ? a.ddy : a.ddx;
  const double sp = xmajor ? sx : sy, sq = xmajor ? sy : sx;
  const double up = xmajor ? ux : uy, uq = xmajor ? uy : ux;
  const double t0 = (p0 - sp) / up, dt = dp / up;
  t.ray[(size_t)v * a.ncols + c] =
      make_float4((float)((sq + t0 * uq - q0) / dq), (float)(dt * uq / dq), (float)t0, (float)dt);
  const uint64_t bits = __ballot(xmajor);   // (a wave: 64 channels from a multiple of 64)
  if ((c & 63) == 0) t.axis[(size_t)v * ((a.ncols + 63) >> 6) + (c >> 6)] = bits;
  if (v < a.states) t.len2[(size_t)rho * a.ncols + c] = (float)(ux * ux + uy * uy);
}

// Whether the planes of (view, channel) are x planes.
__device__ __forceinline__ bool x_planes(const RayTables& t, int ncols, int v, int c) {
  const uint32_t* w = reinterpret_cast<const uint32_t*>(t.axis + (size_t)v * ((ncols + 63) >> 6));
  return w[c >> 5] >> (c & 31) & 1;
}

// The volume with two planes of zeros on every side, in its own order and
// with x and y exchanged, so that the projector reads neighbouring samples of
// neighbouring rays from neighbouring addresses for either plane axis and
// needs no bounds test (a sample's footprint may reach two planes outside).
// T float2: entry (z, y, x) holds slices z and z + 1, so that the four taps
// of a sample are 16 consecutive bytes.
constexpr int kPad = 2;
__device__ __forceinline__ void pad_entry(float* e, float v, float) { *e = v; }
__device__ __forceinline__ void pad_entry(float2* e, float v, float up) { *e = make_float2(v, up); }

template <class T>
__global__ __launch_bounds__(256) void ray_pad_kernel(RayProjArgs a, T* __restrict__ nat,
                                                      T* __restrict__ swp) {
  __shared__ T tile[32][33];
  const int px = a.nx + 2 * kPad, py = a.ny + 2 * kPad;
  const int bx = blockIdx.x * 32, by = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int kz = blockIdx.z; kz < a.nz + 2 * kPad; kz += gridDim.z) {
    const int z = kz - kPad;
    const size_t plane = (size_t)kz * px * py;
    for (int r = ty; r < 32; r += 8) {
      const int X = bx + tx, Y = by + r, x = X - kPad, y = Y - kPad;
      const bool in = x >= 0 && x < a.nx && y >= 0 && y < a.ny;
      auto at = [&](int s) {
        return in && s >= 0 && s < a.nz ? a.vol_in[((size_t)s * a.ny + y) * a.nx + x] : 0.0f;
      };
      T v;
      pad_entry(&v, at(z), sizeof(T) == sizeof(float) ? 0.0f : at(z + 1));
      if (X < px && Y < py) nat[plane + (size_t)Y * px + X] = v;
      tile[r][tx] = v;
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
      const int X = bx + r, Y = by + tx;
      if (X < px && Y < py) swp[plane + (size_t)X * py + Y] = tile[tx][r];
    }
    __syncthreads();
  }
}

// Planes [lo, hi] whose sample A + i B lies in (-1, n), as reals.
__device__ __forceinline__ void plane_span(float A, float B, int n, float* lo, float* hi) {
  if (B == 0.0f) {
    if (!(A > -1.0f && A < (float)n)) *lo = 1.0f, *hi = 0.0f;
    return;
  }
  const float t0 = (-1.0f - A) / B, t1 = ((float)n - A) / B;
  *lo = fmaxf(*lo, fminf(t0, t1));
  *hi = fminf(*hi, fmaxf(t0, t1));
}

constexpr int kRsrcWord3 = 0x00020000;   // raw buffer, 32-bit data format (gfx9)
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// A plane's four taps: one 16-byte load (T float2), or two 8-byte loads
// (slices k and k + 1 at j, j + 1).
struct RayTap {
  u32x2 a, b;
  float wq, wz;
};

template <class T>
struct RayWalk {
  float Aq, Bq, Az, Bz;
  __amdgpu_buffer_rsrc_t r0, r1;   // the padded volume from slice -2 and (float) from slice -1
  // Entries of a plane, bytes of a row, byte offset of (0, 0, 0) past the padding.
  int plane, row_bytes, origin;
  __device__ __forceinline__ RayTap fetch(int i) const {
    RayTap t;
    const float fq = fmaf((float)i, Bq, Aq), fz = fmaf((float)i, Bz, Az);
    const int j = floor_int(fq), k = floor_int(fz);
    t.wq = __builtin_amdgcn_fractf(fq);
    t.wz = __builtin_amdgcn_fractf(fz);
    const int o = (__mul24(k, plane) + j) * (int)sizeof(T) + origin;
    if constexpr (sizeof(T) == sizeof(float2)) {
      const u32x4 q = __builtin_amdgcn_raw_buffer_load_b128(r0, o, i * row_bytes, 0);
      t.a = u32x2{q.x, q.z};
      t.b = u32x2{q.y, q.w};
    } else {
      t.a = __builtin_amdgcn_raw_buffer_load_b64(r0, o, i * row_bytes, 0);
      t.b = __builtin_amdgcn_raw_buffer_load_b64(r1, o, i * row_bytes, 0);
    }
    return t;
  }
};
__device__ __forceinline__ float ray_combine(const RayTap& t) {
  const uint32_t a0 = t.a.x, a1 = t.a.y, b0 = t.b.x, b1 = t.b.y;
  // Products with both weights, not a + w (b - a): an infinite sample gives an
  // infinite value there, as in the general kernel, and not a NaN.
  const float uq = 1.0f - t.wq, uz = 1.0f - t.wz;
  const float lo = fmaf(t.wq, __uint_as_float(a1), uq * __uint_as_float(a0));
  const float hi = fmaf(t.wq, __uint_as_float(b1), uq * __uint_as_float(b0));
  return fmaf(t.wz, hi, uz * lo);
}

// One ray per lane, 64 neighbouring channels of one detector row per wave,
// four rows per workgroup: the waves of a workgroup read the same columns of
// neighbouring slices.  A wave's lanes advance plane by plane together; the
// planes that every one of its rays samples run unmasked, four at a time
// (their loads in flight).  18 VALU instructions and one 16-byte load
// per sample instead of 40 and four loads: 1476 views x 16 x 736 rays through
// 384 x 384 x 32 voxels 30.8 -> 5.9 ms with two 8-byte loads (which bound it:
// 19 cycles of a CU's L1 each, VALU 2.8 ms of the 5.9), 3.9 ms with one of 16
// bytes: address unit 88 % and VALU issue 90 % of its cycles.  1 to 16 rows per workgroup and 2 to 8 planes in flight
// are within 2 %.
constexpr int kRayRows = 4;
template <class T>
__global__ __launch_bounds__(64 * kRayRows) void ray_project_table_kernel(RayProjArgs a, RayTables t,
                                                                const T* __restrict__ nat,
                                                                const T* __restrict__ swp,
                                                                uint32_t pad_bytes) {
  const int cg = (a.ncols + 63) >> 6, rg = (a.nrows + kRayRows - 1) / kRayRows;
  const int id = xcd_block(blockIdx.x, gridDim.x);
  const int v = id / (cg * rg), rest = id - v * cg * rg;
  const int c = (rest % cg) * 64 + (threadIdx.x & 63);
  const int row = __builtin_amdgcn_readfirstlane((rest / cg) * kRayRows + (threadIdx.x >> 6));
  if (row >= a.nrows) return;
  const bool in = c < a.ncols;
  const float4 e = t.ray[(size_t)v * a.ncols + (in ? c : a.ncols - 1)];
  const bool xm = ld_uniform(t.axis + (size_t)v * cg + rest % cg) >> (c & 63) & 1;
  const double oz = a.states > 1 ? t.zsrc[v % a.states] : 0.0;
  const double wz = ((double)row - a.cr) * a.drow - oz;
  const double g = wz / a.ddz;
  RayWalk<T> w;
  w.Aq = e.x;
  w.Bq = e.y;
  w.Az = (float)(t.zoff[v] + (double)e.z * g);
  w.Bz = (float)((double)e.w * g);
  float flo = 0.0f, fhi = (float)((xm ? a.nx : a.ny) - 1);
  plane_span(w.Aq, w.Bq, xm ? a.ny : a.nx, &flo, &fhi);
  plane_span(w.Az, w.Bz, a.nz, &flo, &fhi);
  const bool any_plane = in && flo <= fhi;
  const int ilo = any_plane ? (int)ceilf(flo) : 0, ihi = any_plane ? (int)floorf(fhi) : -1;
  const int px = a.nx + 2 * kPad, py = a.ny + 2 * kPad;
  w.plane = px * py;
  const uint32_t plane_bytes = (uint32_t)w.plane * (uint32_t)sizeof(T);
  float acc = 0.0f;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const bool mine = ilo <= ihi && xm == (m == 1);
    if (!__any(mine)) continue;
    // Planes some lane samples, and those that every lane of this axis does.
    const int u0 = wave_min_i(mine ? ilo : INT32_MAX), u1 = wave_max_i(mine ? ihi : -1);
    const int b0 = wave_max_i(mine ? ilo : -1), b1 = wave_min_i(mine ? ihi : INT32_MAX);
    if (!mine) continue;
    const char* base = reinterpret_cast<const char*>(m ? swp : nat);
    w.r0 = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)pad_bytes, kRsrcWord3);
    w.r1 = __builtin_amdgcn_make_buffer_rsrc((void*)(base + plane_bytes), 0,
                                             (int)(pad_bytes - plane_bytes), kRsrcWord3);
    w.row_bytes = (m ? py : px) * (int)sizeof(T);
    w.origin = kPad * ((int)plane_bytes + w.row_bytes + (int)sizeof(T));
    int i = u0;
    for (; i <= u1 && i < b0; ++i)
      if (i >= ilo && i <= ihi) acc += ray_combine(w.fetch(i));
    for (; i + 3 <= b1; i += 4) {
      RayTap tp[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) tp[k] = w.fetch(i + k);
#pragma unroll
      for (int k = 0; k < 4; ++k) acc += ray_combine(tp[k]);
    }
    for (; i <= u1; ++i)
      if (i >= ilo && i <= ihi) acc += ray_combine(w.fetch(i));
  }
  if (!in) return;
  const double l2 = (double)t.len2[(size_t)(a.states > 1 ? v % a.states : 0) * a.ncols + c];
  a.raw_out[((size_t)v * a.nrows + row) * a.ncols + c] =
      acc * fabsf(e.w) * (float)sqrt(l2 + wz * wz);
}

// Per ray of the transpose: its in-plane sample positions (fq = A + i B, the
// general kernels' FP32 values) and its value times the path length per plane.
// The planes are those of the table, which the projector and the gather read
// too: decided once more here, from the ray with its row's slope, the axis of
// a ray within an FP32 rounding of the diagonal could differ from theirs, and
// the gather lost the ray.
// 32 channels of a view whose rays are all zero (a data term on some of the
// views) get no records and are left out by the gather: bit c >> 5 of nz[view]
// says that there is another value, a byte per block.
__global__ __launch_bounds__(256) void ray_record_kernel(RayProjArgs a, RayTables t,
                                                         float* __restrict__ rec,
                                                         uint8_t* __restrict__ nz) {
  __shared__ uint32_t groups[4];
  const int cg = (a.ncols + 255) >> 8;
  const int v = blockIdx.x / cg, g = blockIdx.x - v * cg, c = g * 256 + threadIdx.x;
  const bool in = c < a.ncols;
  const size_t o0 = (size_t)v * a.nrows * a.ncols + (in ? c : 0);
  bool some = false;
#pragma unroll 8
  for (int row = 0; row < a.nrows; ++row)
    some = some || a.raw_in[o0 + (size_t)row * a.ncols] != 0.0f;
  const uint64_t m = __ballot(in && some);
  const uint32_t half = threadIdx.x & 32 ? (uint32_t)(m >> 32) : (uint32_t)m;
  if ((threadIdx.x & 63) == 0)
    groups[threadIdx.x >> 6] = ((uint32_t)m ? 1u : 0u) | (m >> 32 ? 2u : 0u);
  __syncthreads();
  if (threadIdx.x == 0)
    nz[(size_t)v * 8 + g] =
        (uint8_t)(groups[0] | groups[1] << 2 | groups[2] << 4 | groups[3] << 6);
  if (!in || !half) return;
  const RayDir d = ray_dir(a, v, c);
  const bool xmajor = x_planes(t, a.ncols, v, c);
  for (int row = 0; row < a.nrows; ++row) {
    const Ray r = ray_of(a, d, row);
    const float p0 = xmajor ? a.gx0 : a.gy0, dp = xmajor ? a.gdx : a.gdy;
    const float q0 = xmajor ? a.gy0 : a.gx0, dq = xmajor ? a.gdy : a.gdx;
    const float sp = xmajor ? r.sx : r.sy, sq = xmajor ? r.sy : r.sx;
    const float up = xmajor ? r.ux : r.uy, uq = xmajor ? r.uy : r.ux;
    const float t0 = (p0 - sp) / up, dt = dp / up;
    const size_t o = o0 + (size_t)row * a.ncols;
    rec[3 * o] = (sq + t0 * uq - q0) / dq;
    rec[3 * o + 1] = dt * uq / dq;
    rec[3 * o + 2] = a.raw_in[o] * fabsf(dt);
  }
}

// The transpose as a gather: one wave per tile of 8 x 8 voxel columns and K
// slices, each lane owning a column.  Per view the rays whose planes sample
// the column are a few neighbouring channels around the one through its
// centre (the position of the column on the detector, plus and minus the
// angle of one voxel); each of them meets the K slices in consecutive
// detector rows, whose values are added to the lane's slices in LDS (one read
// and one write of two slices per row, conflict-free: a lane only touches its
// own bank).  No global atomics per tap: 1476 views x 16 x 736 rays into 384
// x 384 x 32 voxels 791 ms (four global atomics per sample) -> 8.8 ms.  LDS
// float atomics in place of the read and write took 130 ms.  K = 32 slices
// of LDS leave 17 waves per CU; K = 16 runs the per-view set-up twice as
// often (9.0 ms), and is used where the volume has no more slices.  The
// views are split so that about 128 waves per CU are launched (at 32 the
// last round of waves leaves the chip half empty: 11.7 ms); each adds its
// sums to the volume once, at its end.  15 VALU instructions and one 12-byte
// load per row; counters: address unit 81 % busy (17 cycles per load), VALU issue
// 79 %, 57 of 64 lanes active.
template <int K, bool FFS>
__global__ __launch_bounds__(64) void ray_gather_kernel(RayProjArgs a, RayTables t, RayGather q) {
  // Slice k at row k + 2; rows 0, 1, K + 2, K + 3 take what falls outside.
  __shared__ float acc[(K + 4) * 64];
  const int lane = threadIdx.x;
  const int tiles = q.tiles_x * q.tiles_y, per = tiles * q.slabs;
  const int id = xcd_block(blockIdx.x, gridDim.x);
  const int split = id / per, rest = id - split * per;
  const int slab = rest / tiles, tile = rest - slab * tiles;
  const int ty = tile / q.tiles_x, tx = tile - ty * q.tiles_x;
  const int ix = tx * 8 + (lane & 7), iy = ty * 8 + (lane >> 3);
  const bool active = ix < a.nx && iy < a.ny;
  const float fix = (float)ix, fiy = (float)iy;
  const float x = fmaf(fix, a.gdx, a.gx0), y = fmaf(fiy, a.gdy, a.gy0);
  const int s0 = slab * K;
#pragma unroll
  for (int k = 0; k < K + 4; ++k) acc[k * 64 + lane] = 0.0f;

  // Views whose cone can reach the slab, and this wave's share of them.
  int va, vb;
  {
    const double z0 = a.dz0 + s0 * a.ddz, z1 = z0 + (K - 1) * a.ddz;
    double f0 = (fmin(z0, z1) - q.reach - a.z0) / a.dz, f1 = (fmax(z0, z1) + q.reach - a.z0) / a.dz;
    const double lo = fmin(f0, f1), hi = fmax(f0, f1);
    va = (int)fmax(0.0, fmin(floor(lo), (double)a.v1));
    vb = (int)fmax(0.0, fmin(ceil(hi) + 1.0, (double)a.v1));
    const int n = max(vb - va, 0), first = va;
    va = first + (int)((long long)n * split / q.nsplit);
    vb = first + (int)((long long)n * (split + 1) / q.nsplit);
  }
  const float adx = fabsf(a.gdx), ady = fabsf(a.gdy), dmax = fmaxf(adx, ady);
  const float inv_dg = (float)(1.0 / a.dgamma), ccf = (float)a.cc, dsd = (float)a.dsd;
  const float az = (float)(a.drow / a.ddz), iaz = (float)(a.ddz / a.drow);

  // (The bytes of channel groups past the detector are not written.)
  const uint64_t groups = ~0ull >> (64 - ((a.ncols + 255) >> 8) * 8);
  for (int v = va; v < vb; ++v) {
    const uint64_t nz = ld_uniform(q.nz + v) & groups;
    if (!nz) continue;
    const float4 e0 = ld_uniform4(t.view + 2 * v), e1 = ld_uniform4(t.view + 2 * v + 1);
    const float ca = e0.x, sa = e0.y, bz = e1.x;
    const float zo = (float)(ld_uniform(t.zoff + v) - (double)s0);
    // The column seen from the focal spot, in the view's frame.
    const float d0 = fmaf(x, ca, fmaf(y, sa, -e0.z)), d1 = fmaf(y, ca, -fmaf(x, sa, e0.w));
    const float l2 = fmaf(d0, d0, d1 * d1), il = __builtin_amdgcn_rsqf(l2), l = l2 * il;
    const float u0 = d0 * il, u1 = d1 * il;
    // Its detector point: |S' + tau u - S| = Dsd around the undeflected S.
    float tau = dsd, tb = d1 / d0;
    if (FFS) {
      const float o0 = e1.y, o1 = e0.w, ou = fmaf(o0, u0, o1 * u1);
      tau = __builtin_amdgcn_sqrtf(fmaf(ou, ou, dsd * dsd - fmaf(o0, o0, o1 * o1))) - ou;
      tb = fmaf(tau, u1, o1) / fmaf(tau, u0, o0);
    }
    const float cp = fmaf(atanf(tb), inv_dg, ccf);
    // Half width in channels: one voxel along the secondary axis of the
    // candidate rays (both axes near the diagonals), the second-order terms
    // and rounding covered by the margins.
    const float ux = fabsf(u0 * ca - u1 * sa), uy = fabsf(u0 * sa + u1 * ca);
    const float hx = ady * ux, hy = adx * uy, thr = fmaf(3.0f * dmax, il, 0.01f);
    const float h = ux - uy > thr ? hx : ux - uy < -thr ? hy : fmaxf(hx, hy);
    const float hw = h * il * inv_dg * fmaf(1.5f * dmax, il, 1.02f) + 0.02f;
    const int c0 = max((int)ceilf(cp - hw), 0);
    const int c1 = active ? min((int)floorf(cp + hw), a.ncols - 1) : -1;
    // Rows that can reach slices (-1, K) of the slab over the candidates.
    const float itau = __builtin_amdgcn_rcpf(tau);
    const float t1 = fmaxf(l - 1.5f * dmax, 1e-3f * l) * itau * 0.99f;
    const float t2 = (l + 1.5f * dmax) * itau * 1.01f;
    const float i1 = __builtin_amdgcn_rcpf(t1), i2 = __builtin_amdgcn_rcpf(t2);
    const float ea = -1.0f - zo, eb = (float)K - zo;
    const float ra = (fminf(ea * i1, ea * i2) - bz) * iaz, rb = (fmaxf(eb * i1, eb * i2) - bz) * iaz;
    const bool some = c0 <= c1 && (nz >> (c0 >> 5) & ((2ull << ((c1 >> 5) - (c0 >> 5))) - 1));
    const int rlo = max(wave_min_i(some ? (int)ceilf(fminf(ra, rb) - 0.01f) : INT32_MAX), 0);
    const int rhi = min(wave_max_i(some ? (int)floorf(fmaxf(ra, rb) + 0.01f) : -1), a.nrows - 1);
    if (rlo > rhi) continue;
    const int nc = wave_max_i(some ? c1 - c0 + 1 : 0);
    const uint32_t row_bytes = (uint32_t)a.ncols * 12u;
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(q.rec + (size_t)v * a.nrows * a.ncols * 3), 0, (int)(row_bytes * a.nrows),
        kRsrcWord3);
    const float4* tv = t.ray + (size_t)v * a.ncols;
    for (int m = 0; m < nc; ++m) {
      const int c = c0 + m;
      const int cc = min(c, a.ncols - 1);
      const float4 e = tv[cc];
      const bool xm = x_planes(t, a.ncols, v, cc);
      const float prim = xm ? fix : fiy, sec = xm ? fiy : fix;
      // (The rows' own positions differ from the table's by rounding.)
      if (!(fabsf(fmaf(prim, e.y, e.x) - sec) < 1.001f) || c > c1 || !(nz >> (cc >> 5) & 1)) continue;
      const float T = fmaf(prim, e.w, e.z), Sz = T * az, F0 = fmaf(T, bz, zo);
      const int co = c * 12;
      auto add = [&](float r, u32x3 d) {
        const uint32_t A = d.x, B = d.y, V = d.z;
        const float w = 1.0f - fabsf(fmaf(prim, __uint_as_float(B), __uint_as_float(A)) - sec);
        const float s = w > 0.0f ? w * __uint_as_float(V) : 0.0f;
        const float fz = fmaf(r, Sz, F0);
        const int k = min(max(floor_int(fz), -2), K);
        const float wz = __builtin_amdgcn_fractf(fz);
        float* p = acc + (k + 2) * 64 + lane;
        const float x0 = p[0], x1 = p[64];
        p[0] = fmaf(s, 1.0f - wz, x0);   // (finite weights: s may be infinite)
        p[64] = fmaf(s, wz, x1);
      };
      int r = rlo;
      for (; r + 3 <= rhi; r += 4) {
        u32x3 d[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          d[u] = __builtin_amdgcn_raw_buffer_load_b96(rv, co, (r + u) * (int)row_bytes, 0);
#pragma unroll
        for (int u = 0; u < 4; ++u) add((float)(r + u), d[u]);
      }
      for (; r <= rhi; ++r)
        add((float)r, __builtin_amdgcn_raw_buffer_load_b96(rv, co, r * (int)row_bytes, 0));
    }
  }
  if (!active) return;
#pragma unroll
  for (int k = 0; k < K; ++k)
    if (s0 + k < a.nz) {
      float* o = a.vol_out + ((size_t)(s0 + k) * a.ny + iy) * a.nx + ix;
      const float s = acc[(k + 2) * 64 + lane];
      if (q.nsplit > 1)
        unsafeAtomicAdd(o, s);
      else
        *o = s;
    }
}

}  // namespace

hipError_t launch_ray_project(const RayProjArgs& a, bool transpose, hipStream_t s) {
  if (a.v1 <= a.v0) return hipSuccess;
  dim3 grid((a.ncols + 255) / 256, a.nrows, a.v1 - a.v0);
  if (transpose)
    hipLaunchKernelGGL(ray_backproject_kernel, grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL(ray_project_kernel, grid, dim3(256), 0, s, a);
  return hipGetLastError();
}


// The table-driven forms take volumes that lie inside the focal spot's circle
// with room to spare (every sampled plane in front of the source, the
// candidate margins of the gather) and whose padded copies a buffer resource
// and 24-bit products address.
bool ray_tables_apply(const RayProjArgs& a) {
  double rc = 0.0;
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j)
      rc = std::max(rc, std::hypot(a.dx0 + (i ? a.nx : -1) * a.ddx, a.dy0 + (j ? a.ny : -1) * a.ddy));
  double defl = 0.0;
  for (int s = 0; s < a.states; ++s)
    defl = std::max(defl, std::hypot(a.ffs_off[s][0], a.ffs_off[s][1]));
  const double room = a.r - defl - rc, fan = a.ncols * a.dgamma;
  const double plane = 4.0 * (a.nx + 2.0 * kPad) * (a.ny + 2.0 * kPad);
  return room > 0.1 * a.r && std::max(std::fabs(a.ddx), std::fabs(a.ddy)) <= 0.1 * room &&
         defl < 0.01 * a.dsd && fan < 2.8 && plane < (double)(1 << 23) &&
         plane * (a.nz + 2.0 * kPad) < 4294967000.0 &&
         (double)a.v1 * a.ncols < 2147483647.0 &&
         (double)a.v1 * ((a.nrows + kRayRows - 1) / kRayRows) * ((a.ncols + 63) / 64) <
             2147483647.0;
}

size_t ray_table_bytes(const RayProjArgs& a) {
  const size_t nv = a.v1;
  return nv * a.ncols * sizeof(float4) + 2 * nv * sizeof(float4) + nv * sizeof(double) +
         nv * ((a.ncols + 63) / 64) * sizeof(uint64_t) +
         (size_t)a.states * a.ncols * sizeof(float);
}

size_t ray_pad_elems(const RayProjArgs& a) {
  return (size_t)(a.nx + 2 * kPad) * (a.ny + 2 * kPad) * (a.nz + 2 * kPad);
}

RayTables ray_table_layout(const RayProjArgs& a, void* mem) {
  RayTables t{};
  char* p = static_cast<char*>(mem);
  auto take = [&](size_t n) {
    char* q = p;
    p += n;
    return q;
  };
  const size_t nv = a.v1;
  t.ray = reinterpret_cast<float4*>(take(nv * a.ncols * sizeof(float4)));
  t.view = reinterpret_cast<float4*>(take(2 * nv * sizeof(float4)));
  t.zoff = reinterpret_cast<double*>(take(nv * sizeof(double)));
  t.axis = reinterpret_cast<uint64_t*>(take(nv * ((a.ncols + 63) / 64) * sizeof(uint64_t)));
  t.len2 = reinterpret_cast<float*>(take((size_t)a.states * a.ncols * sizeof(float)));
  for (int s = 0; s < a.states; ++s) t.zsrc[s] = a.ffs_off[s][2];
  return t;
}

hipError_t launch_ray_table(const RayProjArgs& a, const RayTables& t, hipStream_t s) {
  const int gy = std::min(a.v1, 32768);
  hipLaunchKernelGGL(ray_table_kernel, dim3((a.ncols + 255) / 256, gy, (a.v1 + gy - 1) / gy),
                     dim3(256), 0, s, a, t);
  return hipGetLastError();
}

// Whether a padded copy with two slices per entry is within a buffer
// resource's range too (else the copies hold one).
bool ray_pad_pairs(const RayProjArgs& a) {
  return (double)ray_pad_elems(a) * sizeof(float2) < 4294967000.0;
}

template <class T>
hipError_t launch_project_table(const RayProjArgs& a, const RayTables& t, T* pad, hipStream_t s) {
  const size_t n = ray_pad_elems(a);
  hipLaunchKernelGGL(ray_pad_kernel<T>,
                     dim3((a.nx + 2 * kPad + 31) / 32, (a.ny + 2 * kPad + 31) / 32,
                          std::min(a.nz + 2 * kPad, 65535)),
                     dim3(256), 0, s, a, pad, pad + n);
  const int blocks = a.v1 * ((a.nrows + kRayRows - 1) / kRayRows) * ((a.ncols + 63) / 64);
  hipLaunchKernelGGL(ray_project_table_kernel<T>, dim3(blocks), dim3(64 * kRayRows), 0, s, a, t, pad,
                     pad + n, (uint32_t)(n * sizeof(T)));
  return hipGetLastError();
}

hipError_t launch_ray_project_table(const RayProjArgs& a, const RayTables& t, float* pad,
                                    bool pairs, hipStream_t s) {
  return pairs ? launch_project_table(a, t, reinterpret_cast<float2*>(pad), s)
               : launch_project_table(a, t, pad, s);
}

hipError_t launch_ray_gather(const RayProjArgs& a, const RayTables& t, float* rec, int ncu,
                             hipStream_t s) {
  RayGather q{};
  q.nz = reinterpret_cast<const uint64_t*>(rec);
  rec += 2 * (size_t)a.v1;
  q.rec = rec;
  const int K = a.nz <= 16 ? 16 : 32;
  q.tiles_x = (a.nx + 7) / 8;
  q.tiles_y = (a.ny + 7) / 8;
  q.slabs = (a.nz + K - 1) / K;
  double rc = 0.0, oz = 0.0;
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j)
      rc = std::max(rc, std::hypot(a.dx0 + (i ? a.nx : -1) * a.ddx, a.dy0 + (j ? a.ny : -1) * a.ddy));
  for (int i = 0; i < a.states; ++i) oz = std::max(oz, std::fabs(a.ffs_off[i][2]));
  const double w = std::max(std::fabs(a.cr), std::fabs(a.nrows - 1.0 - a.cr)) * a.drow + oz;
  q.reach = 1.05 * w * (a.r + rc) / (0.98 * a.dsd) + 2.0 * std::fabs(a.ddz) + oz;
  const long long waves = (long long)q.tiles_x * q.tiles_y * q.slabs;
  const double views = (2.0 * q.reach + K * std::fabs(a.ddz)) / std::fabs(a.dz);
  const long long most = std::max(1LL, (long long)(std::min(views, (double)a.v1) / 8.0));
  // Splits of at least 8 views, towards 128 waves per CU.
  q.nsplit = (int)std::min(most, std::max(1LL, (128LL * std::max(ncu, 1) + waves - 1) / waves));
  if (q.nsplit > 1) {
    const hipError_t e = launch_fill(a.vol_out, (size_t)a.nz * a.ny * a.nx, 0.0f, s);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(ray_record_kernel, dim3(a.v1 * ((a.ncols + 255) / 256)), dim3(256), 0, s, a,
                     t, rec, reinterpret_cast<uint8_t*>(const_cast<uint64_t*>(q.nz)));
  const dim3 grid((unsigned)(waves * q.nsplit));
  const bool ffs = a.states > 1;
  if (K == 16 && ffs)
    hipLaunchKernelGGL((ray_gather_kernel<16, true>), grid, dim3(64), 0, s, a, t, q);
  else if (K == 16)
    hipLaunchKernelGGL((ray_gather_kernel<16, false>), grid, dim3(64), 0, s, a, t, q);
  else if (ffs)
    hipLaunchKernelGGL((ray_gather_kernel<32, true>), grid, dim3(64), 0, s, a, t, q);
  else
    hipLaunchKernelGGL((ray_gather_kernel<32, false>), grid, dim3(64), 0, s, a, t, q);
  return hipGetLastError();
}

}  // namespace fct
