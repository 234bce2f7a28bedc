// backproject_v1.hip -- instruction-lean helical WFBP backprojection.
//
// Same arithmetic and selection as backproject.hip (cuda_kernels.cuh:198-287
// restated with the shared FP32 code of wfbp_math.h), organised to spend few
// instructions per selected (voxel, view) sample -- the kernel is bound by
// instruction issue (VALU and vector-memory), not by HBM:
//   * per (theta~, view parity) each lane's z-interval of |q| <= 1 is
//     [zt - kb - lt, zt - kb + lt]; the extremes of its ends over the tile
//     (DPP wave reductions, tabulated once per plan by bp_zbounds_kernel)
//     give, per view, the slices any lane of the wave can select; other
//     slices are skipped wave-uniformly and the exact per-sample selection
//     still runs, so selection is unchanged;
//   * the views of one theta~ are looked at together, lane l at the l-th: two
//     ballots give the views that cover the whole slab and those that cover
//     part of it, and scalar loops over their bits visit no other view.  (A
//     test per view inside the loop made the loop divergent for the
//     compiler and read the window table for every view.)  The view window
//     cuts into a view's slices only near its ends; only those views read
//     the exact slice range (a host table built with the same FP32 test);
//   * the sums over theta~ live in LDS: one read, fma and write per theta~
//     instead of registers that the 72-VGPR kernel spilled.
//     Together: FP16 512 x 512 x 320 49.4 -> 46.0 ms, six FP16 jobs of 256 x
//     256 in one launch 35.6 -> 32.8, BF16 256 x 256 x 64 4.87 -> 4.4, FP32 500
//     x 381 x 88 17.5 -> 17.2 (whole chains; of these the uniform loops 47.6 /
//     32.5 / 4.35 / 17.3);
//   * when a view covers the whole slab (the common case) the slices are
//     processed four at a time without a per-slice branch, the taps of the
//     four in flight together (with FP16 taps also for views covering part of
//     the slab, the slices outside the view's range masked);
//   * the detector row position is one fma per slice, and when the central
//     row is (nrows-1)/2 the cone test |q| <= 1 is implied exactly by the row
//     test, one unsigned compare;
//   * taps: FP32 row pairs (whole chains, kPrecisionPairs) are one 16-byte
//     buffer load, FP32 rows (the stage calls) two 8-byte loads, each at its
//     own vector offset: the texture-address unit takes 16.7 cycles per
//     64-lane gather of 8 bytes and 20.3 of 16, so the pairs took the FP32
//     chain of 500 x 381 x 88 voxels from 17.2 to 12.8 ms and of 256 x 256 x 64
//     from 3.84 to 3.19, bitwise the same volumes; 16-bit row pairs (whole
//     chains) and 2 x 2 quads (stage calls) are one 8-byte load, and are
//     scaled once per scan at the end; FP16 is interpolated across channels
//     by two v_dot2_f32_f16 with the channel weights packed as FP16 (exact
//     products, FP32 sums); lanes that select nothing read whatever the
//     range-checked buffer returns (filtered values of the slab, or 0
//     outside it) and get weight 0 instead of a branch;
//   * the per-theta~ mean uses v_rcp.
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <algorithm>

#include "wave_ops.h"
#include "wfbp_internal.h"

namespace fct {
namespace {

constexpr int kRsrcWord3 = 0x00020000;   // raw buffer, 32-bit data format (gfx9)

// Per (lane, view) bilinear interpolation: fetch() issues the loads of rows
// iq and iq + 1 at channels pf, pf + 1 from the byte offset of (view, iq, pf);
// value() interpolates them across the channels and then between the rows
// with the row fraction fq.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// The filtered projections of a slab as a buffer resource based at the
// slab's first view.
struct BpRsrc {
  __amdgpu_buffer_rsrc_t rows;
};

template <int PREC>
struct ChanInterp;

template <>
struct ChanInterp<FCT_PRECISION_FP32> {   // plain rows: two 8-byte loads
  static constexpr uint32_t kEntry = 4;     // bytes per (row, channel)
  struct Raw {
    u32x2 a, b;
  };
  float wp;
  uint32_t base;   // byte offset of (row 0, pf) in its view; + the view's for fetch()
  __device__ void init(uint32_t pf, float w) {
    wp = w;
    base = pf * kEntry;
  }
  // Row iq + 1 at the vector offset off + rowB: both loads are range-checked
  // (the hardware's check covers the vector offset, not the scalar one), so
  // lanes that select nothing never read past the slab's projections.
  __device__ static Raw fetch(const BpRsrc& r, uint32_t off, uint32_t rowB) {
    return Raw{__builtin_amdgcn_raw_buffer_load_b64(r.rows, (int)off, 0, 0),
               __builtin_amdgcn_raw_buffer_load_b64(r.rows, (int)(off + rowB), 0, 0)};
  }
  __device__ float value(const Raw& t, float fq) const {
    const uint32_t a0 = t.a.x, a1 = t.a.y, b0 = t.b.x, b1 = t.b.y;
    const float fa0 = __uint_as_float(a0), fa1 = __uint_as_float(a1);
    const float fb0 = __uint_as_float(b0), fb1 = __uint_as_float(b1);
    const float r0 = fmaf(wp, fa1 - fa0, fa0), r1 = fmaf(wp, fb1 - fb0, fb0);
    return fmaf(fq, r1 - r0, r0);
  }
};

template <>
struct ChanInterp<kPrecisionPairs> {   // FP32 row pairs: one 16-byte load
  static constexpr uint32_t kEntry = 8;
  typedef u32x4 Raw;
  float wp;
  uint32_t base;
  __device__ void init(uint32_t pf, float w) {
    wp = w;
    base = pf * kEntry;
  }
  // Entries (iq, pf) and (iq, pf + 1).
  __device__ static Raw fetch(const BpRsrc& r, uint32_t off, uint32_t) {
    return __builtin_amdgcn_raw_buffer_load_b128(r.rows, (int)off, 0, 0);
  }
  // The arithmetic of the row layout, term by term.
  __device__ float value(const Raw& t, float fq) const {
    const uint32_t a0 = t.x, b0 = t.y, a1 = t.z, b1 = t.w;
    const float fa0 = __uint_as_float(a0), fa1 = __uint_as_float(a1);
    const float fb0 = __uint_as_float(b0), fb1 = __uint_as_float(b1);
    const float r0 = fmaf(wp, fa1 - fa0, fa0), r1 = fmaf(wp, fb1 - fb0, fb0);
    return fmaf(fq, r1 - r0, r0);
  }
};

// a.lo * b.lo + a.hi * b.hi + c: two FP16 products (exact in FP32) and an
// FP32 sum in one dot instruction.  (Through the builtin, not inline asm: a
// dot result read by another VALU instruction needs wait states that only
// the compiler's hazard recognizer inserts.)
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float dot2_f16(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, a), __builtin_bit_cast(half2_t, b), c,
                                false);
}

template <>
struct ChanInterp<FCT_PRECISION_FP16> {   // quad entries: one 8-byte load
  static constexpr uint32_t kEntry = 8;
  typedef u32x2 Raw;
  // Channel weights (1 - wq, wq) as packed FP16 and their negatives, with
  // wq = fp16_channel_weight(wp): both weights are exact in FP16 and sum to 1
  // (a position error below 2^-12 channel).
  uint32_t w, nw;
  uint32_t base;
  __device__ void init(uint32_t pf, float wp) {
    const float wq = fp16_channel_weight(wp);
    w = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(1.0f - wq, wq));
    nw = w ^ 0x80008000u;
    base = pf * kEntry;
  }
  __device__ static Raw fetch(const BpRsrc& r, uint32_t off, uint32_t) {
    return __builtin_amdgcn_raw_buffer_load_b64(r.rows, (int)off, 0, 0);
  }
  __device__ float value(const Raw& t, float fq) const {
    // -r0 and r1 - r0 from the two rows' FP16 pairs, then r0 + fq (r1 - r0).
    // (Through named scalars: hipcc (ROCm 7.2) folds __builtin_bit_cast of a
    // vector element such as t[1] to element 0.)
    const uint32_t q0 = t.x, q1 = t.y;
    const float nr0 = dot2_f16(q0, nw, 0.0f);
    const float d = dot2_f16(q1, w, nr0);
    return fmaf(fq, d, -nr0);
  }
  // The same for four samples and their sums, num += W value and den += W, as
  // one block of eight v_dot2_f32_f16 in the VOP3P form (the builtin selects
  // the two-address v_dot2c form and copies the accumulator) with the sums
  // updated in place (left to the compiler, the paths of the view loop end in
  // different registers and every view copies all sums at the join).  Every
  // dot result is read at least three instructions after it is written (the
  // wait a dot result needs before another VALU instruction reads it): the
  // second dot of a sample reads the first four instructions later, and the
  // four additions to den follow the last dot.
  __device__ void accumulate4(const Raw* t, const float* fq, const float* W, float* num,
                              float* den) const {
    const uint32_t a0 = t[0].x, a1 = t[1].x, a2 = t[2].x, a3 = t[3].x;
    const uint32_t b0 = t[0].y, b1 = t[1].y, b2 = t[2].y, b3 = t[3].y;
    float n0, n1, n2, n3, d0, d1, d2, d3;
    asm("v_dot2_f32_f16 %0, %16, %24, 0\n\t"
        "v_dot2_f32_f16 %1, %17, %24, 0\n\t"
        "v_dot2_f32_f16 %2, %18, %24, 0\n\t"
        "v_dot2_f32_f16 %3, %19, %24, 0\n\t"
        "v_dot2_f32_f16 %4, %20, %25, %0\n\t"
        "v_dot2_f32_f16 %5, %21, %25, %1\n\t"
        "v_dot2_f32_f16 %6, %22, %25, %2\n\t"
        "v_dot2_f32_f16 %7, %23, %25, %3\n\t"
        "v_add_f32 %12, %12, %30\n\t"
        "v_add_f32 %13, %13, %31\n\t"
        "v_add_f32 %14, %14, %32\n\t"
        "v_add_f32 %15, %15, %33\n\t"
        "v_fma_f32 %4, %26, %4, -%0\n\t"
        "v_fma_f32 %5, %27, %5, -%1\n\t"
        "v_fma_f32 %6, %28, %6, -%2\n\t"
        "v_fma_f32 %7, %29, %7, -%3\n\t"
        "v_fmac_f32 %8, %30, %4\n\t"
        "v_fmac_f32 %9, %31, %5\n\t"
        "v_fmac_f32 %10, %32, %6\n\t"
        "v_fmac_f32 %11, %33, %7"
        : "=&v"(n0), "=&v"(n1), "=&v"(n2), "=&v"(n3), "=&v"(d0), "=&v"(d1), "=&v"(d2),
          "=&v"(d3), "+v"(num[0]), "+v"(num[1]), "+v"(num[2]), "+v"(num[3]), "+v"(den[0]),
          "+v"(den[1]), "+v"(den[2]), "+v"(den[3])
        : "v"(a0), "v"(a1), "v"(a2), "v"(a3), "v"(b0), "v"(b1), "v"(b2), "v"(b3), "v"(nw),
          "v"(w), "v"(fq[0]), "v"(fq[1]), "v"(fq[2]), "v"(fq[3]), "v"(W[0]), "v"(W[1]),
          "v"(W[2]), "v"(W[3]));
  }
};

template <>
struct ChanInterp<FCT_PRECISION_BF16> {   // quad entries: one 8-byte load
  static constexpr uint32_t kEntry = 8;
  typedef u32x2 Raw;
  float wp;
  uint32_t base;
  __device__ void init(uint32_t pf, float w) {
    wp = w;
    base = pf * kEntry;
  }
  __device__ static Raw fetch(const BpRsrc& r, uint32_t off, uint32_t) {
    return __builtin_amdgcn_raw_buffer_load_b64(r.rows, (int)off, 0, 0);
  }
  __device__ float value(const Raw& t, float fq) const {
    const uint32_t q0 = t.x, q1 = t.y;
    const float a0 = __uint_as_float(q0 << 16), a1 = __uint_as_float(q0 & 0xFFFF0000u);
    const float b0 = __uint_as_float(q1 << 16), b1 = __uint_as_float(q1 & 0xFFFF0000u);
    const float r0 = fmaf(wp, a1 - a0, a0), r1 = fmaf(wp, b1 - b0, b0);
    return fmaf(fq, r1 - r0, r0);
  }
};

// 16-bit row pairs: the 8 bytes of entries (iq, pf) and (iq, pf + 1) hold the
// quad's halves in another order (FP16 puts them back for the dot products,
// two instructions per sample).  The gathers cost the same, the lines they
// touch are half as many: 512 x 512 x 320 FP16 46.1 -> 45.5 ms, flying focal
// spot 10.95 -> 10.45, 256 x 256 x 64 BF16 4.28 -> 4.05 (whole chains, bitwise
// the same volumes; six FP16 jobs in one launch 33.0 both).
template <>
struct ChanInterp<kPrecisionPairsF16> : ChanInterp<FCT_PRECISION_FP16> {
  static constexpr uint32_t kEntry = 4;
  __device__ void init(uint32_t pf, float wp) {
    ChanInterp<FCT_PRECISION_FP16>::init(pf, wp);
    base = pf * kEntry;
  }
  __device__ static Raw quad(const Raw& t) {
    const uint32_t x = t.x, y = t.y;
    return Raw{__builtin_amdgcn_perm(y, x, 0x05040100u), __builtin_amdgcn_perm(y, x, 0x07060302u)};
  }
  __device__ float value(const Raw& t, float fq) const {
    return ChanInterp<FCT_PRECISION_FP16>::value(quad(t), fq);
  }
  __device__ void accumulate4(const Raw* t, const float* fq, const float* W, float* num,
                              float* den) const {
    const Raw q[4] = {quad(t[0]), quad(t[1]), quad(t[2]), quad(t[3])};
    ChanInterp<FCT_PRECISION_FP16>::accumulate4(q, fq, W, num, den);
  }
};

template <>
struct ChanInterp<kPrecisionPairsB16> : ChanInterp<FCT_PRECISION_BF16> {
  static constexpr uint32_t kEntry = 4;
  __device__ void init(uint32_t pf, float w) {
    wp = w;
    base = pf * kEntry;
  }
  __device__ float value(const Raw& t, float fq) const {
    const uint32_t q0 = t.x, q1 = t.y;
    const float a0 = __uint_as_float(q0 << 16), b0 = __uint_as_float(q0 & 0xFFFF0000u);
    const float a1 = __uint_as_float(q1 << 16), b1 = __uint_as_float(q1 & 0xFFFF0000u);
    const float r0 = fmaf(wp, a1 - a0, a0), r1 = fmaf(wp, b1 - b0, b0);
    return fmaf(fq, r1 - r0, r0);
  }
};

template <int PREC>
constexpr bool kF16 = PREC == FCT_PRECISION_FP16 || PREC == kPrecisionPairsF16;
template <int PREC>
constexpr bool kRowPairs = PREC >= kPrecisionPairs;   // (whole chains and the matched sum only)

// Per (voxel column, theta~): p, sqrt(R^2 - p^2), the in-plane offset f and
// the cone-angle z term kb (fct_bp_column for the views of both parities,
// which share p, sqrt and asin).
struct BpColumn {
  float p, sq, f, kb;
};

__device__ __forceinline__ BpColumn bp_column(float x, float y, float2 cs, const FctBpConsts& g) {
  BpColumn c;
  c.p = fmaf(x, cs.y, -(y * cs.x));
  c.sq = sqrt_rn_large(fmaf(-c.p, c.p, g.R2));
  c.f = fmaf(x, cs.x, y * cs.y);
  c.kb = g.kappa * fct_asinf(c.p * g.invR);
  return c;
}

// z-interval of |q| <= 1 relative to a view's table z for the voxels of a
// wave's tile in the FOV: [min(-kbs - lt), max(-kbs + lt)] with kbs = kb,
// lt = (sq - f) tan for parity 0 and kbs = -kb, lt = (sq + f) tan for parity
// 1, returned as (min, max, min, max).  It depends on the tile and theta~
// only, so bp_zbounds_kernel tabulates it once per plan.
__device__ __forceinline__ float4 tile_zbounds(const BpColumn& c, bool active,
                                               const FctBpConsts& g) {
  const float BIG = 3.0e38f;
  const float lt0 = (c.sq - c.f) * g.tanc, lt1 = (c.sq + c.f) * g.tanc;
  float4 r;
  r.x = wave_min(active ? -c.kb - lt0 : BIG);
  r.y = wave_max(active ? -c.kb + lt0 : -BIG);
  r.z = wave_min(active ? c.kb - lt1 : BIG);
  r.w = wave_max(active ? c.kb + lt1 : -BIG);
  return r;
}

// One wave per tile (all 64 lanes active, as the reductions need).
__global__ __launch_bounds__(64) void bp_zbounds_kernel(BpArgs a, float4* out) {
  const int tile = blockIdx.x;
  const int lane = threadIdx.x;
  const int tx = tile % a.tiles_x, ty = tile / a.tiles_x;
  const int ix = tx * 8 + (lane & 7), iy = ty * 8 + (lane >> 3);
  const bool inb = ix < a.nx && iy < a.ny;
  const float x = inb ? a.xs[ix] : 0.0f;
  const float y = inb ? a.ys[iy] : 0.0f;
  const bool active = inb && fct_in_fov(x, y, a.g);
  for (int t = 0; t < a.H; ++t) {
    const float4 r = tile_zbounds(bp_column(x, y, a.cs[t], a.g), active, a.g);
    if (lane == 0) out[(size_t)tile * a.H + t] = r;
  }
}

// One (voxel, view, slice) sample in two steps: bp_fetch computes the row
// position and the exact selection and issues the tap loads; bp_add
// interpolates and accumulates into (num, den) or cnt.  Branch-free: lanes
// that select nothing read whatever the range-checked buffer returns at their
// offset and get weight 0.
template <int PREC>
struct BpTap {
  float qi, fq;   // row position and its fraction qi - floor(qi)
  bool sel;
  typename ChanInterp<PREC>::Raw raw;
};

template <int PREC, int MODE, bool CENTERED>
__device__ __forceinline__ BpTap<PREC> bp_fetch(float zsi, float invLh, float row0,
                                                const ChanInterp<PREC>& ci,
                                                const BpRsrc& rf, uint32_t rowB,
                                                bool chan_ok, const FctBpConsts& g) {
  BpTap<PREC> s;
  s.qi = fmaf(zsi, invLh, row0);   // fct_bp_row
  const int iq = floor_int(s.qi);
  // qi - floor(qi), exact for qi >= 0 (the selected rows); v_fract clamps
  // below 1 where that difference would round up, which only happens for
  // tiny negative qi (not selected).
  s.fq = __builtin_amdgcn_fractf(s.qi);
  if (CENTERED)   // |q| <= 1 is implied by the row test when cr = hr
    s.sel = chan_ok && (uint32_t)iq <= (uint32_t)(g.nrows - 2);
  else
    s.sel = chan_ok && !(fabsf(s.qi - g.cr) > g.hr) && iq >= 0 && iq <= g.nrows - 2;
  // 24-bit multiply: exact for selected rows (< 2^24).
  if (MODE != kBpCount)
    s.raw = ChanInterp<PREC>::fetch(rf, ci.base + __umul24((uint32_t)iq, rowB), rowB);
  return s;
}

// Weight of a sample (0 when it is not selected): W(q) for the WFBP sum,
// R / l for the matched projector's plain sum over the views.
//
// FREE (centred rows, cr == hr, WFBP sum): no selection mask.  The ramp
// argument t is clamped to [0, 1] by the fma's clamp modifier; the rows a
// sample may use, qi in [0, nrows - 1), are those with |qi - cr| < hr, and
// every other qi has |qi - cr| >= hr, where t <= 0 exactly (wk is rounded
// up), so W = 0 without a compare and a select.  Lanes whose column misses
// the detector or the FOV enter with row0 = -1e30 and rows per mm 0 (the
// caller's view setup): t = 0 for them too.  Their tap offsets stay inside
// the slab (the 24-bit row product of floor(-1e30) is 0) and the taps they
// read are finite, so num gains 0 * value = 0.
template <int PREC, int MODE, bool FREE = false>
__device__ __forceinline__ float bp_weight(const BpTap<PREC>& s, float fR, const FctBpConsts& g) {
  if (MODE == kBpMatched) return s.sel ? fR : 0.0f;
  if (FREE)
    return fct_w_of_t(
        __builtin_amdgcn_fmed3f(fmaf(-fabsf(s.qi - g.cr), g.wk, FCT_WC), 0.0f, 1.0f));
  const float w = fct_w_of_row(s.qi, g);
  return s.sel ? w : 0.0f;
}

// Accumulation of a sample of weight W (bp_weight) and interpolated value
// val, in place (see accumulate4).
template <int MODE>
__device__ __forceinline__ void bp_acc(float W, float val, float& num, float& den) {
  asm("v_fmac_f32 %0, %1, %2" : "+v"(num) : "v"(W), "v"(val));
  if (MODE != kBpMatched) asm("v_add_f32 %0, %0, %1" : "+v"(den) : "v"(W));
}

template <int PREC, int MODE, bool FREE = false>
__device__ __forceinline__ void bp_add(const BpTap<PREC>& s, const ChanInterp<PREC>& ci, float fR,
                                       const FctBpConsts& g, float& num, float& den, int& cnt) {
  if (MODE == kBpCount) {
    cnt += s.sel ? 1 : 0;
    return;
  }
  bp_acc<MODE>(bp_weight<PREC, MODE, FREE>(s, fR, g), ci.value(s.raw, s.fq), num, den);
}

// Four samples of one view: FP16 through the dot block.
template <int PREC, int MODE, bool FREE = false>
__device__ __forceinline__ void bp_add4(const BpTap<PREC>* s, const ChanInterp<PREC>& ci,
                                        float fR, const FctBpConsts& g, float* num, float* den,
                                        int* cnt) {
  if constexpr (kF16<PREC> && MODE != kBpCount) {
    // The weights first: their arithmetic overlaps the tap loads.
    typename ChanInterp<PREC>::Raw t[4];
    float fq[4], W[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      t[i] = s[i].raw;
      fq[i] = s[i].fq;
      W[i] = bp_weight<PREC, MODE, FREE>(s[i], fR, g);
    }
    ci.accumulate4(t, fq, W, num, den);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      bp_add<PREC, MODE, FREE>(s[i], ci, fR, g, num[i], den[i], cnt[i]);
  }
}

// How the theta~ of a tile are summed: in one sweep; in a.nseg consecutive
// segments by as many waves of a workgroup (their sums added in segment
// order through LDS); or in the same segments one after the other by one
// wave (the persistent kernel), which gives bitwise the same volume.
enum BpSplit { kSweep = 0, kSplitWaves = 1, kSplitSerial = 2 };

// One wave reconstructs tile `lin` (slab-major order) of the job described by
// a; with kSplitWaves its theta~ segment `wave`.  The sums over theta~ live in
// lds, TZ x 64 floats per wave (kSplitSerial 2 TZ x 64): read, added to and
// written once per theta~, they would cost registers the view loops need.
template <int TZ, int PREC, int MODE, bool CENTERED, int SPLIT>
__device__ __forceinline__ void bp_v1_tile(const BpArgs& a, int lin, int wave, float* lds) {
  constexpr uint32_t kEntry = ChanInterp<PREC>::kEntry;
  const int lane = threadIdx.x & 63;
  const int tiles = a.tiles_x * a.tiles_y;
  const int slab = lin / tiles;
  const int2 txy = tile_of(lin - slab * tiles, a.tiles_x, a.tiles_y);
  const int tx = txy.x, ty = txy.y;
  const int tile = ty * a.tiles_x + tx;
  const int ix = tx * 8 + (lane & 7), iy = ty * 8 + (lane >> 3);
  const bool inb = ix < a.nx && iy < a.ny;
  const float x = inb ? a.xs[ix] : 0.0f;
  const float y = inb ? a.ys[iy] : 0.0f;
  const FctBpConsts& g = a.g;
  const bool active = inb && fct_in_fov(x, y, g);
  const int s0 = slab * TZ;
  const int nz = min(TZ, a.n_native - s0);
  if (!__any(active)) {
    if (inb && wave == 0)
      for (int i = 0; i < nz; ++i) {
        const size_t o = ((size_t)(s0 + i) * a.ny + iy) * a.nx + ix;
        if (MODE == kBpAccumulate || MODE == kBpMatched) a.native[o] = 0.0f;
        if (MODE == kBpCount) a.counts[o] = 0;
      }
    return;
  }
  const int chunk = s0 / fct_tables::kSliceChunk;
  float zs[TZ];
#pragma unroll
  for (int i = 0; i < TZ; ++i) zs[i] = ld_uniform(a.zs + s0 + (i < nz ? i : nz - 1));
  // Slice spacing inside the slab (uniform, FP32; used only for skipping).
  const float zfirst = zs[0], zlast = ld_uniform(a.zs + s0 + nz - 1);
  const float dzs = nz > 1 ? (zlast - zfirst) / (float)(nz - 1) : 1.0f;
  const float inv_dzs = 1.0f / dzs, ninv_dzs = -inv_dzs;
  // Centred WFBP sums: the whole-slab samples take their weight without a
  // selection mask (bp_weight), the lanes whose column misses the detector
  // parked at row -1e30 with 0 rows per mm (the per-slice masks of the
  // partial-slab paths already exclude those lanes).
  constexpr bool kFree = CENTERED && MODE == kBpAccumulate;
  const float* ztc = a.zt + (size_t)chunk * a.nviews;
  const int* wrc = reinterpret_cast<const int*>(a.wrange + (size_t)chunk * a.nviews);
  const float half_feed = g.kappa * 3.14159265f, z_inside = g.zrot - 0.5f * fabsf(dzs);
  const int* vrp = reinterpret_cast<const int*>(a.slab_vrange + slab);
  const int2 vr = make_int2(ld_uniform(vrp), ld_uniform(vrp + 1));
  const int H = a.H;
  // The views of theta~ t are t + k H, k in [qx + (t < rx), qy + (t < ry)).
  const int qx = vr.x / H, rx = vr.x - qx * H, qy = vr.y / H, ry = vr.y - qy * H;
  const uint32_t vstride = (uint32_t)g.nrows * (uint32_t)a.cpitch;   // entries per view
  const uint32_t rowB = (uint32_t)a.cpitch * kEntry;                 // bytes per row

  // Buffer resource based at the slab's first view (keeps offsets < 4 GiB;
  // the planner checks that a slab's views fit).
  const char* fb = static_cast<const char*>(a.filt) + (size_t)vr.x * vstride * kEntry;
  const uint32_t fbytes =
      (uint32_t)min((size_t)(vr.y - vr.x) * vstride * kEntry, (size_t)0xFFFFFFF0u);
  BpRsrc rf;
  rf.rows = __builtin_amdgcn_make_buffer_rsrc((void*)fb, 0, fbytes, kRsrcWord3);

  float* acc = lds + lane;   // slice i at acc[i * 64]
  int cnt[TZ];
  int seg = SPLIT == kSplitWaves ? wave : 0;
  do {
#pragma unroll
    for (int i = 0; i < TZ; ++i) {
      if (MODE != kBpCount) acc[i * 64] = 0.0f;
      cnt[i] = 0;
    }
    const int t0 = SPLIT == kSweep ? 0 : H * seg / a.nseg;
    const int t1 = SPLIT == kSweep ? H : H * (seg + 1) / a.nseg;
    for (int t = t0; t < t1; ++t) {
      const int kmin = qx + (t < rx ? 1 : 0), kmax = qy + (t < ry ? 1 : 0);
      if (kmin >= kmax) continue;
      const float* csp = reinterpret_cast<const float*>(a.cs + t);
      const float2 cs = make_float2(ld_uniform(csp), ld_uniform(csp + 1));
      const BpColumn col = bp_column(x, y, cs, g);
      // The tile's z-interval extremes for this theta~ (tabulated per plan).
      const float4 zb = ld_uniform4(a.zbounds + (size_t)tile * H + t);
      float num[TZ], den[TZ];
#pragma unroll
      for (int i = 0; i < TZ; ++i) {
        // 1e-30 is below half an ulp of any nonzero weight sum (W >= ~1e-13
        // when a sample is selected), so den ends as the exact sum when a
        // view contributes and 1e-30 (num = 0, no change to acc) otherwise.
        // (Through an empty asm: as literals the compiler materialised both
        // start values again at the view loop's entry, 32 instead of 14 moves
        // per theta~.)
        float zero = 0.0f, tiny = 1e-30f;
        asm("" : "+v"(zero));
        asm("" : "+v"(tiny));
        num[i] = zero;
        den[i] = tiny;
      }
      for (int kb = kmin; kb < kmax; kb += 64) {   // (rarely more than one pass)
        // Lane l looks at view kb + l: its slice range [ilo, ihi] inside the
        // slab, from the z-interval of |q| <= 1 over the tile (z relative to
        // the view's table z; one slice of margin on each side covers the
        // rounding, the per-sample test is exact).  The views of a theta~ are
        // half a feed apart.  The view window ends none of the slices of a
        // view whose slices lie at least half a slice inside it; for the
        // others (near) the exact table applies.  (The matched projector pair
        // uses every view that sees the voxel: no view window.)
        const int kl = kb + lane;
        const float zl = fmaf((float)lane, half_feed, ld_uniform(ztc + t + kb * H));
        const bool odd = kl & 1;
        const float A = odd ? zb.z : zb.x, B = odd ? zb.w : zb.y;
        const float ca = (A - zfirst) * inv_dzs, cb = (B - zfirst) * inv_dzs;
        const int flo = floor_int(fmaf(zl, inv_dzs, inv_dzs > 0.0f ? ca : cb));
        const int fhi = floor_int(fmaf(zl, ninv_dzs, inv_dzs > 0.0f ? -cb : -ca));   // -ceil
        const int ilo_l = max(0, flo - 1), ihi_l = min(nz - 1, 1 - fhi);
        const bool some = kl < kmax && ilo_l <= ihi_l;
        const float zrel = zl - zfirst;
        const bool near =
            MODE != kBpMatched && some &&
            fmaxf(fabsf(fmaf((float)-ilo_l, dzs, zrel)), fabsf(fmaf((float)-ihi_l, dzs, zrel))) >
                z_inside;
        const uint64_t m_some = __builtin_amdgcn_ballot_w64(some);
        const uint64_t m_near = __builtin_amdgcn_ballot_w64(near);
        const uint64_t m_whole =
            __builtin_amdgcn_ballot_w64(some && !near && ilo_l == 0 && ihi_l == nz - 1);
#pragma unroll
        for (int par = 0; par < 2; ++par) {
          const uint64_t m_par = (kb & 1) == par ? 0x5555555555555555ull : 0xAAAAAAAAAAAAAAAAull;
          uint64_t whole = m_whole & m_par, part = m_some & ~m_whole & m_par;
          if (!(whole | part)) continue;
          const float pidx = par ? fmaf(-col.p, g.inv_ds, g.cc) : fmaf(col.p, g.inv_ds, g.cc);
          const float lt = (par ? col.sq + col.f : col.sq - col.f) * g.tanc;
          const float kbs = par ? -col.kb : col.kb;
          const float pfl = floorf(pidx);
          const bool chan_ok = active && pfl >= 0.0f && pfl <= (float)(g.ncols - 2);
          // Rows per mm of z; 0 for the lanes parked off the detector (kFree).
          const float invLh = kFree && !chan_ok ? 0.0f : div_rn_normal(g.hr, lt);
          ChanInterp<PREC> ci;
          ci.init(chan_ok ? (uint32_t)(int)pfl : 0u, pidx - pfl);
          // Matched mode: R / l, the voxel-driven footprint's depth correction
          // (a row spans drow l / Dsd of z at distance l from the source).
          const float fR = MODE == kBpMatched ? g.tanc / (lt * g.invR) : 0.0f;
          const uint32_t base = ci.base;
          auto view = [&](int l, float ztv, float* row0) {
            *row0 = kFree && !chan_ok ? -1.0e30f : fmaf(kbs - ztv, invLh, g.cr);   // fct_bp_row0
            ci.base = base + (uint32_t)(t + (kb + l) * H - vr.x) * vstride * kEntry;
          };
          // The view's table z is loaded one view ahead.
          auto ahead = [&](uint64_t m) {
            return ld_uniform(ztc + t + (kb + (m ? __builtin_ctzll(m) : 0)) * H);
          };
          float zt_next = ahead(whole);
          while (whole) {
            // Every slice of the slab (the common case): no per-slice branch,
            // and the taps of four slices are in flight before the first is
            // used (four, not TZ: more would cost waves per SIMD).  With
            // nz < TZ the extra slices repeat the last one and are not stored.
            // Centred WFBP sums take the weight without a selection mask
            // (bp_weight; the lanes off the detector are parked at row -1e30).
            const int l = __builtin_ctzll(whole);
            whole &= whole - 1;
            const float ztv = zt_next;
            zt_next = ahead(whole);
            float row0;
            view(l, ztv, &row0);
#pragma unroll
            for (int h = 0; h < TZ; h += 4) {
              BpTap<PREC> tap[4];
#pragma unroll
              for (int i = 0; i < 4; ++i)
                tap[i] = bp_fetch<PREC, MODE, CENTERED>(zs[h + i], invLh, row0, ci, rf, rowB,
                                                        chan_ok, g);
              // FP16: the four loads are issued before the weight arithmetic
              // that waits for them (the scheduler would sink them otherwise).
              if (kF16<PREC>) __builtin_amdgcn_sched_barrier(0);
              bp_add4<PREC, MODE, kFree>(tap, ci, fR, g, num + h, den + h, cnt + h);
            }
          }
          while (part) {
            const int l = __builtin_ctzll(part);
            part &= part - 1;
            int ilo = __builtin_amdgcn_readlane(ilo_l, l);
            int ihi = __builtin_amdgcn_readlane(ihi_l, l);
            const int v = t + (kb + l) * H;
            const float ztv = ld_uniform(ztc + v);
            if (m_near >> l & 1) {   // the window's exact slice range
              ilo = max(ilo, ld_uniform(wrc + 2 * v) - s0);
              ihi = min(ihi, ld_uniform(wrc + 2 * v + 1) - s0);
              if (ilo > ihi) continue;
            }
            float row0;
            view(l, ztv, &row0);
            if constexpr (kF16<PREC>) {
              // Part of the slab, FP16: groups of four slices that meet
              // [ilo, ihi] through the dot block, the slices outside the range
              // masked like unselected samples (cheaper than per-slice samples
              // with the two-address dot form; for FP32 / BF16 the masked slices
              // cost more than they save).
#pragma unroll
              for (int h = 0; h < TZ; h += 4) {
                if (ilo > h + 3 || ihi < h) continue;
                BpTap<PREC> tap[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                  tap[i] = bp_fetch<PREC, MODE, CENTERED>(
                      zs[h + i], invLh, row0, ci, rf, rowB,
                      chan_ok && h + i >= ilo && h + i <= ihi, g);
                __builtin_amdgcn_sched_barrier(0);
                bp_add4<PREC, MODE>(tap, ci, fR, g, num + h, den + h, cnt + h);
              }
            } else {
#pragma unroll
              for (int i = 0; i < TZ; ++i)
                if (i >= ilo && i <= ihi) {
                  const BpTap<PREC> tp = bp_fetch<PREC, MODE, CENTERED>(zs[i], invLh, row0, ci, rf,
                                                                        rowB, chan_ok, g);
                  bp_add<PREC, MODE>(tp, ci, fR, g, num[i], den[i], cnt[i]);
                }
            }
          }
        }
      }
      if (MODE == kBpAccumulate) {
#pragma unroll
        for (int i = 0; i < TZ; ++i)
          acc[i * 64] = fmaf(num[i], __builtin_amdgcn_rcpf(den[i]), acc[i * 64]);
      } else if (MODE == kBpMatched) {
#pragma unroll
        for (int i = 0; i < TZ; ++i) acc[i * 64] += num[i];
      }
    }
    if (SPLIT == kSplitSerial && a.nseg > 1) {
#pragma unroll
      for (int i = 0; i < TZ; ++i) {
        if (seg > 0) acc[i * 64] += acc[(TZ + i) * 64];
        acc[(TZ + i) * 64] = acc[i * 64];
      }
    }
  } while (SPLIT == kSplitSerial && ++seg < a.nseg);
  if (SPLIT == kSplitWaves) __syncthreads();
  if (!inb) return;
  if (MODE == kBpAccumulate || MODE == kBpMatched) {
    // FP16 / BF16 projections carry one storage scale per scan.
    const float out_scale =
        PREC == FCT_PRECISION_FP32 || PREC == kPrecisionPairs
            ? a.scale
            : a.scale * ld_uniform(a.filt_scale);
    // The segments' waves share the slices out; each sums the segments of its
    // slices in order.
    const int nw = SPLIT == kSplitWaves ? a.nseg : 1;
    const float* part = lds + lane - (SPLIT == kSplitWaves ? wave * TZ * 64 : 0);
    for (int i = SPLIT == kSplitWaves ? wave : 0; i < nz; i += nw) {
      float sum = part[i * 64];
      for (int w = 1; w < nw; ++w) sum += part[(w * TZ + i) * 64];
      a.native[((size_t)(s0 + i) * a.ny + iy) * a.nx + ix] =
          sum * out_scale;
    }
  } else if (MODE == kBpCount) {
    unsigned long long tot = 0;
#pragma unroll
    for (int i = 0; i < TZ; ++i)
      if (i < nz) {
        a.counts[((size_t)(s0 + i) * a.ny + iy) * a.nx + ix] = cnt[i];
        tot += (unsigned long long)cnt[i];
      }
    if (tot) atomicAdd(a.total, tot);
  }
}

// The tile of a launch block: block b runs on XCD b mod 8 and takes the next
// tile of that XCD's share (BpArgs::xcd_first); -1 past its end.
__device__ __forceinline__ int bp_launch_tile(const BpArgs& a) {
  const int x = blockIdx.x & 7, lin = a.xcd_first[x] + (int)(blockIdx.x >> 3);
  return lin < a.xcd_first[x + 1] ? lin : -1;
}

// Occupancy floor at TZ <= 8: at least seven waves per SIMD (72 VGPRs; only
// the persistent FP32 kernel spills, five in the per-theta~ set-up; eight
// spill in every kernel but BF16).  At TZ = 16 five: left to itself the
// allocator takes 97 VGPRs for FP16 and 114 for FP32 row pairs, whose chain
// of 500 x 381 x 88 then takes 20.6 instead of 16.0 ms.
template <int TZ, int PREC>
constexpr int bp_min_waves() {
  return TZ <= 8 ? 7 : TZ == 16 ? 5 : 1;
}

template <int TZ, int PREC, int MODE, bool CENTERED>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(TZ >= 8 ? bp_min_waves<TZ, PREC>() : 1, 8)))
void bp_v1_kernel(BpArgs a) {
  __shared__ float bp_lds[MODE == kBpCount ? 1 : TZ * 64];
  const int lin = bp_launch_tile(a);
  if (lin < 0) return;
  bp_v1_tile<TZ, PREC, MODE, CENTERED, kSweep>(a, lin, 0, bp_lds);
}

// A workgroup of a.nseg waves per tile.
template <int TZ, int PREC, int MODE, bool CENTERED>
__global__ __launch_bounds__(64 * (TZ > 16 ? 256 / TZ : kBpMaxSegments))
__attribute__((amdgpu_waves_per_eu(TZ >= 8 ? bp_min_waves<TZ, PREC>() : 1, 8)))
void bp_v1_split_kernel(BpArgs a) {
  extern __shared__ float bp_lds[];
  const int lin = bp_launch_tile(a);
  if (lin < 0) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  bp_v1_tile<TZ, PREC, MODE, CENTERED, kSplitWaves>(
      a, lin, wave, bp_lds + wave * TZ * 64);
}

// Persistent backprojection of many jobs in one launch.  The tiles of all
// jobs form one list (job-major, slab-major inside a job) split into eight
// contiguous ranges, one per XCD (workgroup b runs on XCD b mod 8), so that
// neighbouring tiles -- which read the same projection rows -- share an L2.
// A wave takes the next tile of its XCD's range with one atomic and moves on
// to the other ranges when its own is exhausted; every wave exits once all
// eight counters have passed their range ends.  A tile is computed by the
// same code as in bp_v1_kernel, so each job's volume is bitwise identical to
// its own single-job launch with the same tile_z.
// (The occupancy floors of bp_v1_kernel, also at TZ = 4.)
template <int TZ, int PREC, bool CENTERED>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(bp_min_waves<TZ, PREC>(), 8)))
void bp_batch_kernel(BpBatchArgs b,
                                                      const BpArgs* __restrict__ jobs,
                                                      const int32_t* __restrict__ tile_start) {
  __shared__ float lds[2 * TZ * 64];
  const int xcd = blockIdx.x & 7;
  for (int step = 0; step < 8; ++step) {
    const int r = (xcd + step) & 7;
    const int lo = (int)(((long long)b.total_tiles * r) >> 3);
    const int hi = (int)(((long long)b.total_tiles * (r + 1)) >> 3);
    while (true) {
      uint32_t got = 0;
      if (threadIdx.x == 0) got = atomicAdd(&b.queue[r], 1u);
      const int tile = lo + (int)__builtin_amdgcn_readfirstlane(__shfl(got, 0, 64));
      if (tile >= hi) break;
      int j = 0;   // job: last j with tile_start[j] <= tile
      for (int span = 32; span > 0; span >>= 1)
        if (j + span < b.n_jobs && ld_uniform(tile_start + j + span) <= tile) j += span;
      bp_v1_tile<TZ, PREC, kBpAccumulate, CENTERED, kSplitSerial>(
          jobs[j], tile - ld_uniform(tile_start + j), 0, lds);
    }
  }
}

template <int TZ, int PREC, bool C>
hipError_t launch3(const BpArgs& a, int mode, hipStream_t s) {
  int share = 0;
  for (int x = 0; x < 8; ++x) share = std::max(share, a.xcd_first[x + 1] - a.xcd_first[x]);
  const int blocks = 8 * share;
  if (a.nseg > 1 && mode == kBpAccumulate) {
    hipLaunchKernelGGL((bp_v1_split_kernel<TZ, PREC, kBpAccumulate, C>), dim3(blocks),
                       dim3(64 * a.nseg), a.nseg * TZ * 64 * sizeof(float), s, a);
    return hipGetLastError();
  }
  if constexpr (PREC == FCT_PRECISION_FP32 || PREC == kPrecisionPairs) {
    if (a.nseg > 1 && mode == kBpMatched) {
      hipLaunchKernelGGL((bp_v1_split_kernel<TZ, PREC, kBpMatched, C>), dim3(blocks),
                         dim3(64 * a.nseg), a.nseg * TZ * 64 * sizeof(float), s, a);
      return hipGetLastError();
    }
  }
  if (mode == kBpAccumulate)
    hipLaunchKernelGGL((bp_v1_kernel<TZ, PREC, kBpAccumulate, C>), dim3(blocks), dim3(64), 0, s, a);
  else if (mode == kBpCount && !kRowPairs<PREC>)
    hipLaunchKernelGGL((bp_v1_kernel<TZ, kRowPairs<PREC> ? FCT_PRECISION_FP32 : PREC, kBpCount, C>), dim3(blocks), dim3(64), 0, s, a);
  else if (mode == kBpMatched && (PREC == FCT_PRECISION_FP32 || PREC == kPrecisionPairs))
    hipLaunchKernelGGL((bp_v1_kernel<TZ, PREC == kPrecisionPairs ? kPrecisionPairs : FCT_PRECISION_FP32, kBpMatched, C>), dim3(blocks), dim3(64), 0, s, a);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

template <int TZ, int PREC>
hipError_t launch2(const BpArgs& a, int mode, hipStream_t s) {
  const bool centered = a.g.cr == a.g.hr;
  return centered ? launch3<TZ, PREC, true>(a, mode, s) : launch3<TZ, PREC, false>(a, mode, s);
}

template <int TZ>
hipError_t launch1(const BpArgs& a, int precision, int mode, hipStream_t s) {
  switch (precision) {
    case FCT_PRECISION_FP32: return launch2<TZ, FCT_PRECISION_FP32>(a, mode, s);
    case FCT_PRECISION_FP16: return launch2<TZ, FCT_PRECISION_FP16>(a, mode, s);
    case FCT_PRECISION_BF16: return launch2<TZ, FCT_PRECISION_BF16>(a, mode, s);
    case kPrecisionPairs: return launch2<TZ, kPrecisionPairs>(a, mode, s);
    case kPrecisionPairsF16: return launch2<TZ, kPrecisionPairsF16>(a, mode, s);
    case kPrecisionPairsB16: return launch2<TZ, kPrecisionPairsB16>(a, mode, s);
  }
  return hipErrorInvalidValue;
}

template <int TZ, int PREC>
hipError_t launch_batch2(const BpBatchArgs& b, bool centered, int grid, hipStream_t s) {
  if (centered)
    hipLaunchKernelGGL((bp_batch_kernel<TZ, PREC, true>), dim3(grid), dim3(64), 0, s, b, b.jobs,
                       b.tile_start);
  else
    hipLaunchKernelGGL((bp_batch_kernel<TZ, PREC, false>), dim3(grid), dim3(64), 0, s, b, b.jobs,
                       b.tile_start);
  return hipGetLastError();
}

template <int TZ>
hipError_t launch_batch1(const BpBatchArgs& b, int precision, bool centered, int grid,
                         hipStream_t s) {
  switch (precision) {
    case FCT_PRECISION_FP32: return launch_batch2<TZ, FCT_PRECISION_FP32>(b, centered, grid, s);
    case FCT_PRECISION_FP16: return launch_batch2<TZ, FCT_PRECISION_FP16>(b, centered, grid, s);
    case FCT_PRECISION_BF16: return launch_batch2<TZ, FCT_PRECISION_BF16>(b, centered, grid, s);
    case kPrecisionPairs: return launch_batch2<TZ, kPrecisionPairs>(b, centered, grid, s);
    case kPrecisionPairsF16: return launch_batch2<TZ, kPrecisionPairsF16>(b, centered, grid, s);
    case kPrecisionPairsB16: return launch_batch2<TZ, kPrecisionPairsB16>(b, centered, grid, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_backproject_batch(const BpBatchArgs& b, int tile_z, int precision,
                                    bool centered, int grid, hipStream_t s) {
  if (b.n_jobs < 1 || b.n_jobs > 64 || grid < 8 || (grid & 7)) return hipErrorInvalidValue;
  switch (tile_z) {
    case 4: return launch_batch1<4>(b, precision, centered, grid, s);
    case 8: return launch_batch1<8>(b, precision, centered, grid, s);
    case 16: return launch_batch1<16>(b, precision, centered, grid, s);
    case 32: return launch_batch1<32>(b, precision, centered, grid, s);
  }
  return hipErrorInvalidValue;
}

hipError_t backproject_batch_waves_per_cu(int tile_z, int precision, int* waves) {
  // Occupancy of the FP32 / FP16 / BF16 instantiations (the centred and
  // general forms use the same registers to within a few).
  const void* f = nullptr;
#define FCT_BATCH_K(TZ)                                                                       \
  case TZ: {                                                                                  \
    const void* k[] = {(const void*)bp_batch_kernel<TZ, FCT_PRECISION_FP32, false>,           \
                       (const void*)bp_batch_kernel<TZ, FCT_PRECISION_FP16, false>,           \
                       (const void*)bp_batch_kernel<TZ, FCT_PRECISION_BF16, false>,           \
                       (const void*)bp_batch_kernel<TZ, kPrecisionPairs, false>,              \
                       (const void*)bp_batch_kernel<TZ, kPrecisionPairsF16, false>,           \
                       (const void*)bp_batch_kernel<TZ, kPrecisionPairsB16, false>};          \
    if (precision < 0 || precision > kPrecisionPairsB16) return hipErrorInvalidValue;         \
    f = k[precision];                                                                         \
    break;                                                                                    \
  }
  switch (tile_z) {
    FCT_BATCH_K(4)
    FCT_BATCH_K(8)
    FCT_BATCH_K(16)
    FCT_BATCH_K(32)
    default: return hipErrorInvalidValue;
  }
#undef FCT_BATCH_K
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(waves, f, 64, 0);
}

hipError_t launch_bp_zbounds(const BpArgs& a, float4* zbounds, hipStream_t s) {
  const int tiles = a.tiles_x * a.tiles_y;
  if (tiles <= 0 || a.H <= 0) return hipSuccess;
  hipLaunchKernelGGL(bp_zbounds_kernel, dim3(tiles), dim3(64), 0, s, a, zbounds);
  return hipGetLastError();
}

hipError_t launch_backproject_v1(const BpArgs& a, int tile_z, int precision, int mode,
                                 hipStream_t s) {
  // Slabs [slab0, slab0 + slab_count) inside the volume (slab_count 0: every slab).
  if (a.slab0 < 0 || a.slab_count < 0 || (a.slab_count == 0 && a.slab0 != 0) ||
      a.slab0 + a.slab_count > a.nslabs)
    return hipErrorInvalidValue;
  // The XCDs' shares are those of this range (bp_share).
  const int tiles = a.tiles_x * a.tiles_y;
  if (a.xcd_first[0] != a.slab0 * tiles ||
      a.xcd_first[8] != (a.slab0 + (a.slab_count ? a.slab_count : a.nslabs)) * tiles)
    return hipErrorInvalidValue;
  switch (tile_z) {
    case 4: return launch1<4>(a, precision, mode, s);
    case 8: return launch1<8>(a, precision, mode, s);
    case 16: return launch1<16>(a, precision, mode, s);
    case 32: return launch1<32>(a, precision, mode, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace fct
