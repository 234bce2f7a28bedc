// wfbp_internal.h -- plan layout and kernel launcher interface (not exported).
#pragma once

#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "../../include/fct_wfbp_gpu.h"
#include "chain_buffers.h"
#include "ffs_geometry.h"
#include "wfbp_math.h"

namespace fct {

// Device-side rebinning entry per parallel channel and effective-row parity
// (FP32 weights from the FP64 recipes of wfbp_math.h / ffs_geometry.h).
// state: 0 = no fan sample (output 0), else 1 + the focal state rho; the
// state's projection m = j + aoff (+1) is clamped to [0, mmax] and read at
// raw view m * states + rho.
struct RebinDev {
  int32_t b0, b1, aoff, state;
  float fb, fa;
  int32_t mmax;   // >= 0 (0 for entries without a fan sample)
  uint32_t boff;  // byte offset of (focal state, raw row 0, fan channel b0) in a view group
};

// Filtered projections in HBM.
//  * FP32: plain rows, [view][row][cpitch] floats.
//  * FP16 / BF16: bilinear "quad" entries, [view][row][cpitch][4] 16-bit
//    values, entry (r, c) = (y[r][c], y[r][c+1], y[r+1][c], y[r+1][c+1]) / s,
//    so that one 8-byte load fetches the 2 x 2 footprint of a sample.  Slots
//    beyond the detector (c + 1 = cpitch, r + 1 = nrows) hold 0.  s is one
//    power of two per scan, chosen from a bound on |y| so that |y| / s < 2^15
//    (no overflow); it is kept in scale[0] of the scan's scale buffer.
// [0] s, [1] max |raw| bits (rebin+filter scratch), [2] rescale factor of the
// streaming reconstruction, [3] the s its backprojections read.
constexpr int kScaleElems = 4;

// Channel weight of the FP16 tap interpolation: the fraction wp rounded to a
// multiple of 2^-11, so that it and 1 - it are exact FP16 values summing to 1
// (the backprojection multiplies the FP16 taps by them in v_dot2_f32_f16).
__device__ __forceinline__ float fp16_channel_weight(float wp) {
  return __builtin_rintf(wp * 2048.0f) * (1.0f / 2048.0f);
}

// The rebinning table by the raw channel it reads: parallel channel c (low 16
// bits) and effective-row parity (high), view offset, and the weights of the
// second view and of this raw channel.
struct RebinTDev {
  int32_t c, aoff;
  float fa, wb;
};

// Everything the rebin + filter kernel reads.
struct RebinFilterArgs {
  const float* raw;          // [view][row][ncols]
  void* out;                 // filtered projections (layout above)
  float* scale;              // [kScaleElems] (FP16 / BF16) or null
  float hsum;                // sum |h_k| of the filter taps (bound on |y| / max|x|)
  int64_t raw_elems;         // raw floats (the abs-max pass)
  const RebinDev* tab;       // [ncols]
  const float* Hn;           // [nfft] real filter spectrum / nfft
  const float2* tw;          // [nfft] exp(-2 pi i k / nfft)
  int32_t nviews, nrows, ncols, cpitch, nfft, log2n;
  int32_t precision;
  int32_t nlines;            // nviews * nrows
  const float* lines_in;     // filter-only mode: [line][cpitch] FP32 input (no rebinning)
  int32_t ncu;               // compute units of the device (persistent grid size)
  int32_t raw_nrows, raw_ncols;   // raw detector (differs from nrows / ncols with FFS)
  int32_t states;            // focal states S (1 without FFS)
  int32_t zshift;            // 1 with z FFS: effective row q = 2 r + parity
  int32_t rebin_only;        // 1: write the rebinned rows (FP32) without filtering
  // Lines [line0, line0 + nlines) of the scan (line0 even, so the line pairs
  // are those of a whole-scan launch); the streaming reconstruction filters
  // views as they arrive.
  int32_t line0;
  int32_t skip_scale;        // 1: the FP16 / BF16 bound is already in scale[1]
  // The gather's raw window (rebinning): bytes per view group (S focal states
  // x raw rows x raw channels), and the smallest aoff and mmax of the table.
  uint32_t group_bytes;
  int32_t aoff_min, mmax_min;
  int32_t pairs;             // 1: output as row pairs (kPrecisionPairs and its 16-bit forms)
};

// FP32 projections stored as row pairs, the layout between the rebinning and
// the backprojection of the whole chains (plan_pairs): entry (view, row,
// channel) holds (y[row][channel], y[row + 1][channel]), 0 past the last row,
// so that the 2 x 2 taps of a sample are 16 consecutive bytes.  An FP32
// backprojection of rows needs two 8-byte gathers per sample, and the
// texture-address unit takes 16.7 cycles per 64-lane gather of 8 bytes and
// 20.3 of 16 (measured, taps of an 8 x 8 tile in L1): 86 % of the kernel's
// time.  The stage calls keep the row layout of their interface.
//
// FP16 / BF16 chains keep the same pairs in 16 bits (4 bytes per entry, the
// scan's scale as for the quads): the taps are 8 consecutive bytes as with
// the quads of the interface, in half the lines.
constexpr int kPrecisionPairs = 3, kPrecisionPairsF16 = 4, kPrecisionPairsB16 = 5;
inline int pair_storage(int precision) {
  return precision == FCT_PRECISION_FP32   ? kPrecisionPairs
         : precision == FCT_PRECISION_FP16 ? kPrecisionPairsF16
                                           : kPrecisionPairsB16;
}

// Everything the backprojection kernel reads.
struct BpArgs {
  const void* filt;          // filtered projections (layout above)
  const float* filt_scale;   // scale buffer of FP16 / BF16 projections
  float* native;             // [slice][y][x]
  int32_t* counts;           // count mode: [slice][y][x]
  unsigned long long* total; // count mode
  int32_t* sel;              // selection mode: [nviews]
  const float* xs;           // [nx]
  const float* ys;           // [ny]
  const float2* cs;          // [H] (cos, sin)
  const float* zs;           // [n_native] slice z relative to its chunk reference
  const float* zt;           // [nchunks][nviews] view z relative to the chunk reference
  const int2* slab_vrange;   // [nslabs] views [x, y) a slab can select
  const int2* wrange;        // [nchunks][nviews] native slices [x, y] inside the view window
  // [tiles_y * tiles_x][H] per 8 x 8 voxel tile and theta~: the extremes over
  // the tile's voxels in the FOV of the z-offsets from a view's table z at
  // which |q| = 1, (min, max) for the view parity 0 then 1
  // (launch_bp_zbounds).
  const float4* zbounds;
  FctBpConsts g;
  float scale;               // 2 pi / ppr
  int32_t nx, ny, n_native, nviews, H, cpitch;
  int32_t tiles_x, tiles_y, nslabs;
  int32_t sel_ix, sel_iy, sel_is;
  // Slabs [slab0, slab0 + slab_count) of a launch (slab_count 0: all); the
  // streaming reconstruction backprojects groups of slabs as their views
  // arrive.  Unused by the persistent batch kernel.
  int32_t slab0, slab_count;
  int32_t nseg;              // theta~ segments summed apart (bp_segments)
  // Tiles [xcd_first[x], xcd_first[x + 1]) of the launch, in slab-major order,
  // go to XCD x (plan_bp_share).  Unused by the persistent batch kernel.
  int32_t xcd_first[9];
};
constexpr int kBpMaxSegments = 16;

__host__ __device__ __forceinline__ int imin(int a, int b) { return a < b ? a : b; }

// Order of the tiles of a slab: square blocks of kSuper x kSuper tiles
// (row-major blocks, row-major tiles inside a block; partial blocks at the
// right and bottom edges), so that the tiles an XCD runs at the same time
// cover compact patches of the slice rather than a band of whole tile rows:
// a narrower detector footprint per view in the XCD's L2 (FP16 full
// workload 52.5 -> 48.6 ms against row-major order; blocks of 8 or 16
// tiles alike, 4 and 32 slower).  Only the order changes: every tile is
// computed as before.
constexpr int kSuper = 16;
__host__ __device__ __forceinline__ int2 tile_of(int l, int tiles_x, int tiles_y) {
  const int band = kSuper * tiles_x;                 // tiles of a full block row
  const int sy = l / band, r = l - sy * band;
  const int h = imin(kSuper, tiles_y - sy * kSuper);  // rows of this block row
  const int sx = r / (kSuper * h), r2 = r - sx * kSuper * h;
  const int w = imin(kSuper, tiles_x - sx * kSuper);  // columns of this block
  return make_int2(sx * kSuper + r2 % w, sy * kSuper + r2 / w);
}

// Segments of theta~ that a volume of so many tiles per slab sums apart, so
// that a small volume still fills the GPU (a wave per tile and segment): a
// power of two, up to 16 384 waves (2.3 rounds of the 7 x 1024 resident
// ones), at least four theta~ each.  Measured (FP32 / BF16 whole chains, 1 /
// 2 / 4 / 8 / 16 segments): 36 tiles 517 / 290 / 166 / 100 / 64 us; 4096
// tiles 5.78 / 5.81 / 5.45 / 5.40 / 6.02 ms; 8192 tiles 6.34 / 5.78 / 5.88 /
// 5.85 / 7.48 ms and 4.89 / 4.81 / 4.84 / 5.32 / 7.08 ms; 33 264 tiles 17.7 /
// 17.6 / 17.7 / 18.2 / 22.8 ms; 163 840 tiles 50.2 / 50.9 / 51.5 / 56.8 /
// 77.6 ms (more segments read more views at a time through each L2).  Tiles of 32
// slices (four waves per SIMD, half the sums per 64 KB of LDS): up to 2560 waves
// and 8 segments; 768 tiles FP32 / FP16 16.3 / 7.0 ms in one, 9.3 / 4.3 in two, 5.5 / 2.8
// in four; 2048 tiles 15.4 / 7.2, 9.2 / 6.8, 9.5 / 5.4; 3072 tiles 10.7 / 7.4 (backprojection
// 9.7 / 5.4), in two 11.2 / 6.9 (10.5 / 6.6).  It
// depends on the volume and the tile depth only, so that every entry point
// (streamed slab groups, batches) sums in the same order.
inline int bp_segments(int tiles, int nslabs, int H, int tile_z) {
  int s = 1;
  const int most = imin(kBpMaxSegments, 256 / tile_z), waves = tile_z > 16 ? 2560 : 16384;
  while (s < most && (int64_t)tiles * nslabs * s < waves && H / (2 * s) >= 4) s *= 2;
  return s;
}

// Persistent multi-job backprojection (backproject_v1.hip).
struct BpBatchArgs {
  const BpArgs* jobs;        // [n_jobs] device copy of each job's arguments
  const int32_t* tile_start; // [n_jobs + 1] first global tile of each job
  uint32_t* queue;           // [8] per-range tile counters, zero at launch
  int32_t n_jobs;            // <= 64
  int32_t total_tiles;
};

struct ThickenArgs {
  const float* native;
  float* out;
  const int32_t* off;        // [n_req + 1] into idx/w
  const int32_t* idx;        // native slice indices
  const float* w;            // normalised weights
  int32_t plane;             // nx*ny
  int32_t n_req;             // slices [s0, s0 + n_req) of the output
  int32_t s0;
  int32_t hu;                // 1: store 1000 (mu - mu_water) / mu_water = mu hu_scale - 1000
  float hu_scale;            // 1000 / mu_water
};

struct PhantomArgs {
  float* out;
  const fct_ellipsoid* ell;  // device copy
  int32_t n_ell;
  int32_t ncols, nrows, v0, v1;
  double r, dsd, dgamma, drow, cc, cr, angle0, dtheta, z0, dz;
  double cyl_r, cyl_mu, i0;
  unsigned long long seed;
  int32_t states;            // focal states (1: no FFS)
  int32_t mirror;            // 1: clockwise scan, rays mirrored y -> -y
  double ffs_off[4][3];      // per state (dr, da, dz) along (e_w, e_u, e_z)
};

// Ray-driven projector of the native volume onto the raw fan data
// (rayproj.hip), in the plan's frame (a clockwise scan mirrored).
struct RayProjArgs {
  const float* vol_in;       // project: native [slice][y][x]
  float* vol_out;            // transpose: native, accumulated into
  const float* raw_in;       // transpose: [view - v0][row][ch]
  float* raw_out;            // project: [view - v0][row][ch]
  int32_t ncols, nrows, v0, v1, nx, ny, nz, states;
  double r, dsd, dgamma, drow, cc, cr, angle0, dtheta, z0, dz;
  double ffs_off[4][3];      // per focal state (dr, da, dz) along (e_w, e_u, e_z)
  float gx0, gdx, gy0, gdy, gz0, gdz;   // voxel-centre grids (FP32 of FP64)
  double dx0, ddx, dy0, ddy, dz0, ddz;  // and in FP64
};

// Geometry tables of the table-driven ray projector (rayproj.hip).
struct RayTables {
  float4* ray;     // [view][channel] A, B, T0, DT
  float4* view;    // [view][2]: cos, sin, R + o0, o1; (-cr drow - oz) / gdz, o0, -, -
  double* zoff;    // [view] focal spot z in slices
  uint64_t* axis;  // [view][64 channels] bit: the ray's planes are x planes
  float* len2;     // [focal state][channel] squared in-plane source-detector distance
  double zsrc[4];  // focal state's z offset
};

struct RayGather {
  int32_t tiles_x, tiles_y, slabs, nsplit;   // 8 x 8 column tiles, slabs, splits of the views
  const float* rec;  // [view][row][channel] A, B, value x path length (ray_record_kernel)
  const uint64_t* nz;  // [view] bit per 32 channels: some ray is not zero
  double reach;    // mm of table z beyond a slab whose views can meet it
};

struct BpAdjArgs {
  BpArgs bp;                 // geometry tables (filt/native unused)
  const float* xbar;         // [slice][y][x] native-volume cotangent
  float* gbar;               // [view][row][cpitch] FP32, accumulated into
};

// Gathered transpose of the backprojection (adjoint.hip) for the theta~
// [t0, t0 + nt), all with the same primary axis (x planes: swap 1).
struct AdjGather {
  float* wgt;      // [nt][primary][slice][secondary] xbar scale / sum W; matched: the volume, swapped
  float4* col;     // [nt][primary][secondary] per-column geometry (bp_adjoint_column_kernel)
  int32_t t0, nt, swap, tile_z, nsplit;   // nsplit: waves sharing a ray's planes
  double gx0, gdx, gy0, gdy, dz;   // voxel-centre grid, slice step (mm, signed)
};

struct RebinAdjArgs {
  const float* gbar;         // [view][row][cpitch] (parallel, effective detector)
  float* pbar;               // [raw view][raw row][raw ch], overwritten
  const int32_t* off;        // [states * raw_ncols + 1] into ent
  const RebinTDev* ent;
  uint32_t* flags;           // [nviews] scratch: the view has a value
  int32_t nviews, nrows, cpitch;          // parallel views, effective rows
  int32_t raw_nviews, raw_nrows, raw_ncols, states, zshift;
};

hipError_t launch_rebin_filter(const RebinFilterArgs& a, hipStream_t s);
// Ray-driven projection of vol_in onto raw_out (views [v0, v1)), or with
// transpose its exact transpose from raw_in into vol_out (accumulated).
hipError_t launch_ray_project(const RayProjArgs& a, bool transpose, hipStream_t s);
// Table-driven forms: whether they apply, the tables (of ray_table_bytes) and
// the projector's padded volume copies (2 x ray_pad_elems entries of one
// slice, or of two where ray_pad_pairs).
bool ray_tables_apply(const RayProjArgs& a);
size_t ray_table_bytes(const RayProjArgs& a);
size_t ray_pad_elems(const RayProjArgs& a);
bool ray_pad_pairs(const RayProjArgs& a);
RayTables ray_table_layout(const RayProjArgs& a, void* mem);
hipError_t launch_ray_table(const RayProjArgs& a, const RayTables& t, hipStream_t s);
hipError_t launch_ray_project_table(const RayProjArgs& a, const RayTables& t, float* pad,
                                    bool pairs, hipStream_t s);
// rec: 2 floats per view and 3 per ray.
hipError_t launch_ray_gather(const RayProjArgs& a, const RayTables& t, float* rec, int ncu,
                             hipStream_t s);
// Adaptive filtration of raw views [v0, v1): per view the largest finite
// |p| (vmax), then every sample blended with its 3 x 3 (row, channel) mean by
// lambda = clamp((p - (1 - s) vmax) / (s vmax), 0, 1).  out != in.
hipError_t launch_adaptive_filter(const float* in, float* out, float* vmax, int v0, int v1,
                                  int nrows, int ncols, float s, hipStream_t st);
// FP16 / BF16 storage bound in scale[1]: cleared, raised to max|x| over n
// floats (accumulating over calls), or set from a caller's max|raw|.
hipError_t launch_scale_reset(float* scale, hipStream_t s);
hipError_t launch_absmax(const float* x, int64_t n, float* scale, int ncu, hipStream_t s);
hipError_t launch_scale_set(float* scale, float max_abs_raw, hipStream_t s);
// Streaming FP16 / BF16: scale[0] from the bound so far, scale[2] the factor
// for the quads already stored; then those n_entries quads rescaled by it.
hipError_t launch_scale_update(float* scale, float hsum, hipStream_t s);
hipError_t launch_scale_commit(float* scale, hipStream_t s);
hipError_t launch_quad_rescale(void* quads, size_t n_entries, int precision, const float* scale,
                               int ncu, hipStream_t s);
hipError_t launch_backproject_adjoint(const BpAdjArgs& a, int tile_z, hipStream_t s,
                                      bool matched = false);
// The gathered form of launch_backproject_adjoint, theta~ batch by batch: the
// column table, the voxels' weights (not for the matched projector, which reads the volume,
// swapped for x planes), then the detector samples (gbar overwritten).
hipError_t launch_adjoint_columns(const BpAdjArgs& a, const AdjGather& q, hipStream_t s);
hipError_t launch_adjoint_weights(const BpAdjArgs& a, const AdjGather& q, hipStream_t s);
hipError_t launch_swap_volume(const float* in, float* out, int nx, int ny, int nz, hipStream_t s);
int adjoint_gather_waves(const BpArgs& b);   // waves per theta~
hipError_t launch_adjoint_gather(const BpAdjArgs& a, const AdjGather& q, bool matched,
                                 hipStream_t s);
hipError_t launch_rebin_adjoint(const RebinAdjArgs& a, hipStream_t s);
hipError_t launch_fill(float* p, size_t n, float v, hipStream_t s);
hipError_t launch_backproject(const BpArgs& a, int tile_z, int variant, int precision, int mode,
                              hipStream_t s);
// Fills a.zbounds (a BpArgs whose zbounds member is the output) for the
// plan's tiles and theta~ (backproject_v1.hip).
hipError_t launch_bp_zbounds(const BpArgs& a, float4* zbounds, hipStream_t s);
hipError_t launch_backproject_v1(const BpArgs& a, int tile_z, int precision, int mode,
                                 hipStream_t s);
hipError_t launch_backproject_batch(const BpBatchArgs& b, int tile_z, int precision,
                                    bool centered, int grid, hipStream_t s);
hipError_t backproject_batch_waves_per_cu(int tile_z, int precision, int* waves);
hipError_t launch_thicken(const ThickenArgs& a, hipStream_t s);
hipError_t launch_row_pairs(const float* rows, void* out, int nviews, int nrows, int cpitch,
                            hipStream_t s);
hipError_t launch_phantom(const PhantomArgs& a, hipStream_t s);

// kBpMatched: the plain R / l-weighted sum over every view that sees the
// voxel (no view window, no W normalisation) -- the transpose of the matched
// projector of adjoint.hip's matched mode.
enum BpMode { kBpAccumulate = 0, kBpCount = 1, kBpSelect = 2, kBpMatched = 3 };

}  // namespace fct

struct fct_wfbp_gpu_plan;

namespace fct {
// Plan helpers shared by capi.hip and batch.hip.
BpArgs plan_bp_args(const fct_wfbp_gpu_plan* p);   // tables only (no buffers)
// Slabs [slab0, slab0 + count) of a launch (count 0: all), shared among the XCDs.
void plan_bp_share(const fct_wfbp_gpu_plan* p, int slab0, int count, BpArgs* a);
int plan_set_tile_z(fct_wfbp_gpu_plan* p, int tz);  // rebuilds the slab view ranges
// Rebin + filter of the lines some slab reads (the whole-chain entry points).
int chain_rebin_filter(fct_wfbp_gpu_plan* p, const float* raw, void* filtered, float* scale,
                       bool pairs);
// The lean backprojection of filtered projections in the plan's own layout
// (pairs), or in the interface's.
int chain_backproject(fct_wfbp_gpu_plan* p, const void* filtered, const float* scale,
                      float* native, bool pairs);
// alloc_chain on the current device, for n plans of one precision: the scale
// and native volumes, `extra`, then the filtered projections, as pairs in all of
// the plans or in none (p->pairs).  reserve: pairs only where they leave what
// the plans' other calls allocate (later_bytes).
hipError_t plans_alloc_chain(fct_wfbp_gpu_plan* const* plans, int n, const Buffer* extra,
                             int n_extra, bool reserve);
}  // namespace fct

struct fct_wfbp_gpu_ctx {
  int device = 0;
  std::string last_error;
  // The streaming chain's copy stream and two backprojection streams,
  // shared by the context's plans (created on first use): with a few
  // hardware queues per process (GPU_MAX_HW_QUEUES), streams of every plan
  // would share queues with the plans' own streams, and a copy queued
  // behind a kernel waits for it.
  hipStream_t copy_stream = nullptr;
  hipStream_t bp_stream[2] = {nullptr, nullptr};
};

struct fct_wfbp_gpu_plan {
  fct_wfbp_gpu_ctx* ctx = nullptr;
  int device = 0;
  hipStream_t stream = nullptr;
  fct_scan_geometry scan{};         // interleaved (effective) geometry, ffs_mode none
  fct_scan_geometry raw_scan{};     // as given (raw detector, FFS mode)
  fct_ffs::Geometry ffs{};
  fct_recon_config recon{};
  fct_exec_options opts{};

  int ncols = 0, nrows = 0, nviews = 0, ppr = 0, H = 0, nfft = 0, log2n = 0, cpitch = 0;
  int n_native = 0, n_req = 0, nchunks = 0, tile_z = 16, variant = 0, nslabs = 0;
  int ncu = 0;                      // compute units of the plan's device
  double dgamma = 0, ds = 0, dtheta = 0, dz = 0, csw = 0, acq = 0;
  FctBpConsts g{};
  float scale = 0;
  int out_hu = 0;                   // thickened volume in HU (fct_wfbp_gpu_set_output_units)
  double mu_water = 0;
  int af_on = 0;                    // adaptive filtration of the raw scan before rebinning
  float af_s = 0;                   // its strength s in (0, 1]

  // Device tables owned by the plan.
  float* d_xs = nullptr;
  float* d_ys = nullptr;
  float2* d_cs = nullptr;
  float* d_zs = nullptr;
  float* d_zt = nullptr;
  int2* d_slab_vrange = nullptr;
  int2* d_wrange = nullptr;
  float4* d_zbounds = nullptr;
  fct::RebinDev* d_rebin = nullptr;
  fct::RebinTDev* d_rebinT = nullptr;   // by raw channel; its offsets follow the entries
  int rebinT_entries = 0;
  uint32_t* d_view_flags = nullptr;     // [nviews] scratch of the rebinning's transpose
  float* d_Hn = nullptr;
  float2* d_tw = nullptr;
  int32_t* d_thk_off = nullptr;
  int32_t* d_thk_idx = nullptr;
  float* d_thk_w = nullptr;

  // Intermediate buffers for fct_wfbp_gpu_reconstruct (allocated on first use).
  bool pairs = false;               // d_filtered holds row pairs (kPrecisionPairs)
  void* d_filtered = nullptr;
  float* d_scale = nullptr;
  float* d_native = nullptr;
  float* d_raw_stage = nullptr;
  float* d_vol_stage = nullptr;
  void* d_ray_tab = nullptr;        // ray projector tables (first use; ready: filled)
  bool ray_tab_ready = false;
  float* d_ray_pad = nullptr;       // padded volume copies of the ray projector (first use)
  bool ray_pad_pairs = false;       // with two slices per entry
  float* d_ray_rec = nullptr;       // per-ray records of its transpose (first use)
  // Gathered transposes (first use of each): columns and voxel weights of the
  // backprojection's, columns and swapped volume of the matched projector's.
  float* d_adj_scratch[2] = {nullptr, nullptr};
  std::vector<uint8_t> h_xplanes;   // per theta~: its parallel rays run along x planes
  float* d_gbar = nullptr;          // adjoint scratch, [view][row][cpitch] FP32
  int32_t* d_thkT_off = nullptr;    // transposed thickening table
  int32_t* d_thkT_idx = nullptr;
  float* d_thkT_w = nullptr;
  float* d_af_raw = nullptr;        // adaptively filtered raw scan (allocated on first use)
  float* d_af_vmax = nullptr;       // per raw view max |p|

  // Streaming reconstruction (fct_wfbp_gpu_reconstruct_stream and the host
  // path of fct_wfbp_gpu_reconstruct), created on first use.
  hipEvent_t ev_compute = nullptr;
  float* h_stage[2] = {nullptr, nullptr};   // pinned staging for a view reader
  int stage_views = 0;
  hipEvent_t ev_bp[2] = {nullptr, nullptr};   // after the latest piece on each stream
  hipEvent_t ev_rebin = nullptr;         // after the latest rebinning launch
  hipEvent_t ev_ratio = nullptr;         // after the storage-scale ratio's copy to h_ratio
  float* h_ratio = nullptr;              // pinned: scale[2] of the latest scale update
  std::vector<int2> h_slab_vrange;      // host copy of d_slab_vrange
  std::vector<int32_t> h_tile_active;   // [tiles + 1] tiles with a voxel in the FOV before tile l
  std::vector<fct::RebinDev> h_rebin;   // host copy of d_rebin
  std::vector<int32_t> h_thk_need;      // per requested slice: 1 + its last native slice (0: none)
  std::vector<hipEvent_t> ev_chunk;     // per chunk: its copy has landed
  int rebin_reach = 0;                  // parallel view j reads raw projections < j S + reach
  int rebin_aoff_min = 0, rebin_mmax_min = 0;   // over the rebinning table (the gather window)

  int64_t raw_elems() const {
    return (int64_t)raw_scan.n_views * raw_scan.n_rows * raw_scan.n_channels;
  }
  size_t filtered_entry_bytes() const {   // FP32 value, or 4 x 16-bit quad
    return opts.precision == FCT_PRECISION_FP32 ? 4 : 8;
  }
  size_t filtered_bytes() const {
    return (size_t)nviews * nrows * cpitch * filtered_entry_bytes();
  }
  // The plan's own buffer between the stages of a whole chain.
  int storage() const { return pairs ? fct::pair_storage(opts.precision) : opts.precision; }
  size_t storage_bytes() const { return pairs ? pairs_bytes() : filtered_bytes(); }
  size_t storage_entry_bytes() const { return storage_bytes() / ((size_t)nviews * nrows * cpitch); }
  size_t pairs_bytes() const {
    return (size_t)nviews * nrows * cpitch * (opts.precision == FCT_PRECISION_FP32 ? 8 : 4);
  }
  size_t native_bytes() const {
    return (size_t)n_native * recon.ny * recon.nx * sizeof(float);
  }
  size_t volume_bytes() const { return (size_t)n_req * recon.ny * recon.nx * sizeof(float); }
  // What calls beside the chain on device buffers may still have to allocate
  // and have no way around: the host paths' staging, the adjoint's lines.
  size_t later_bytes() const {
    return (d_raw_stage ? 0 : (size_t)raw_elems() * sizeof(float)) +
           (d_vol_stage ? 0 : volume_bytes()) +
           (d_gbar ? 0 : (size_t)nviews * nrows * cpitch * sizeof(float));
  }
  size_t scale_elems() const {
    return opts.precision == FCT_PRECISION_FP32 ? 0 : (size_t)fct::kScaleElems;
  }
  double hsum = 0;                  // sum |h_k| of the filter taps
};
