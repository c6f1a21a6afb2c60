// Tile rasterization (front-to-back alpha compositing) forward / backward for
// gfx950.
//
// Forward: one block per (image, tile) with tile_size^2 lanes, one pixel per
// lane (16x16 tiles -> 4 wave64s, each covering an 8x8 block). The tile's
// sorted Gaussian list is walked in batches of blockDim entries: each lane
// gathers one Gaussian record (mean, conic, opacity, colors) into LDS and
// tests it against every wave's pixel rectangle, then each wave evaluates
// only the records that may touch it. The forward stops when every lane of
// the block has saturated (block vote).
//
// Backward: one block per tile, dispatched heaviest tile first, replays the
// tile's list back-to-front from its largest last_id, rebuilding
// transmittance per pixel, and each batch ends with one atomic per (record,
// nonzero component). raster_bwd_rows_kernel keeps 16 records in a wave's lanes
// and runs the pixel recurrences across them; raster_bwd_kernel (short lists,
// other tile sides, more than four channels, absolute gradients) keeps pixels in
// lanes and sums each record's partial gradients over the wave by a transposed
// DPP/permlane reduction into per-wave LDS slots. The forward has the same two
// forms: raster_fwd_rows_kernel and raster_fwd_kernel.
//
// Per-pixel math follows gsplat_core/gsplat_rasterize.cpp:291-368 (forward)
// and :432-554 (backward) operation for operation; the Gaussian falloff and
// alpha tests are evaluated exactly as the reference (no FMA contraction in
// this file; the backward's gradient arithmetic uses explicit FMAs) so
// compositing decisions match it.
#include <algorithm>
#include <atomic>
#include <climits>
#include <mutex>
#include <type_traits>

#include "common.hpp"
#include "scan.hpp"

// Scratch of gsplat_hip_rasterize_bwd_noalloc: the backward's tile schedule
// (cost and order per tile) and background-gradient partials (per tile and
// channel), in device memory that every GPU the library runs on holds from
// load to process end. Host code never uses this name as an address: the
// address is looked up per device (noalloc_scratch below).
constexpr size_t kNoAllocScratchBytes = static_cast<size_t>(8) << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace gsplat_hip {
namespace {

constexpr int kMaxChannels = 64;

// Words of one backward batch record in LDS: conic xyz + opacity, then mean
// xy, the CH staged colours (none for CH == 0), the Gaussian id and the
// per-wave touch mask, padded to 16 bytes.
__host__ __device__ constexpr int bwd_record_words(int ch) { return 4 + (2 + ch + 2 + 3) / 4 * 4; }

// The rows kernels' forward record also carries the touch mask.
__host__ __device__ constexpr int fwd_rows_record_words(int ch) { return 4 + (2 + ch + 1 + 3) / 4 * 4; }

struct RasterArgs {
  const float* means2d;
  const float* conics;
  const float* colors;
  const float* opacities;
  const float* backgrounds;
  const uint8_t* masks;
  const int32_t* tile_offsets;
  const int32_t* flatten_ids;
  int64_t N;
  int channels;
  int W, H, ts, tw, th;
  int64_t I;
  int64_t n_isects;
  int64_t G;  // Gaussian rows: I * N (dense) or nnz (packed)
};

// Range of the tile's list; the last tile of the last image ends at n_isects
// (gsplat_rasterize.cpp:296-299).
__device__ __forceinline__ void tile_range(const RasterArgs& a, int64_t image, int tile, int64_t* start,
                                           int64_t* end) {
  const int64_t n_tiles = static_cast<int64_t>(a.tw) * a.th;
  const int64_t oi = image * n_tiles + tile;
  const int64_t s = a.tile_offsets[oi];
  const int64_t e = (oi + 1 == a.I * n_tiles) ? a.n_isects : a.tile_offsets[oi + 1];
  // consistent offsets already satisfy 0 <= s <= e <= n_isects; clamping only
  // keeps reads in bounds for inconsistent caller data
  *start = min(max<int64_t>(s, 0), a.n_isects);
  *end = min(max(e, *start), a.n_isects);
}

// Gaussian record of list entry j; ids outside [0, G) read as a
// zero-opacity Gaussian (never contributes) instead of reading out of bounds.
__device__ __forceinline__ int32_t load_gaussian(const RasterArgs& a, int64_t j, float2* xy, float4* co) {
  int32_t g = a.flatten_ids[j];
  if (g < 0 || static_cast<int64_t>(g) >= a.G) {
    *xy = make_float2(0.0f, 0.0f);
    *co = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    return 0;
  }
  const int64_t gg = g;
  *xy = make_float2(a.means2d[gg * 2], a.means2d[gg * 2 + 1]);
  *co = make_float4(a.conics[gg * 3], a.conics[gg * 3 + 1], a.conics[gg * 3 + 2], a.opacities[gg]);
  return g;
}

// exp(y) by Cody-Waite reduction: y log2(e) = n + f with the product kept
// exact to about 2^-48 (log2(e) split into a float head and tail, the head's
// rounding error recovered by an FMA), 2^f from v_exp_f32, scaled by 2^n.
// The tail is log2(e) - head truncated to float (0x32a5705f), the value the
// device library's expf uses, which makes this bit-identical to expf for
// every float y > -103 (compared exhaustively on gfx950); it only drops
// expf's range selects.
//
// Below -104 the argument is raised to -104 first (IEEE maximum: one
// v_maximum3_f32, NaN passes through). Without it the reduction breaks down
// for y < -2.98e9, where ulp(y log2 e) >= 256 leaves a residual f >= 128 and
// 2^f overflows (ldexp(inf, n) = inf), and for y = -inf, where the head's
// error term is inf - inf = NaN. With it every y <= -104 gives at most
// 2^-149, so o * exp fails the 1/255 alpha test for any finite opacity, as
// expf's 0 does; a NaN argument still yields NaN (alpha = min(0.99, NaN) =
// 0.99, the reference's std::min result).
__device__ __forceinline__ float exp_alpha(float y) {
  const float head = 1.44269502162933349609375f;  // float(log2 e)
  const float tail = __uint_as_float(0x32a5705fu);
  y = __builtin_elementwise_maximum(y, -104.0f);
  const float ph = y * head;
  float pl = __builtin_fmaf(y, head, -ph);
  pl = __builtin_fmaf(y, tail, pl);
  const float n = __builtin_rintf(ph);
  const float f = (ph - n) + pl;
  return __builtin_ldexpf(__builtin_amdgcn_exp2f(f), static_cast<int>(n));
}

// exp_alpha for y in (-1.48e9, 0] without the lower clamp: the same bits down to
// -103, and below that at most 2^-149 as well, which no alpha test passes. The
// conversion of n bounds the range (|n| < 2^31).
__device__ __forceinline__ float exp_alpha_bounded(float y) {
  const float head = 1.44269502162933349609375f;  // float(log2 e)
  const float tail = __uint_as_float(0x32a5705fu);
  const float ph = y * head;
  float pl = __builtin_fmaf(y, head, -ph);
  pl = __builtin_fmaf(y, tail, pl);
  const float n = __builtin_rintf(ph);
  const float f = (ph - n) + pl;
  return __builtin_ldexpf(__builtin_amdgcn_exp2f(f), static_cast<int>(n));
}

// Classes of records whose alpha needs fewer tests for the same result
// (staged with the record's touch mask, bits above the waves'):
// - kGeneralRecord clear: a conic well inside the positive definite ones
//   (det > 1e-4 c0 c2 keeps the computed sigma >= 0: its rounding is below
//   1e-6 of c0 dx^2 + c2 dy^2, the form above 5e-5 of it, and neither
//   underflows), and an opacity up to 1. A visiting wave's 8x8 pixels have a
//   point with sigma below 6 within 9.9 of every pixel; sqrt(sigma) is a norm of
//   the offset, at most sqrt((c0 + c2) / 2) <= 1000 per pixel, so sigma stays below
//   (2.5 + 9900)^2 < 1e8 and the exponential needs no clamp.
// - kCappedRecord clear: also an opacity up to 0.99, so alpha = o exp(-sigma)
//   never meets the cap.
// - kNonFiniteRecord: a non-finite staged colour, in the backward also a
//   non-finite mean (records in lanes: a colour beyond kTameColor).
constexpr uint32_t kNonFiniteRecord = 1u << 31;
constexpr uint32_t kGeneralRecord = 1u << 30;
constexpr uint32_t kCappedRecord = 1u << 29;

__device__ __forceinline__ uint32_t record_class(float2 m, float4 co) {
  const bool plain = co.x > 1.0e-15f && co.z > 1.0e-15f && co.x < 1.0e6f && co.z < 1.0e6f &&
                     co.x * co.z - co.y * co.y > 1.0e-4f * co.x * co.z && fabsf(m.x) < 1.0e9f &&
                     fabsf(m.y) < 1.0e9f && co.w <= 1.0f;
  if (!plain) return kGeneralRecord | kCappedRecord;
  return co.w <= kMaxAlpha ? 0u : kCappedRecord;
}

// sigma of a record with a halved conic diagonal: (0.5 c0 dx) dx + (0.5 c2 dy) dy
// equals 0.5 ((c0 dx) dx + (c2 dy) dy) bit for bit (scaling by 2 commutes with
// rounding away from the subnormal range), one multiply less per visit.
__device__ __forceinline__ float halved_sigma(const float4& co, float dx, float dy) {
  return (co.x * dx * dx + co.z * dy * dy) + co.y * dx * dy;
}

// ---------------------------------------------------------------------------
// Per-wave culling. When a batch record is staged, its loader tests it once
// against every wave's pixel rectangle and stores a bit mask; each wave
// collects the set bits of 64 records at a time with one ballot and visits
// only those records. A bit is cleared only when no pixel of the wave can
// pass the alpha test: alpha = min(0.99, o exp(-sigma)) >= 1/255 needs
// sigma <= ln(255 o), and the minimum of sigma over the rectangle of the
// wave's pixel centres (a positive-definite quadratic: zero if the mean is
// inside, else the smallest of the four clamped edge minima) exceeds
// 1.05 ln(255 o) + 1e-4. For conics with det > 1e-4 c0 c2 the float32
// rounding of that minimum and of the per-pixel sigma, exp and threshold is
// below 1%, well inside the slack; other conics, non-finite values and NaN
// opacities are never culled, and opacities <= 0 always are (alpha <= 0).
// Culled records cannot change a pixel of that wave, so results are
// unchanged.
struct PixRect {
  float x0, x1, y0, y1;
};

// Lane -> pixel of a tile. When the tile side is a multiple of 8, each
// wave64 owns an 8x8 block (waves row-major over the blocks); the square
// footprint is touched by fewer Gaussians than a 16x4 strip of the same
// area, so fewer records pass the per-wave cull. Other tile sides map lanes
// row-major. Lanes past ts*ts (padding) map outside the tile.
__device__ __forceinline__ void lane_pixel(int t, int ts, int* qx, int* qy) {
  if ((ts & 7) == 0) {
    const int w = t / kWave, l = t % kWave;
    const int bpr = ts >> 3;  // 8x8 blocks per tile row
    *qx = (w % bpr) * 8 + (l & 7);
    *qy = (w / bpr) * 8 + (l >> 3);
  } else {
    *qx = t % ts;
    *qy = t / ts;
  }
}

// Bounding rectangle of the pixel centres owned by wave w (lane_pixel's map).
__device__ __forceinline__ PixRect wave_rect(int w, int ts, int tx, int ty) {
  int c0, c1, r0, r1;
  if ((ts & 7) == 0) {
    const int bpr = ts >> 3;
    c0 = (w % bpr) * 8;
    c1 = c0 + 7;
    r0 = (w / bpr) * 8;
    r1 = r0 + 7;
  } else {
    const int q0 = w * kWave;
    const int q1 = min(q0 + kWave, ts * ts) - 1;
    r0 = q0 / ts;
    r1 = q1 / ts;
    c0 = 0;
    c1 = ts - 1;
    if (r0 == r1) {
      c0 = q0 % ts;
      c1 = q1 % ts;
    }
  }
  PixRect r;
  r.x0 = static_cast<float>(tx * ts + c0) + 0.5f;
  r.x1 = static_cast<float>(tx * ts + c1) + 0.5f;
  r.y0 = static_cast<float>(ty * ts + r0) + 0.5f;
  r.y1 = static_cast<float>(ty * ts + r1) + 0.5f;
  return r;
}

__device__ __forceinline__ float quad_form(float c0, float c1, float c2, float dx, float dy) {
  return 0.5f * (c0 * dx * dx + c2 * dy * dy) + c1 * dx * dy;
}

// A record's cull constants, formed once for all the rectangles it is tested
// against: the bound 1.05 ln(255 o) + 1e-4 on the minimum of sigma, and the
// conic's reciprocal diagonal for the clamped edge minimisers. Both come from
// the hardware approximations (v_log_f32, v_rcp_f32: about 1 ulp), far inside
// the slack; a denormal 255 o that v_log_f32 flushes gives ln = -inf, which
// culls the record as the exact logarithm (about -90) does. `always`: never
// culled (ill-conditioned or non-finite values, NaN opacity); `never`: always
// culled (opacity <= 0).
struct CullRec {
  float mx, my, c0, c1, c2, ic0, ic2, bound;
  bool always, never;
};

__device__ __forceinline__ CullRec cull_rec(float2 m, float4 co) {
  CullRec r;
  r.mx = m.x;
  r.my = m.y;
  r.c0 = co.x;
  r.c1 = co.y;
  r.c2 = co.z;
  const float o = co.w;
  r.never = o <= 0.0f;
  const float t = __builtin_amdgcn_logf(255.0f * o) * 0.69314718055994531f;  // log2 -> ln
  r.always = !r.never && (!(t < 1.0e30f) || !(r.c0 > 0.0f && r.c2 > 0.0f && r.c0 < 1.0e30f && r.c2 < 1.0e30f) ||
                          !(r.c0 * r.c2 - r.c1 * r.c1 > 1.0e-4f * r.c0 * r.c2) || !(fabsf(m.x) < 1.0e30f) ||
                          !(fabsf(m.y) < 1.0e30f));
  r.ic0 = __builtin_amdgcn_rcpf(r.c0);
  r.ic2 = __builtin_amdgcn_rcpf(r.c2);
  r.bound = 1.05f * t + 1.0e-4f;
  return r;
}

__device__ __forceinline__ bool may_touch(const CullRec& c, const PixRect& r) {
  if (c.never) return false;
  if (c.always) return true;
  if (c.mx >= r.x0 && c.mx <= r.x1 && c.my >= r.y0 && c.my <= r.y1) return true;
  float best = __builtin_huge_valf();
  // vertical edges (dx fixed), then horizontal edges (dy fixed)
  for (int e = 0; e < 2; ++e) {
    const float dx = c.mx - (e ? r.x1 : r.x0);
    const float dy = fminf(fmaxf(-c.c1 * dx * c.ic2, c.my - r.y1), c.my - r.y0);
    best = fminf(best, quad_form(c.c0, c.c1, c.c2, dx, dy));
  }
  for (int e = 0; e < 2; ++e) {
    const float dy = c.my - (e ? r.y1 : r.y0);
    const float dx = fminf(fmaxf(-c.c1 * dy * c.ic0, c.mx - r.x1), c.mx - r.x0);
    best = fminf(best, quad_form(c.c0, c.c1, c.c2, dx, dy));
  }
  return !(best > c.bound);
}

// The block's wave rectangles (x0, x1, y0, y1 per wave), formed once per
// block into LDS so that the staging lanes read them instead of converting
// the integer bounds for every record; visible after the block's next
// barrier.
__device__ __forceinline__ void store_wave_rects(float4* s_rect, int n_waves, int ts, int tx, int ty) {
  const int w = threadIdx.x;
  if (w < n_waves) {
    const PixRect r = wave_rect(w, ts, tx, ty);
    s_rect[w] = make_float4(r.x0, r.x1, r.y0, r.y1);
  }
}

__device__ __forceinline__ uint32_t touch_mask(float2 m, float4 co, int n_waves, const float4* s_rect) {
  const CullRec c = cull_rec(m, co);
  uint32_t mask = 0;
  for (int w = 0; w < n_waves; ++w) {
    const float4 r = s_rect[w];
    if (may_touch(c, PixRect{r.x, r.y, r.z, r.w})) mask |= 1u << w;
  }
  return mask;
}

// Words of one forward batch record in LDS: conic xyz + opacity, then mean xy
// and the CH staged colours (CH == 0: the Gaussian id), padded to 16 bytes.
__host__ __device__ constexpr int fwd_record_words(int ch) { return 4 + (2 + (ch > 0 ? ch : 1) + 3) / 4 * 4; }
// CH in 1..4: colors staged in LDS; CH == 0: runtime channel count (<= 64),
// colors read from global memory.
//
// Records are visited in pairs (the two falloffs and alpha tests are
// straight-line code that overlaps; compositing stays in list order, an odd
// count ends with an inert second visit). Each composite is an exec-masked
// branch taken by the lanes that keep the record.
template <int CH>
__global__ void __launch_bounds__(1024) raster_fwd_kernel(RasterArgs a, float* __restrict__ render_colors,
                                                          float* __restrict__ render_alphas,
                                                          int32_t* __restrict__ last_ids) {
  constexpr int FW = fwd_record_words(CH);
  extern __shared__ float smem[];
  const int BS = blockDim.x;
  float* s_rec = smem;                                               // [BS][FW]
  uint32_t* s_mask = reinterpret_cast<uint32_t*>(smem + FW * BS);   // [BS] per-wave touch bits
  float4* s_rect = reinterpret_cast<float4*>(smem + (FW + 1) * BS);  // [n_waves] wave pixel rects

  const int channels = CH > 0 ? CH : a.channels;
  const int tx = blockIdx.x, ty = blockIdx.y;
  const int64_t image = blockIdx.z;
  const int tile = ty * a.tw + tx;
  const int t = threadIdx.x;
  const int lane = t % kWave;
  const int wave = t / kWave;
  const int n_waves = BS / kWave;
  int qx, qy;
  lane_pixel(t, a.ts, &qx, &qy);
  const int x = tx * a.ts + qx;
  const int y = ty * a.ts + qy;
  // blocks are padded to whole wave64s; padding lanes own no pixel
  const bool inside = t < a.ts * a.ts && x < a.W && y < a.H;
  const int64_t pix = (image * a.H + y) * static_cast<int64_t>(a.W) + x;
  const float* bg = a.backgrounds ? a.backgrounds + image * channels : nullptr;
  const int64_t n_tiles = static_cast<int64_t>(a.tw) * a.th;

  if (a.masks && !a.masks[image * n_tiles + tile]) {
    if (inside) {
      render_alphas[pix] = 0.0f;
      for (int c = 0; c < channels; ++c) render_colors[pix * channels + c] = bg ? bg[c] : 0.0f;
      last_ids[pix] = 0;
    }
    return;
  }
  int64_t start, end;
  tile_range(a, image, tile, &start, &end);
  store_wave_rects(s_rect, n_waves, a.ts, tx, ty);
  const float px = static_cast<float>(x) + 0.5f;
  const float py = static_cast<float>(y) + 0.5f;
  float T = 1.0f;
  int32_t cur = 0;
  float acc[CH > 0 ? CH : kMaxChannels];
#pragma unroll
  for (int c = 0; c < (CH > 0 ? CH : kMaxChannels); ++c) acc[c] = 0.0f;
  bool done = !inside;

  for (int64_t b0 = start; b0 < end; b0 += BS) {
    if (__syncthreads_count(done) == BS) break;  // also fences the previous batch's LDS reads
    const int64_t j = b0 + t;
    if (j < end) {
      float2 xy;
      float4 co;
      const int32_t g = load_gaussian(a, j, &xy, &co);
      float* rec = s_rec + t * FW;
      // conic diagonal pre-halved: (0.5 c0 dx) dx + (0.5 c2 dy) dy equals
      // 0.5 ((c0 dx) dx + (c2 dy) dy) bit for bit (scaling by 2 commutes with
      // rounding away from the subnormal range), one multiply less per visit
      *reinterpret_cast<float4*>(rec) = make_float4(0.5f * co.x, co.y, 0.5f * co.z, co.w);
      float tail[FW - 4];
#pragma unroll
      for (int i = 0; i < FW - 4; ++i) tail[i] = 0.0f;
      tail[0] = xy.x;
      tail[1] = xy.y;
      const uint32_t mask = touch_mask(xy, co, n_waves, s_rect);
      if constexpr (CH > 0) {
#pragma unroll
        for (int c = 0; c < CH; ++c) tail[2 + c] = a.colors[static_cast<int64_t>(g) * CH + c];
      } else {
        tail[2] = __int_as_float(g);
      }
#pragma unroll
      for (int i = 0; i < FW - 4; i += 4)
        *reinterpret_cast<float4*>(rec + 4 + i) = make_float4(tail[i], tail[i + 1], tail[i + 2], tail[i + 3]);
      s_mask[t] = mask;
    }
    __syncthreads();
    const int cnt = static_cast<int>(min<int64_t>(BS, end - b0));

    // Compositing of one visit after its falloff (list order): skip when
    // sigma < 0 or alpha < 1/255; stop (without this record) when T would
    // fall to the threshold. The update is a branch, so the lanes that do not
    // take the record run it with their exec bit clear: they add nothing,
    // not even a non-finite colour, and a record no lane takes costs no
    // update at all.
    auto composite = [&](int k, const float4& xc, const float4& ex, bool pass_in, float alpha) {
      const bool pass = !done && pass_in;
      const float next_T = T * (1.0f - alpha);
      // next_T is never NaN (alpha = min(0.99, .) is not, and T only takes
      // values above the threshold), so one comparison decides both ways
      const bool live = next_T > kTransmittanceThreshold;
      done = done || (pass && !live);
      if (pass && live) {
        const float vis = alpha * T;
        if constexpr (CH > 0) {
          const float col[4] = {xc.z, xc.w, ex.x, ex.y};
#pragma unroll
          for (int c = 0; c < CH; ++c) acc[c] = __builtin_fmaf(col[c], vis, acc[c]);
        } else {
          const float* colp = a.colors + static_cast<int64_t>(__float_as_int(xc.z)) * channels;
          for (int c = 0; c < channels; ++c) acc[c] += colp[c] * vis;
        }
        cur = static_cast<int32_t>(b0 + k);
        T = next_T;
      }
    };
    auto falloff = [&](const float4& co, const float4& xc, bool* pass, float* alpha) {
      const float dx = xc.x - px;
      const float dy = xc.y - py;
      const float sigma = (co.x * dx * dx + co.z * dy * dy) + co.y * dx * dy;  // co.x, co.z pre-halved
      *alpha = fminf(kMaxAlpha, co.w * exp_alpha(-sigma));
      *pass = !(sigma < 0.0f || *alpha < kAlphaThreshold);
    };
    auto load = [&](int k, float4& co, float4& xc, float4& ex) {
      const float4* rec = reinterpret_cast<const float4*>(s_rec + k * FW);
      co = rec[0];
      xc = rec[1];
      if constexpr (FW > 8) ex = rec[2];
    };
    for (int c0 = 0; c0 < cnt; c0 += kWave) {
      // records of this 64-slot chunk that may touch this wave (all lanes vote)
      const int kl = c0 + lane;
      const uint32_t mk = kl < cnt ? s_mask[kl] : 0u;
      const bool mine = (mk >> wave) & 1u;
      uint64_t bits = __ballot(mine);
      if (__ballot(!done) == 0) bits = 0;  // every pixel of the wave has saturated
      while (bits) {
        const int k1 = c0 + __builtin_ctzll(bits);
        bits &= bits - 1;
        const bool two = bits != 0;
        const int k2 = two ? c0 + __builtin_ctzll(bits) : k1;
        bits &= bits - 1;
        float4 co1, xc1, ex1 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        float4 co2, xc2, ex2 = ex1;
        load(k1, co1, xc1, ex1);
        load(k2, co2, xc2, ex2);
        bool p1, p2;
        float al1, al2;
        falloff(co1, xc1, &p1, &al1);
        falloff(co2, xc2, &p2, &al2);
        composite(k1, xc1, ex1, p1, al1);
        composite(k2, xc2, ex2, p2 && two, al2);
      }
    }
  }
  if (!inside) return;
  render_alphas[pix] = 1.0f - T;
  if constexpr (CH > 0) {
#pragma unroll
    for (int c = 0; c < CH; ++c) render_colors[pix * CH + c] = acc[c] + T * (bg ? bg[c] : 0.0f);
  } else {
    for (int c = 0; c < channels; ++c) render_colors[pix * channels + c] = acc[c] + T * (bg ? bg[c] : 0.0f);
  }
  last_ids[pix] = cur;
}

// The pixels of a wave and of its lanes in the kernels that keep 16 records in
// lanes: lane l holds record l % 16 of a group and, in lane group l / 16, NX
// columns of two rows of the wave's BX x BY pixel block. P = 64: an 8x8 block,
// lane group g has rows g and g + 4. P = 32 (8x4) and P = 16 (4x4): lane groups
// are 2 x 2 over the block, two adjacent rows each. Pixel (x, y) of the block
// has index y BX + x.
template <int P>
struct RowBlock {
  static constexpr int BX = P == 16 ? 4 : 8, BY = P / BX;
  static constexpr int NX = P / 8;                    // columns of a lane
  static constexpr int HS = P == 64 ? 4 : 1;          // rows between a lane's two
  static __device__ __forceinline__ int x0(int g) { return P == 64 ? 0 : (g & 1) * NX; }
  static __device__ __forceinline__ int y0(int g) { return P == 64 ? g : (g >> 1) * 2; }
  static __device__ __forceinline__ PixRect rect(int w, int ts, int tx, int ty) {
    const int bpr = ts / BX;
    PixRect r;
    r.x0 = static_cast<float>(tx * ts + (w % bpr) * BX) + 0.5f;
    r.x1 = r.x0 + static_cast<float>(BX - 1);
    r.y0 = static_cast<float>(ty * ts + (w / bpr) * BY) + 0.5f;
    r.y1 = r.y0 + static_cast<float>(BY - 1);
    return r;
  }
};

// Forward with records in lanes: tile sides 8 and 16, one to four channels
// (fwd_rows_faster says where).
// Staging and culling are raster_fwd_kernel's, and so are every alpha,
// transmittance and sum, bit for bit. A wave takes the records that may touch
// its pixels in groups of 16, in two steps:
// 1. records in lanes: each lane evaluates the alphas of its record at its
//    columns and rows (RowBlock; a column's (0.5 c0 dx) dx and c1 dx serve two
//    rows, a row's (0.5 c2 dy) dy every column) and stores them in LDS, 0 where
//    the alpha test fails. Groups without capped or general records skip the
//    cap's and sigma's tests.
// 2. one pixel per lane: the group's records in list order, without a branch.
//
// The kernel with pixels in lanes throughout was bound by VALU issue too (0.99):
// 37 instructions per (wave, record) visit and 22 scalar ones for the visits'
// bit masks and branches, here 17 + 11 and few: 155 -> 135 us at 1M Gaussians,
// 1297x840 (1.81 -> 1.73 ms over 8 images of 1920x1080, 714 -> 671 us at
// 3840x2160). Batches of 128 records keep 6 blocks per CU by LDS (135 us, 192:
// 142 us, 256: 161 us). Skipping step 2's tests in waves whose pixels all
// stay live was slower (138 us), as was branching around records.
//
// Small grids (P < 64, the tile split over 64 / P blocks of its own): few tiles
// leave most SIMDs idle while the heaviest tile runs, so a tile's 8x8 pixel
// blocks are cut into 8x4 or 4x4 ones with a wave each, and a block takes half
// or a quarter of the tile. More waves repeat step 2's lanes and the staging,
// so this stops paying once the tiles fill the chip (10,000 Gaussians at
// 256x256, 256 tiles: 61 us before, 40 at P = 64, 31 at 32, 29 at 16; at
// 320x320 106, 87 and 98 us for 700,000 Gaussians; from 1024 tiles on P = 64
// is the fastest).
constexpr int kRowsBatch = 256;
constexpr int kRowsSmallBatch = 128;

template <int CH, int P>
__global__ void __launch_bounds__(256) raster_fwd_rows_kernel(RasterArgs a, int BB, int split,
                                                               float* __restrict__ render_colors,
                                                               float* __restrict__ render_alphas,
                                                               int32_t* __restrict__ last_ids) {
  using RB = RowBlock<P>;
  constexpr int FW = fwd_rows_record_words(CH);
  constexpr int MW = 6 + CH;  // word of the touch mask and class
  constexpr int PS = P + 4;  // alpha words per record: 16 records' rows start in distinct banks
  extern __shared__ float smem[];
  const int BS = blockDim.x;
  const int n_waves = BS / kWave;
  float* s_rec = smem;                                                    // [BB][FW]
  float* s_alpha = s_rec + BB * FW;                                       // [n_waves][16][PS]
  float4* s_col = reinterpret_cast<float4*>(s_alpha + n_waves * 16 * PS);  // [n_waves][16] colours (and entry)
  float4* s_rect = s_col + n_waves * 16;                                  // [n_waves]
  int* s_pos = reinterpret_cast<int*>(s_rect + n_waves);                  // [n_waves][16] entry (CH == 4)
  uint8_t* s_list = reinterpret_cast<uint8_t*>(s_pos + (CH == 4 ? n_waves * 16 : 0));  // [n_waves][BB]
  auto s_mask = [&](int k) { return __float_as_uint(s_rec[k * FW + MW]); };

  const int tx = blockIdx.x / split, ty = blockIdx.y;
  const int64_t image = blockIdx.z;
  const int tile = ty * a.tw + tx;
  const int t = threadIdx.x;
  const int lane = t % kWave;
  const int wave = t / kWave;
  const int wave0 = (blockIdx.x % split) * n_waves;  // this block's first wave of the tile
  const int bpr = a.ts / RB::BX;
  const int x = tx * a.ts + ((wave0 + wave) % bpr) * RB::BX + lane % RB::BX;
  const int y = ty * a.ts + ((wave0 + wave) / bpr) * RB::BY + (lane % P) / RB::BX;
  const bool inside = lane < P && x < a.W && y < a.H;
  const int64_t pix = (image * a.H + y) * static_cast<int64_t>(a.W) + x;
  const float* bg = a.backgrounds ? a.backgrounds + image * CH : nullptr;
  const int64_t n_tiles = static_cast<int64_t>(a.tw) * a.th;

  if (a.masks && !a.masks[image * n_tiles + tile]) {
    if (inside) {
      render_alphas[pix] = 0.0f;
#pragma unroll
      for (int c = 0; c < CH; ++c) render_colors[pix * CH + c] = bg ? bg[c] : 0.0f;
      last_ids[pix] = 0;
    }
    return;
  }
  int64_t start, end;
  tile_range(a, image, tile, &start, &end);
  if (t < n_waves) {
    const PixRect r = RB::rect(wave0 + t, a.ts, tx, ty);
    s_rect[t] = make_float4(r.x0, r.x1, r.y0, r.y1);
  }
  const PixRect wr = RB::rect(wave0 + wave, a.ts, tx, ty);
  const int ri = lane & 15, rk = lane >> 4;
  const float lx0 = wr.x0 + static_cast<float>(RB::x0(rk));
  const float py0 = wr.y0 + static_cast<float>(RB::y0(rk)), py1 = py0 + static_cast<float>(RB::HS);
  float* alpha_out = s_alpha + (wave * 16 + ri) * PS + RB::y0(rk) * RB::BX + RB::x0(rk);
  const float* alpha_in = s_alpha + wave * 16 * PS + lane % P;
  float4* wave_col = s_col + wave * 16;
  int* wave_pos = s_pos + wave * 16;
  uint8_t* list = s_list + wave * BB;

  // T > 0: the pixel's transmittance; T < 0: minus the final one (saturated,
  // or no pixel)
  float T = inside ? 1.0f : -1.0f;
  int32_t cur = 0;
  float acc[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) acc[c] = 0.0f;

  float2 r_xy = make_float2(0.0f, 0.0f);
  float4 r_co = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  float r_col[CH];
  auto load_records = [&](int64_t b0) {
    const int64_t j = b0 + t;
    if (t < BB && j < end) {
      const int32_t g = load_gaussian(a, j, &r_xy, &r_co);
#pragma unroll
      for (int c = 0; c < CH; ++c) r_col[c] = a.colors[static_cast<int64_t>(g) * CH + c];
    }
  };
  load_records(start);
  for (int64_t b0 = start; b0 < end; b0 += BB) {
    if (__syncthreads_count(T < 0.0f) == BS) break;  // also fences the previous batch's LDS reads
    if (t < BB && b0 + t < end) {
      float* rec = s_rec + t * FW;
      *reinterpret_cast<float4*>(rec) = make_float4(0.5f * r_co.x, r_co.y, 0.5f * r_co.z, r_co.w);
      float tail[FW - 4];
#pragma unroll
      for (int i = 0; i < FW - 4; ++i) tail[i] = 0.0f;
      tail[0] = r_xy.x;
      tail[1] = r_xy.y;
      bool finite = true;
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        tail[2 + c] = r_col[c];
        finite = finite && fabsf(r_col[c]) <= 3.402823466e38f;
      }
      tail[MW - 4] = __uint_as_float(touch_mask(r_xy, r_co, n_waves, s_rect) | record_class(r_xy, r_co) |
                                     (finite ? 0u : kNonFiniteRecord));
#pragma unroll
      for (int i = 0; i < FW - 4; i += 4)
        *reinterpret_cast<float4*>(rec + 4 + i) = make_float4(tail[i], tail[i + 1], tail[i + 2], tail[i + 3]);
    }
    __syncthreads();
    load_records(b0 + BB);
    const int cnt = static_cast<int>(min<int64_t>(BB, end - b0));
    int n = 0;
    if (__ballot(T > 0.0f) != 0) {
      for (int c0 = 0; c0 < cnt; c0 += kWave) {
        const int kl = c0 + lane;
        const bool mine = kl < cnt && ((s_mask(kl) >> wave) & 1u);
        const uint64_t bits = __ballot(mine);
        const int below = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(bits >> 32),
                                                    __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(bits), 0));
        if (mine) list[n + below] = static_cast<uint8_t>(kl);
        n += __popcll(bits);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int g0 = 0; g0 < n; g0 += 16) {
      const bool live = g0 + ri < n;
      const int slot = list[min(g0 + ri, n - 1)];
      const float* rec = s_rec + slot * FW;
      float4 co = reinterpret_cast<const float4*>(rec)[0];
      if (!live) co.w = 0.0f;  // alpha 0 past the list
      const float4 xc = reinterpret_cast<const float4*>(rec)[1];
      float4 ex = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if constexpr (FW > 8) ex = reinterpret_cast<const float4*>(rec)[2];
      const uint32_t bits = s_mask(slot);
      const int entry = static_cast<int>(b0) + slot;
      if (rk == 0) {
        wave_col[ri] = make_float4(xc.z, xc.w, ex.x, CH == 4 ? ex.y : __int_as_float(entry));
        if constexpr (CH == 4) wave_pos[ri] = entry;
      }
      const float dy[2] = {xc.y - py0, xc.y - py1};
      const float cy[2] = {co.z * dy[0] * dy[0], co.z * dy[1] * dy[1]};
      auto falloffs = [&](auto level_c) {
        constexpr int kLevel = decltype(level_c)::value;
        float px = lx0;
#pragma unroll
        for (int cx = 0; cx < RB::NX; cx += 2) {
          float al[2][2];
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            const float dx = xc.x - px;
            px += 1.0f;
            const float ax = co.x * dx * dx;
            const float bx = co.y * dx;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const float sigma = (ax + cy[h]) + bx * dy[h];  // halved_sigma's operations
              float alpha;
              bool pass;
              if constexpr (kLevel < 2) {
                alpha = co.w * exp_alpha_bounded(-sigma);
                if constexpr (kLevel == 1) alpha = fminf(kMaxAlpha, alpha);
                pass = alpha >= kAlphaThreshold;
              } else {
                alpha = fminf(kMaxAlpha, co.w * exp_alpha(-sigma));
                pass = live && !(sigma < 0.0f || alpha < kAlphaThreshold);
              }
              al[h][p] = pass ? alpha : 0.0f;
            }
          }
#pragma unroll
          for (int h = 0; h < 2; ++h)
            *reinterpret_cast<float2*>(alpha_out + cx + h * RB::HS * RB::BX) = make_float2(al[h][0], al[h][1]);
        }
      };
      if (__ballot(live && (bits & kCappedRecord)) == 0) {
        falloffs(std::integral_constant<int, 0>{});
      } else if (__ballot(live && (bits & kGeneralRecord)) == 0) {
        falloffs(std::integral_constant<int, 1>{});
      } else {
        falloffs(std::integral_constant<int, 2>{});
      }
      const bool finite = __ballot(live && (bits & kNonFiniteRecord)) == 0;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // alphas and colours: written and read by this wave
      // The group's records in list order, one pixel per lane, four at a time.
      // The transmittance chain is one product per record: it never rises, so
      // each record's test against the threshold stands alone.
      auto composite4 = [&](int k0, auto careful_c) {
        constexpr bool kCareful = decltype(careful_c)::value;
        float al[4], tb[4], ta = T;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          al[k] = alpha_in[(k0 + k) * PS];
          tb[k] = ta;
          ta *= 1.0f - al[k];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float4 col = wave_col[k0 + k];
          const float next_T = k < 3 ? tb[k < 3 ? k + 1 : 3] : ta;
          const bool keep = next_T > kTransmittanceThreshold;
          const float vis = keep ? al[k] * tb[k] : 0.0f;
          T = keep ? next_T : -fabsf(T);
          const bool take = vis > 0.0f;
          const float cc[4] = {col.x, col.y, col.z, col.w};
#pragma unroll
          for (int c = 0; c < CH; ++c) {
            const float v = __builtin_fmaf(cc[c], vis, acc[c]);
            acc[c] = !kCareful || take ? v : acc[c];
          }
          cur = take ? (CH == 4 ? wave_pos[k0 + k] : __float_as_int(col.w)) : cur;
        }
      };
      const int m = min(16, n - g0);
      if (finite) {
#pragma unroll
        for (int k = 0; k < 16; k += 4)
          if (k < m) composite4(k, std::false_type{});
      } else {
        for (int k = 0; k < m; k += 4) composite4(k, std::true_type{});
      }
      if (__ballot(T > 0.0f) == 0) break;  // every pixel of the wave has saturated
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }
  if (!inside) return;
  T = fabsf(T);
  render_alphas[pix] = 1.0f - T;
#pragma unroll
  for (int c = 0; c < CH; ++c) render_colors[pix * CH + c] = acc[c] + T * (bg ? bg[c] : 0.0f);
  last_ids[pix] = cur;
}

// Wave-wide sums of N values per lane by transposition (gfx950): three
// exchange levels halve the number of live values while doubling the lanes
// each one covers -- permlane32_swap (lane ^ 32), permlane16_swap (lane ^ 16),
// DPP row_ror:8 (lane ^ 8) -- then quad_perm / row_half_mirror DPP adds finish
// the sums inside each group of 8 lanes. A pair (a, b) at a level leaves the
// sum of a on lanes whose level bit is 0 and of b where it is 1; an unpaired
// last value is summed on its bit-0 side only at the permlane levels (its
// partner register holds a dead value) and on both sides at the DPP level. After the call, value y[m] on a lane with bits
// h = lane[5], r = lane[4], e = lane[3] is the wave total of input
// red_index<N>(m, h, r, e) (N: not a total, to be discarded); all 8 lanes of
// a group hold the same values.
// Costs about 2.3 VALU per value instead of 6 DPP steps per value.
template <int N>
struct Red {
  static constexpr int NA = (N + 1) / 2;   // after lane ^ 32
  static constexpr int NB = (NA + 1) / 2;  // after lane ^ 16
  static constexpr int NC = (NB + 1) / 2;  // after lane ^ 8
};

// Input index of y[m] on a lane with bits (h, r, e), or N where that lane's
// y[m] is not a total: an unpaired value at the permlane levels is exchanged
// with a dead register (no copy), so only its bit-0 side holds its sum.
template <int N>
__device__ __forceinline__ int red_index(int m, int h, int r, int e) {
  int c = 2 * m + e;
  if (c >= Red<N>::NB) c = 2 * m;
  const int b = 2 * c + r;
  if (b >= Red<N>::NA) return N;
  const int v = 2 * b + h;
  return v < N ? v : N;
}

__device__ __forceinline__ float fbits(unsigned u) { return __builtin_bit_cast(float, u); }
__device__ __forceinline__ unsigned ubits(float f) { return __builtin_bit_cast(unsigned, f); }

template <int N>
__device__ __forceinline__ void wave_transpose_reduce(const float (&v)[N], float (&y)[Red<N>::NC], bool e_bit) {
  constexpr int NA = Red<N>::NA, NB = Red<N>::NB, NC = Red<N>::NC;
  static_assert(N >= 3, "the unpaired exchange reuses the previous pair's register");
  // the unpaired value's partner is the previous pair's second swap output,
  // dead once added, so no register is copied for it
  float w[NA];
  unsigned spare = 0u;
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const unsigned b = (2 * i + 1 < N) ? ubits(v[2 * i + 1]) : spare;
    const auto sw = __builtin_amdgcn_permlane32_swap(ubits(v[2 * i]), b, false, false);
    w[i] = fbits(sw[0]) + fbits(sw[1]);
    spare = sw[1];
  }
  float x[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const unsigned b = (2 * i + 1 < NA) ? ubits(w[2 * i + 1]) : spare;
    const auto sw = __builtin_amdgcn_permlane16_swap(ubits(w[2 * i]), b, false, false);
    x[i] = fbits(sw[0]) + fbits(sw[1]);
    spare = sw[1];
  }
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const float a = x[2 * i];
    if (2 * i + 1 < NB) {
      const float b = x[2 * i + 1];
      const float send = e_bit ? a : b;
      const float keep = e_bit ? b : a;
      y[i] = keep + fbits(__builtin_amdgcn_update_dpp(0u, ubits(send), 0x128, 0xf, 0xf, false));  // row_ror:8
    } else {
      y[i] = a + fbits(__builtin_amdgcn_update_dpp(0u, ubits(a), 0x128, 0xf, 0xf, false));
    }
  }
#pragma unroll
  for (int i = 0; i < NC; ++i) y[i] += fbits(__builtin_amdgcn_update_dpp(0u, ubits(y[i]), 0xB1, 0xf, 0xf, false));   // lane ^ 1
#pragma unroll
  for (int i = 0; i < NC; ++i) y[i] += fbits(__builtin_amdgcn_update_dpp(0u, ubits(y[i]), 0x4E, 0xf, 0xf, false));   // lane ^ 2
#pragma unroll
  for (int i = 0; i < NC; ++i) y[i] += fbits(__builtin_amdgcn_mov_dpp(ubits(y[i]), 0x141, 0xf, 0xf, true));  // 7 - lane
}

// Backward. One block per tile, in the heavy-first tile order of `order`
// (see below); one lane owns one pixel of the tile (blocks are padded to
// whole wave64s; padding lanes own nothing). The tile's list is walked
// back-to-front in batches of BB entries from the tile's largest last_id; the
// next batch's records are loaded into registers while the current one is
// processed, and each staged record carries its per-wave touch mask. For each
// entry a wave visits (ballot over 64 slots, past-last and culled entries
// skipped), every lane computes its pixel's partial gradients in a reduced
// basis (below); a wave with a contributing lane sums them over the wave
// (wave_transpose_reduce) and one lane per 8-lane group stores its totals
// into the wave's accumulator slot for that entry (plain LDS stores; each
// (wave, entry) slot is written at most once per batch). After the batch the
// block adds up the per-wave slots, maps them back to gradients and flushes
// one global atomic per (entry, nonzero component).
//
// Per pixel, with the reference's per-channel `buffer` (gsplat_rasterize.cpp:
// 500-546) folded into B = sum_c buffer_c * v_rc_c and D = sum_c col_c * v_rc_c:
//   v_alpha = T D + ra (coef - B),  B += fac D,
// and the geometry gradients accumulated as h = v_sigma * (dx, dy):
//   v_conic = (hx dx / 2, hx dy, hy dy / 2),  v_mean2d = conic * (sum hx, sum hy)
// (the conic is the same for every pixel of an entry, so it is applied once
// after the reduction). Accumulated components: colors (CH), hx dx, hx dy,
// hy dy, hx, hy, vis * v_alpha, and |v_mean2d| per pixel (x, y) with absgrad.
// The contribution is computed on every lane of a visiting wave and selected
// to zero where the pixel does not contribute (no branches, no accumulators
// to clear). CH == 0 (runtime channel count) sends colour gradients straight
// to global memory.
// Six waves per SIMD (at most 80 VGPRs) where that needs no spills: one to
// three channels without absgrad; the register need leaves the others as they
// are.
constexpr int bwd_min_waves(int ch, bool abs) { return (!abs && ch >= 1 && ch <= 3) ? 6 : 1; }
// s_waitcnt immediate (gfx9 encoding): vmcnt 0 (bits 3:0 and 15:14), expcnt 7
// (bits 6:4) and lgkmcnt 15 (bits 11:8), i.e. wait for vector memory only
constexpr int kWaitVmemOnly = 0x0F70;
// flush lanes per entry (output components: CH colours, 3 conic, 2 mean, 1
// opacity, 2 |mean| with absgrad: at most 12) and the kinds of component
constexpr int kFlushLanes = 16;
constexpr int kFlushPlain = 0, kFlushMean = 1, kFlushOpacity = 2;

template <int CH, bool ABS>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(bwd_min_waves(CH, ABS))))
raster_bwd_kernel(
    RasterArgs a, int BB, int64_t n_units, const int32_t* __restrict__ order, const int32_t* __restrict__ cost,
    const float* __restrict__ render_alphas, const int32_t* __restrict__ last_ids,
    const float* __restrict__ v_render_colors, const float* __restrict__ v_render_alphas,
    float* __restrict__ v_means2d_abs, float* __restrict__ v_means2d, float* __restrict__ v_conics,
    float* __restrict__ v_colors, float* __restrict__ v_opacities, float* __restrict__ v_backgrounds) {
  constexpr int LC = CH > 0 ? CH : 1;
  constexpr int AC = CH > 0 ? CH : kMaxChannels;
  constexpr int NG = ABS ? 8 : 6;  // geometry components
  constexpr int NV = (CH > 0 ? CH : 0) + NG;
  constexpr int o = CH > 0 ? CH : 0;  // first geometry component
  constexpr int NC = Red<2 * NV>::NC;  // sums per lane of a record pair's reduction
  constexpr int NS = NV + 1;  // accumulator words per (wave, slot); the last takes discarded values
  constexpr int RW = bwd_record_words(CH);
  extern __shared__ float smem[];
  const int BS = blockDim.x;
  const int n_waves = BS / kWave;
  // one record per batch slot, read through a single address: conic xyz +
  // opacity, mean xy, colours (CH > 0), Gaussian id, per-wave touch bits
  constexpr int GW = 6 + o;  // word of the Gaussian id; the touch mask follows
  float* s_rec = smem;                  // [BB][RW]
  float* s_acc = smem + RW * BB;        // [n_waves][BB][NS]
  float4* s_rect = reinterpret_cast<float4*>(s_acc + n_waves * BB * NS);  // [n_waves] wave pixel rects
  auto s_g = [&](int k) { return __float_as_int(s_rec[k * RW + GW]); };
  auto s_mask = [&](int k) { return __float_as_uint(s_rec[k * RW + GW + 1]); };

  const int channels = CH > 0 ? CH : a.channels;
  const int t = threadIdx.x;
  const int lane = t % kWave;
  const int wave = t / kWave;
  const bool e_bit = (lane >> 3) & 1;
  const bool red_slot = (lane & 7) == 7;  // lane 7 of each 8-lane group stores
  const bool second_half = (lane >> 5) & 1;  // holds the pair's second record's sums
  // this lane's accumulator words for entry slot 0 (slot k adds k * NS): the
  // pair reduction's input 2 i + h is component i of record h, h = lane bit 5;
  // inputs that are not totals on this lane go to the discard word NV
  float* red_at[NC];
#pragma unroll
  for (int m = 0; m < NC; ++m) {
    const int in = red_index<2 * NV>(m, (lane >> 5) & 1, (lane >> 4) & 1, (lane >> 3) & 1);
    red_at[m] = s_acc + wave * BB * NS + (in < 2 * NV ? in / 2 : NV);
  }
  const int64_t n_tiles = static_cast<int64_t>(a.tw) * a.th;
  const int acc_words = n_waves * BB * NS;
  // this thread's flush role (the same for every slot it flushes, as the
  // block size is a multiple of kFlushLanes): output component c = t % 16 of
  // an entry, read from accumulator word(s) fl_word0 (fl_word1) and added to
  // fl_base[g * fl_stride + fl_comp]
  const int fc = t % kFlushLanes;
  int fl_word0 = -1, fl_word1 = -1, fl_kind = kFlushPlain, fl_comp = 0, fl_stride = 1;
  float fl_scale = 1.0f;
  float* fl_base = v_opacities;
  if (fc < (CH > 0 ? CH : 0)) {
    fl_word0 = fc, fl_base = v_colors, fl_stride = CH, fl_comp = fc;
  } else if (fc < o + 3) {
    fl_word0 = fc, fl_base = v_conics, fl_stride = 3, fl_comp = fc - o, fl_scale = fc - o == 1 ? 1.0f : 0.5f;
  } else if (fc < o + 5) {
    fl_word0 = o + 3, fl_word1 = o + 4, fl_kind = kFlushMean, fl_base = v_means2d, fl_stride = 2, fl_comp = fc - o - 3;
  } else if (fc == o + 5) {
    fl_word0 = o + 5, fl_kind = kFlushOpacity, fl_base = v_opacities;
  } else if (ABS && fc < o + 8) {
    fl_word0 = fc, fl_base = v_means2d_abs, fl_stride = 2, fl_comp = fc - o - 6;
  }

  // One block per tile, launched in the cost-sorted order: block b takes the
  // tile at rank b. The dispatcher starts blocks in index order as resident
  // blocks finish, so the heaviest tiles start first and the launch ends on
  // the lightest (longest-first balancing done by the hardware; a persistent
  // grid dealing about three tiles per block, statically or from a shared
  // counter, left CUs idle while their last blocks finished).
  {
    const int64_t unit = blockIdx.x;
    if (unit >= n_units) return;  // uniform across the block
    const int64_t it = order[unit];
    const int64_t image = it / n_tiles;
    const int tile = static_cast<int>(it % n_tiles);
    const int tx = tile % a.tw, ty = tile / a.tw;
    // masked tiles contribute nothing; their cost is 0, so the walk is empty
    int64_t start, end;
    tile_range(a, image, tile, &start, &end);
    // the tile's replay length (largest last_id - start + 1) from the schedule
    // pass; the first batch is fetched before the pixel state is read
    const int64_t stop = start + cost[it];
    // Register pipeline of batch records (lanes t < BB; slot t of the batch
    // [lo, hi) holds entry hi - 1 - t, back to front): the flatten ids are
    // loaded two batches ahead and the records one batch ahead, and nothing
    // waits for them until the batch is staged, where the touch mask is
    // formed. Ids outside [0, G) stage a zero-opacity record (never
    // contributes) and no colour read.
    int32_t r_id = 0;
    float2 r_xy = make_float2(0.0f, 0.0f);
    float4 r_co = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    int32_t r_g = 0;
    float r_col[LC];
    auto load_ids = [&](int64_t hi, int64_t lo) {
      const int64_t j = hi - 1 - t;
      if (t < BB && j >= lo) r_id = a.flatten_ids[j];
    };
    auto load_records = [&](int64_t hi, int64_t lo) {  // of the ids in r_id
      const int64_t j = hi - 1 - t;
      if (t < BB && j >= lo) {
        const int32_t g = r_id;
        const bool ok = g >= 0 && static_cast<int64_t>(g) < a.G;
        const int64_t gg = ok ? g : 0;
        r_g = ok ? g : 0;
        if (ok) {
          r_xy = make_float2(a.means2d[gg * 2], a.means2d[gg * 2 + 1]);
          r_co = make_float4(a.conics[gg * 3], a.conics[gg * 3 + 1], a.conics[gg * 3 + 2], a.opacities[gg]);
        } else {
          r_xy = make_float2(0.0f, 0.0f);
          r_co = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        if constexpr (CH > 0) {
#pragma unroll
          for (int c = 0; c < CH; ++c) r_col[c] = ok ? a.colors[gg * CH + c] : 0.0f;
        }
      }
    };
    if (stop > start) {
      const int64_t lo0 = max<int64_t>(start, stop - BB);
      load_ids(stop, lo0);
      load_records(stop, lo0);
      if (lo0 > start) load_ids(lo0, max<int64_t>(start, lo0 - BB));
    }

    store_wave_rects(s_rect, n_waves, a.ts, tx, ty);  // read after the batch loop's first barrier
    int qx, qy;
    lane_pixel(t, a.ts, &qx, &qy);
    const int x = tx * a.ts + qx;
    const int y = ty * a.ts + qy;
    const bool inside = t < a.ts * a.ts && x < a.W && y < a.H;
    const int64_t pix = (image * a.H + y) * static_cast<int64_t>(a.W) + x;
    const float px = static_cast<float>(x) + 0.5f;
    const float py = static_cast<float>(y) + 0.5f;
    const float T_final = inside ? 1.0f - render_alphas[pix] : 1.0f;
    float T = T_final;
    int last_rel = -1;  // last contributor relative to start, -1 for none
    if (inside) {
      const int64_t l = min<int64_t>(end - 1, last_ids[pix]) - start;
      last_rel = static_cast<int>(max<int64_t>(-1, min<int64_t>(l, INT32_MAX)));
    }
    float v_rc[AC];
    float bg_dot = 0.0f;
    for (int c = 0; c < channels; ++c) v_rc[c] = inside ? v_render_colors[pix * channels + c] : 0.0f;
    const float v_ra = inside && v_render_alphas ? v_render_alphas[pix] : 0.0f;
    if (a.backgrounds) {
      const float* bg = a.backgrounds + image * channels;
      for (int c = 0; c < channels; ++c) bg_dot += bg[c] * v_rc[c];
    }
    // d(final-transmittance terms)/d(alpha) = ra * coef
    const float coef = T_final * v_ra + -T_final * bg_dot;
    float Bc = coef;  // coef - B, B the running colour buffer (starts at 0)
    // the wave's colour cotangents and final transmittances are all finite
    // (then a lane that does not contribute can add fac * v_rc = 0 without a
    // select)
    bool rc_finite = fabsf(T_final) <= 3.402823466e38f;
    for (int c = 0; c < channels; ++c) rc_finite = rc_finite && fabsf(v_rc[c]) <= 3.402823466e38f;
    const bool wave_rc_finite = __ballot(!rc_finite) == 0;
    // entries past every pixel of the wave's last contributor are skipped
    int wave_last = last_rel;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) wave_last = max(wave_last, __shfl_xor(wave_last, off, kWave));


    for (int64_t b1 = stop; b1 > start; b1 -= BB) {
      const int64_t b0 = max<int64_t>(start, b1 - BB);
      __syncthreads();  // previous batch fully consumed and flushed
      if (t < BB && b1 - 1 - t >= b0) {
        const uint32_t r_mask = touch_mask(r_xy, r_co, n_waves, s_rect);
        float* rec = s_rec + t * RW;
        // conic diagonal pre-halved, as in the forward (the same sigma bit for
        // bit); the flush and the absolute gradients double it back exactly
        *reinterpret_cast<float4*>(rec) = make_float4(0.5f * r_co.x, r_co.y, 0.5f * r_co.z, r_co.w);
        float tail[RW - 4];
#pragma unroll
        for (int i = 0; i < RW - 4; ++i) tail[i] = 0.0f;
        tail[0] = r_xy.x;
        tail[1] = r_xy.y;
        if constexpr (CH > 0) {
#pragma unroll
          for (int c = 0; c < CH; ++c) tail[2 + c] = r_col[c];
        }
        tail[GW - 4] = __int_as_float(r_g);
        bool rec_finite = fabsf(r_xy.x) <= 3.402823466e38f && fabsf(r_xy.y) <= 3.402823466e38f;
        if constexpr (CH > 0) {
#pragma unroll
          for (int c = 0; c < CH; ++c) rec_finite = rec_finite && fabsf(r_col[c]) <= 3.402823466e38f;
        }
        tail[GW - 3] = __uint_as_float(r_mask | (rec_finite ? 0u : kNonFiniteRecord));
#pragma unroll
        for (int i = 0; i < RW - 4; i += 4)
          *reinterpret_cast<float4*>(rec + 4 + i) = make_float4(tail[i], tail[i + 1], tail[i + 2], tail[i + 3]);
      }
      // acc_words is a multiple of 4 (BB is a multiple of 64)
      for (int w = t * 4; w < acc_words; w += BS * 4)
        *reinterpret_cast<float4*>(s_acc + w) = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      __syncthreads();
      // the next batch's records and the ids of the batch after it, in flight
      // during this one
      if (b0 > start) {
        const int64_t lo1 = max<int64_t>(start, b0 - BB);
        load_records(b0, lo1);
        if (lo1 > start) load_ids(lo1, max<int64_t>(start, lo1 - BB));
      }
      const int cnt = static_cast<int>(b1 - b0);
      const int k_rel0 = static_cast<int>(b1 - 1 - start);  // entry of slot 0, relative to start
      // Visits come in pairs of straight-line code so that the two records'
      // falloff, alpha and gradient terms overlap and their wave sums are
      // one reduction; only transmittance T and the buffer (Bc) pass from the
      // first visit to the second (list order, back to front). A chunk with
      // an odd number of visits ends with an inert second visit: no lane
      // valid, its sums not stored.
      struct Fall {
        float dx, dy, vis, a_raw, alpha;
        bool valid;
      };
      // falloff of this lane's pixel under the record of slot k (co: conic +
      // opacity, xc: mean xy + colours 0-1, ex: colours 2-3 when CH > 2)
      auto falloff = [&](int k, const float4& co, const float4& xc) {
        Fall f;
        const int k_rel = k_rel0 - k;
        f.dx = xc.x - px;
        f.dy = xc.y - py;
        const float sigma = (co.x * f.dx * f.dx + co.z * f.dy * f.dy) + co.y * f.dx * f.dy;  // co.x, co.z pre-halved
        f.vis = exp_alpha(-sigma);
        f.a_raw = co.w * f.vis;
        f.alpha = fminf(kMaxAlpha, f.a_raw);
        f.valid = k_rel <= last_rel && !(sigma < 0.0f || f.alpha < kAlphaThreshold);
        return f;
      };
      // this lane's partial gradients for slot k (v, reduced by the caller)
      auto contribute = [&](int k, const float4& co, const float4& xc, const float4& ex, const Fall& f,
                            bool store, bool careful, float (&v)[NV]) {
        const bool valid = f.valid;
        // A lane that does not contribute takes ra = 1 and alpha = 0, so T
        // stays exactly T and fac is 0; the geometry terms are still
        // selected, and (careful: the chunk holds a record with a non-finite
        // mean or colour, or the wave a non-finite colour cotangent) so are
        // the colour terms, the buffer update and the offsets, so non-finite
        // values of the record or of a pixel's cotangent never reach another
        // pixel's sums. Otherwise D is finite and fac D is exactly 0 for such
        // a lane, which leaves the buffer as it is without a select.
        const float ra = valid ? __builtin_amdgcn_rcpf(fmaxf(kMinOneMinusAlpha, 1.0f - f.alpha)) : 1.0f;
        const float T_new = T * ra;
        const float fac = (valid ? f.alpha : 0.0f) * T_new;
        float D;
        if constexpr (CH > 0) {
          D = xc.z * v_rc[0];
          v[0] = (careful && !valid) ? 0.0f : fac * v_rc[0];
#pragma unroll
          for (int c = 1; c < CH; ++c) {
            const float colc = c == 1 ? xc.w : (c == 2 ? ex.x : ex.y);
            D = __builtin_fmaf(colc, v_rc[c], D);
            v[c] = (careful && !valid) ? 0.0f : fac * v_rc[c];
          }
        } else {
          const int64_t gg = s_g(k);
          const float* gcol = a.colors + gg * channels;
          D = 0.0f;
          for (int c = 0; c < channels; ++c) D = __builtin_fmaf(gcol[c], v_rc[c], D);
          for (int c = 0; c < channels; ++c) {
            const float sum = wave_sum_uniform(valid ? fac * v_rc[c] : 0.0f);
            if (store && lane == 0 && sum != 0.0f) unsafeAtomicAdd(v_colors + gg * channels + c, sum);
          }
        }
        // Bc = coef - B, the reference's (coef - B) with B its running buffer
        const float v_alpha = __builtin_fmaf(T_new, D, ra * Bc);
        Bc = (CH == 0 || careful) ? (valid ? __builtin_fmaf(-fac, D, Bc) : Bc) : __builtin_fmaf(-fac, D, Bc);
        T = T_new;
        const bool geo = valid && f.a_raw <= kMaxAlpha;
        const float v_sigma = geo ? -f.a_raw * v_alpha : 0.0f;
        const float gx = (careful && !geo) ? 0.0f : f.dx;
        const float gy = (careful && !geo) ? 0.0f : f.dy;
        const float hx = v_sigma * gx;
        const float hy = v_sigma * gy;
        v[o + 0] = hx * gx;
        v[o + 1] = hx * gy;
        v[o + 2] = hy * gy;
        v[o + 3] = hx;
        v[o + 4] = hy;
        // vis v_alpha = -v_sigma / opacity: the flush divides the sum once
        v[o + 5] = v_sigma;
        if constexpr (ABS) {
          v[o + 6] = geo ? fabsf(__builtin_fmaf(co.x + co.x, hx, co.y * hy)) : 0.0f;
          v[o + 7] = geo ? fabsf(__builtin_fmaf(co.y, hx, (co.z + co.z) * hy)) : 0.0f;
        }
      };
      auto load = [&](int k, float4& co, float4& xc, float4& ex) {
        const float4* rec = reinterpret_cast<const float4*>(s_rec + k * RW);
        co = rec[0];
        xc = rec[1];
        if constexpr (RW > 8) ex = rec[2];
      };
      for (int c0 = 0; c0 < cnt; c0 += kWave) {
        // slots of this chunk that may touch this wave and are not past its
        // last contributor (all lanes vote)
        const int kl = c0 + lane;
        const uint32_t mk = kl < cnt ? s_mask(kl) : 0u;
        const bool mine = k_rel0 - kl <= wave_last && ((mk >> wave) & 1u);
        uint64_t bits = __ballot(mine);
        const bool careful = !wave_rc_finite || __ballot(mine && (mk & kNonFiniteRecord)) != 0;
        while (bits) {
          const int k1 = c0 + __builtin_ctzll(bits);
          bits &= bits - 1;
          const bool two = bits != 0;
          const int k2 = two ? c0 + __builtin_ctzll(bits) : k1;
          bits &= bits - 1;
          float4 co1, xc1, ex1 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
          float4 co2, xc2, ex2 = ex1;
          load(k1, co1, xc1, ex1);
          load(k2, co2, xc2, ex2);
          const Fall f1 = falloff(k1, co1, xc1);
          Fall f2 = falloff(k2, co2, xc2);
          f2.valid = f2.valid && two;
          float v1[NV], v2[NV];
          if (careful) {
            contribute(k1, co1, xc1, ex1, f1, true, true, v1);
            contribute(k2, co2, xc2, ex2, f2, two, true, v2);
          } else {
            contribute(k1, co1, xc1, ex1, f1, true, false, v1);
            contribute(k2, co2, xc2, ex2, f2, two, false, v2);
          }
          // interleaved, so lanes 0-31 end with the first record's sums and
          // lanes 32-63 with the second's
          float vv[2 * NV], y[NC];
#pragma unroll
          for (int i = 0; i < NV; ++i) {
            vv[2 * i] = v1[i];
            vv[2 * i + 1] = v2[i];
          }
          wave_transpose_reduce<2 * NV>(vv, y, e_bit);
          if (red_slot && (two || !second_half)) {
            // 24-bit multiply: full rate, unlike a 32-bit one (slots < BB)
            const int off = __mul24(second_half ? k2 : k1, NS);
#pragma unroll
            for (int mm = 0; mm < NC; ++mm) red_at[mm][off] = y[mm];
          }
        }
      }
      __syncthreads();
      // The vector memory counter counts loads, stores and atomics in issue
      // order, so the loaders' wait for the next batch's records (issued
      // before the visits) would also wait for the atomics below. Waiting for
      // vector memory here, before the atomics, leaves those records ready.
      __builtin_amdgcn_s_waitcnt(kWaitVmemOnly);
      // Flush: 16 lanes per slot, lane c of the group adds output component
      // c of the slot's entry (summed over the waves), so one atomic
      // instruction covers four entries and each entry's colours, conic and
      // mean are each one cache line: the memory system serves atomics per
      // cache line, whatever the number of lanes that hit it.
      for (int idx = t; idx < cnt * kFlushLanes; idx += BS) {
        const int slot = idx / kFlushLanes;
        if (fl_word0 < 0) continue;  // lanes past the slot's components
        float v = 0.0f, v2 = 0.0f;
        for (int w = 0; w < n_waves; ++w) {
          v += s_acc[(w * BB + slot) * NS + fl_word0];
          if (fl_word1 >= 0) v2 += s_acc[(w * BB + slot) * NS + fl_word1];
        }
        const int64_t gg = s_g(slot);
        if (fl_kind == kFlushMean) {
          // v_mean2d = conic (sum hx, sum hy); the conic applies only to
          // geometry terms some pixel produced: with none, the reference adds
          // nothing, even for a non-finite conic (0 * NaN would otherwise
          // reach the mean's gradient)
          if (v == 0.0f && v2 == 0.0f) continue;
          const float4 co = *reinterpret_cast<const float4*>(s_rec + slot * RW);
          v = fl_comp == 0 ? (co.x + co.x) * v + co.y * v2 : co.y * v + (co.z + co.z) * v2;
        } else if (fl_kind == kFlushOpacity) {
          // sum of v_sigma = -opacity vis v_alpha: the opacity is at least
          // 1/255 wherever a pixel contributed (alpha passed the threshold)
          if (v == 0.0f) continue;
          v = -v / s_rec[slot * RW + 3];
        } else {
          v *= fl_scale;
        }
        if (v != 0.0f) unsafeAtomicAdd(fl_base + gg * fl_stride + fl_comp, v);
      }
    }
  }
}

// Inclusive prefix product / sum over each row of 16 lanes, four independent
// values at a time: DPP row shifts by 1, 2, 4, 8 in place, a lane without a
// source keeps its value. The four chains are interleaved, so each DPP read
// comes at least two wait states after the write it depends on (the s_nop
// covers the values' producers).
#define GSPLAT_ROW_STEP(OP, SH)                              \
  OP " %0, %0, %0 row_shr:" SH " row_mask:0xf bank_mask:0xf\n\t" \
  OP " %1, %1, %1 row_shr:" SH " row_mask:0xf bank_mask:0xf\n\t" \
  OP " %2, %2, %2 row_shr:" SH " row_mask:0xf bank_mask:0xf\n\t" \
  OP " %3, %3, %3 row_shr:" SH " row_mask:0xf bank_mask:0xf\n\t"
__device__ __forceinline__ void row16_product4(float (&v)[4]) {
  asm("s_nop 1\n\t" GSPLAT_ROW_STEP("v_mul_f32_dpp", "1") GSPLAT_ROW_STEP("v_mul_f32_dpp", "2")
          GSPLAT_ROW_STEP("v_mul_f32_dpp", "4") GSPLAT_ROW_STEP("v_mul_f32_dpp", "8")
      : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
}
// v: inclusive sums; before: each lane's exclusive sum (the previous lane's
// inclusive one), lane 0 of the row keeps the value it came with.
__device__ __forceinline__ void row16_sum4(float (&v)[4], float (&before)[4]) {
  asm("s_nop 1\n\t" GSPLAT_ROW_STEP("v_add_f32_dpp", "1") GSPLAT_ROW_STEP("v_add_f32_dpp", "2")
          GSPLAT_ROW_STEP("v_add_f32_dpp", "4") GSPLAT_ROW_STEP("v_add_f32_dpp", "8")
      "v_mov_b32_dpp %4, %0 row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_mov_b32_dpp %5, %1 row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_mov_b32_dpp %6, %2 row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_mov_b32_dpp %7, %3 row_shr:1 row_mask:0xf bank_mask:0xf\n\t"
      : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(before[0]), "+v"(before[1]), "+v"(before[2]),
        "+v"(before[3]));
}
#undef GSPLAT_ROW_STEP

// Backward with records in lanes: tile sides 8, 16 and 24, one to four channels,
// no absolute gradients, lists long enough (bwd_rows_faster). Block, schedule,
// staging and flush are raster_bwd_kernel's; a wave still owns an 8x8 block of
// pixels, but evaluates 16 records at a time: lane l holds record l % 16 of
// the group (in list order, back to front) and the pixel rows l / 16 and
// l / 16 + 4, and steps over the 8 columns.
// - A record's gradient sums stay in its lane's registers over all the wave's
//   pixels; one exchange over the four rows per group replaces a 64-lane
//   reduction per record.
// - The pixel recurrences run across the 16 lanes instead of over time: T is a
//   prefix product of 1 / (1 - alpha) and the buffer a prefix sum, four DPP
//   steps each; lane 0 brings the pixel's state in, lane 15 leaves it in LDS.
// - A column's (0.5 c0 dx) dx and c1 dx serve both of the lane's rows, a
//   row's (0.5 c2 dy) dy all eight columns; sigma keeps the forward's operations
//   and rounding. Sums over y need no per-pixel products: with S and Hx the
//   sums of v_sigma and v_sigma dx over one row, sum v_sigma dy = S dy.
// - Groups without capped or general records (see above) skip the cap's and
//   sigma's tests.
// - The waves add their sums to one slot per entry in double (LDS atomics), so
//   the order in which waves arrive hardly ever shows in the rounded result.
//
// - While entries remain before a batch, a wave evaluates whole groups only;
//   the next batch starts at the first entry some wave left over (each wave
//   skips what it has done, and the entries' sums move along, so an entry is
//   flushed once). Groups then hold the same records whatever the
//   tile's list holds beside them, so the same pixels' recurrences round the
//   same with AABB and ellipse lists.
//
// Bound by VALU issue (0.98 of the issue slots at 1M Gaussians, 1297x840):
// 46 instructions per 64 (pixel, record) evaluations and about 10 around them,
// against 78 of the kernel with pixels in lanes. There 313 -> 231 us; 4.12 ->
// 3.23 ms over 8 images of 1920x1080, 470 -> 343 us for large faint splats,
// 114 -> 81 us at 512x512. About 120 VGPRs hold four evaluations in flight
// (their scans interleave without wait states); at five waves per SIMD (96
// VGPRs) the loop spills, 293 us, and unrolled further it does at four.
//
// kTameColor, kTameBuffer: bounds of the colours (and their cotangents) and of
// the entering buffer for which levels 0 and 1 run. Up to four products of a
// colour and a cotangent, their sums weighted by at most 1 in all, the entering
// buffer and its 1 / (1 - alpha) <= 100 fold then stay below 1e33, so v_alpha is
// finite at every pixel.
constexpr float kTameColor = 1.0e15f, kTameBuffer = 1.0e30f;
constexpr int kNeutral = 40;  // entries of the neutral state: columns 0-7 of two rows 32 apart

template <int CH>
__global__ void __launch_bounds__(576) __attribute__((amdgpu_waves_per_eu(4))) raster_bwd_rows_kernel(
    RasterArgs a, int BB, int64_t n_units, const int32_t* __restrict__ order, const int32_t* __restrict__ cost,
    const float* __restrict__ render_alphas, const int32_t* __restrict__ last_ids,
    const float* __restrict__ v_render_colors, const float* __restrict__ v_render_alphas,
    float* __restrict__ v_means2d, float* __restrict__ v_conics, float* __restrict__ v_colors,
    float* __restrict__ v_opacities) {
  constexpr int NV = CH + 6;
  constexpr int NS = NV | 1;  // accumulator words per slot (odd: no bank conflicts between records)
  constexpr int RW = bwd_record_words(CH);
  constexpr int GW = 6 + CH;
  extern __shared__ float smem[];
  const int BS = blockDim.x;
  const int n_waves = BS / kWave;
  double* s_acc = reinterpret_cast<double*>(smem);                  // [BB][NS]
  float4* s_pix = reinterpret_cast<float4*>(s_acc + BB * NS + (BB * NS & 1));  // [BS] colour cotangents (and last id)
  float2* s_state = reinterpret_cast<float2*>(s_pix + BS);          // [BS] T, Bc
  int* s_last = reinterpret_cast<int*>(s_state + BS);               // [BS]
  float2* s_neutral = reinterpret_cast<float2*>(s_last + (CH == 4 ? BS : 0));  // [kNeutral] (1, 0)
  float* s_rec = reinterpret_cast<float*>(s_neutral + kNeutral);          // [BB][RW]
  float4* s_rect = reinterpret_cast<float4*>(s_rec + RW * BB);      // [n_waves]
  int* s_next = reinterpret_cast<int*>(s_rect + n_waves);           // [n_waves]
  uint16_t* s_list = reinterpret_cast<uint16_t*>(s_next + n_waves); // [n_waves][BB]
  auto s_g = [&](int k) { return __float_as_int(s_rec[k * RW + GW]); };
  auto s_mask = [&](int k) { return __float_as_uint(s_rec[k * RW + GW + 1]); };

  const int t = threadIdx.x;
  const int lane = t % kWave;
  const int wave = t / kWave;
  const int64_t n_tiles = static_cast<int64_t>(a.tw) * a.th;
  // flush role of this thread (raster_bwd_kernel)
  const int fc = t % kFlushLanes;
  int fl_word0 = -1, fl_word1 = -1, fl_kind = kFlushPlain, fl_comp = 0, fl_stride = 1;
  float fl_scale = 1.0f;
  float* fl_base = v_opacities;
  if (fc < CH) {
    fl_word0 = fc, fl_base = v_colors, fl_stride = CH, fl_comp = fc;
  } else if (fc < CH + 3) {
    fl_word0 = fc, fl_base = v_conics, fl_stride = 3, fl_comp = fc - CH, fl_scale = fc - CH == 1 ? 1.0f : 0.5f;
  } else if (fc < CH + 5) {
    fl_word0 = CH + 3, fl_word1 = CH + 4, fl_kind = kFlushMean, fl_base = v_means2d, fl_stride = 2, fl_comp = fc - CH - 3;
  } else if (fc == CH + 5) {
    fl_word0 = CH + 5, fl_kind = kFlushOpacity, fl_base = v_opacities;
  }

  const int64_t unit = blockIdx.x;
  if (unit >= n_units) return;  // uniform across the block
  const int64_t it = order[unit];
  const int64_t image = it / n_tiles;
  const int tile = static_cast<int>(it % n_tiles);
  const int tx = tile % a.tw, ty = tile / a.tw;
  int64_t start, end;
  tile_range(a, image, tile, &start, &end);
  const int64_t stop = start + cost[it];
  int32_t r_id = 0;
  float2 r_xy = make_float2(0.0f, 0.0f);
  float4 r_co = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  int32_t r_g = 0;
  float r_col[CH];
  auto load_ids = [&](int64_t hi, int64_t lo) {
    const int64_t j = hi - 1 - t;
    if (t < BB && j >= lo) r_id = a.flatten_ids[j];
  };
  auto load_records = [&](int64_t hi, int64_t lo) {  // of the ids in r_id
    const int64_t j = hi - 1 - t;
    if (t < BB && j >= lo) {
      const int32_t g = r_id;
      const bool ok = g >= 0 && static_cast<int64_t>(g) < a.G;
      const int64_t gg = ok ? g : 0;
      r_g = ok ? g : 0;
      if (ok) {
        r_xy = make_float2(a.means2d[gg * 2], a.means2d[gg * 2 + 1]);
        r_co = make_float4(a.conics[gg * 3], a.conics[gg * 3 + 1], a.conics[gg * 3 + 2], a.opacities[gg]);
      } else {
        r_xy = make_float2(0.0f, 0.0f);
        r_co = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      }
#pragma unroll
      for (int c = 0; c < CH; ++c) r_col[c] = ok ? a.colors[gg * CH + c] : 0.0f;
    }
  };
  if (stop > start) {
    const int64_t lo0 = max<int64_t>(start, stop - BB);
    load_ids(stop, lo0);
    load_records(stop, lo0);
  }

  store_wave_rects(s_rect, n_waves, a.ts, tx, ty);
  int wave_last;
  bool wave_tame;
  {
    int qx, qy;
    lane_pixel(t, a.ts, &qx, &qy);
    const int x = tx * a.ts + qx;
    const int y = ty * a.ts + qy;
    const bool inside = t < a.ts * a.ts && x < a.W && y < a.H;
    const int64_t pix = (image * a.H + y) * static_cast<int64_t>(a.W) + x;
    const float T_final = inside ? 1.0f - render_alphas[pix] : 1.0f;
    int last_rel = -1;  // last contributor relative to start, -1 for none
    if (inside) {
      const int64_t l = min<int64_t>(end - 1, last_ids[pix]) - start;
      last_rel = static_cast<int>(max<int64_t>(-1, min<int64_t>(l, INT32_MAX - 1)));
    }
    float v_rc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    float bg_dot = 0.0f;
#pragma unroll
    for (int c = 0; c < CH; ++c) v_rc[c] = inside ? v_render_colors[pix * CH + c] : 0.0f;
    const float v_ra = inside && v_render_alphas ? v_render_alphas[pix] : 0.0f;
    if (a.backgrounds) {
      const float* bg = a.backgrounds + image * CH;
#pragma unroll
      for (int c = 0; c < CH; ++c) bg_dot += bg[c] * v_rc[c];
    }
    const float coef = T_final * v_ra + -T_final * bg_dot;
    // all of the wave's pixel values tame: then a record that a pixel does not
    // take adds -0 v_alpha = 0 without a select (levels 0 and 1 below)
    bool rc_tame = fabsf(T_final) <= 3.402823466e38f && fabsf(coef) <= kTameBuffer;
#pragma unroll
    for (int c = 0; c < CH; ++c) rc_tame = rc_tame && fabsf(v_rc[c]) <= kTameColor;
    wave_tame = __ballot(!rc_tame) == 0;
    wave_last = last_rel;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) wave_last = max(wave_last, __shfl_xor(wave_last, off, kWave));
    s_pix[t] = make_float4(v_rc[0], v_rc[1], v_rc[2], CH == 4 ? v_rc[3] : __int_as_float(last_rel));
    s_state[t] = make_float2(T_final, coef);
    if constexpr (CH == 4) s_last[t] = last_rel;
    if (t < kNeutral) s_neutral[t] = make_float2(1.0f, 0.0f);  // read after the batch loop's first barrier
  }
  const PixRect wr = wave_rect(wave, a.ts, tx, ty);
  const int ri = lane & 15, rk = lane >> 4;  // record of the group, pixel row (and row + 4)
  const float4* pix_row = s_pix + wave * kWave + rk * 8;
  float2* state_row = s_state + wave * kWave + rk * 8;
  // lane 0 of the row brings the pixel's state into the scans, the others
  // their neutral elements
  const float2* state_in = ri == 0 ? state_row : s_neutral;
  const int* last_row = s_last + wave * kWave + rk * 8;  // CH == 4 only
  uint16_t* list = s_list + wave * BB;
  const float py0 = wr.y0 + static_cast<float>(rk), py1 = wr.y0 + static_cast<float>(rk + 4);

  int skip = 0;  // slots of the batch that this wave has already evaluated
  int carried = 0, carried_from = 0;  // slots carried over, and the first of them in the last batch
  for (int64_t b1 = stop; b1 > start;) {
    const int64_t b0 = max<int64_t>(start, b1 - BB);
    __syncthreads();  // previous batch fully consumed and flushed
    if (t < BB && b1 - 1 - t >= b0) {
      const uint32_t cls = record_class(r_xy, r_co);
      const uint32_t r_mask = touch_mask(r_xy, r_co, n_waves, s_rect) | cls;
      float* rec = s_rec + t * RW;
      *reinterpret_cast<float4*>(rec) = make_float4(0.5f * r_co.x, r_co.y, 0.5f * r_co.z, r_co.w);
      float tail[RW - 4];
#pragma unroll
      for (int i = 0; i < RW - 4; ++i) tail[i] = 0.0f;
      tail[0] = r_xy.x;
      tail[1] = r_xy.y;
#pragma unroll
      for (int c = 0; c < CH; ++c) tail[2 + c] = r_col[c];
      tail[GW - 4] = __int_as_float(r_g);
      bool rec_finite = fabsf(r_xy.x) <= 3.402823466e38f && fabsf(r_xy.y) <= 3.402823466e38f;
#pragma unroll
      for (int c = 0; c < CH; ++c) rec_finite = rec_finite && fabsf(r_col[c]) <= kTameColor;
      tail[GW - 3] = __uint_as_float(r_mask | (rec_finite ? 0u : kNonFiniteRecord));
#pragma unroll
      for (int i = 0; i < RW - 4; i += 4)
        *reinterpret_cast<float4*>(rec + 4 + i) = make_float4(tail[i], tail[i + 1], tail[i + 2], tail[i + 3]);
    }
    // the sums of slots carried over move to the batch's first slots (at most
    // half a batch, below the first one carried), the others clear
    for (int w = t; w < BB * NS; w += BS) {
      if (w < carried * NS) {
        s_acc[w] = s_acc[carried_from * NS + w];
        s_acc[carried_from * NS + w] = 0.0;
      } else if (w < carried_from * NS || w >= (carried_from + carried) * NS) {
        s_acc[w] = 0.0;
      }
    }
    __syncthreads();
    const int cnt = static_cast<int>(b1 - b0);
    const int k_rel0 = static_cast<int>(b1 - 1 - start);  // entry of slot 0, relative to start
    int n = 0;
    for (int c0 = 0; c0 < cnt; c0 += kWave) {
      const int kl = c0 + lane;
      const uint32_t mk = kl < cnt ? s_mask(kl) : 0u;
      const bool mine = kl >= skip && k_rel0 - kl <= wave_last && ((mk >> wave) & 1u);
      const uint64_t bits = __ballot(mine);
      const int below = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(bits >> 32),
                                                  __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(bits), 0));
      if (mine) list[n + below] = static_cast<uint16_t>(kl);
      n += __popcll(bits);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // list: written and read by this wave
    // Only whole groups are evaluated while entries remain before this batch:
    // the next one starts at the first slot that some wave left over, unless
    // that wave's few records reach back over half a batch.
    int left = cnt;  // this wave's first slot left over
    if (b0 > start && (n & 15)) {
      const int first = __builtin_amdgcn_readfirstlane(static_cast<int>(list[n & ~15]));
      if (2 * first >= BB) {
        left = first;
        n &= ~15;
      }
    }
    if (lane == 0) s_next[wave] = left;
    __syncthreads();
    int advance = cnt;
    for (int w = 0; w < n_waves; ++w) advance = min(advance, s_next[w]);
    skip = left - advance;
    carried = cnt - advance;
    carried_from = advance;
    const int64_t b1n = b1 - advance;
    const int64_t b0n = max<int64_t>(start, b1n - BB);
    // the next batch's ids, then (behind the first group) its records
    load_ids(b1n, b0n);
    if (n == 0) load_records(b1n, b0n);
    for (int g0 = 0; g0 < n; g0 += 16) {
      const bool live = g0 + ri < n;
      const int slot = list[min(g0 + ri, n - 1)];
      const float* rec = s_rec + slot * RW;
      const float4 co = reinterpret_cast<const float4*>(rec)[0];
      const float4 xc = reinterpret_cast<const float4*>(rec)[1];
      float4 ex = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if constexpr (RW > 8) ex = reinterpret_cast<const float4*>(rec)[2];
      const float col[4] = {xc.z, xc.w, ex.x, ex.y};
      const uint32_t bits = s_mask(slot);
      const int k_rel = live ? k_rel0 - slot : INT_MAX;
      const float dy[2] = {xc.y - py0, xc.y - py1};
      const float cy[2] = {co.z * dy[0] * dy[0], co.z * dy[1] * dy[1]};
      float vc[CH], S[2] = {0.0f, 0.0f}, Hx[2] = {0.0f, 0.0f}, Hxx = 0.0f;
#pragma unroll
      for (int c = 0; c < CH; ++c) vc[c] = 0.0f;
      auto walk = [&](auto level_c) {
        constexpr int kLevel = decltype(level_c)::value;
        constexpr bool kCareful = kLevel == 2;
        float px = wr.x0;
        const float4* pix = pix_row;
        const float2* in = state_in;
        float2* out = state_row;
#pragma unroll 1
        for (int x = 0; x < 8; x += 2, pix += 2, in += 2, out += 2) {
          float4 vr[4];
          float Tn[4], Bb[4], al[4], araw[4], ra[4], fac[4], D[4], Ba[4];
          bool valid[4];
          float dx[2];
#pragma unroll
          for (int q = 0; q < 4; ++q) {  // q = 2 * column + half
            const int at = (q >> 1) + 32 * (q & 1);
            vr[q] = pix[at];
            const float2 st = in[at];
            Tn[q] = st.x;
            Bb[q] = st.y;
            const int last = CH == 4 ? last_row[x + at] : __float_as_int(vr[q].w);
            valid[q] = k_rel <= last;
          }
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            dx[p] = xc.x - px;
            px += 1.0f;
            const float ax = co.x * dx[p] * dx[p];
            const float bx = co.y * dx[p];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int q = 2 * p + h;
              const float sigma = (ax + cy[h]) + bx * dy[h];  // halved_sigma's operations
              float alpha;
              if constexpr (kLevel < 2) {
                araw[q] = co.w * exp_alpha_bounded(-sigma);
                alpha = kLevel == 0 ? araw[q] : fminf(kMaxAlpha, araw[q]);
                valid[q] = valid[q] && alpha >= kAlphaThreshold;
              } else {
                araw[q] = co.w * exp_alpha(-sigma);
                alpha = fminf(kMaxAlpha, araw[q]);
                valid[q] = valid[q] && !(sigma < 0.0f || alpha < kAlphaThreshold);
              }
              al[q] = valid[q] ? alpha : 0.0f;
              ra[q] = __builtin_amdgcn_rcpf(1.0f - al[q]);  // alpha <= 0.99; 1 for alpha = 0
              Tn[q] *= ra[q];
            }
          }
          row16_product4(Tn);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            fac[q] = al[q] * Tn[q];
            const float vrq[4] = {vr[q].x, vr[q].y, vr[q].z, vr[q].w};
            D[q] = col[0] * vrq[0];
#pragma unroll
            for (int c = 1; c < CH; ++c) D[q] = __builtin_fmaf(col[c], vrq[c], D[q]);
            if constexpr (kCareful) {
              Ba[q] = valid[q] ? __builtin_fmaf(-fac[q], D[q], Bb[q]) : Bb[q];
#pragma unroll
              for (int c = 0; c < CH; ++c) vc[c] += valid[q] ? fac[q] * vrq[c] : 0.0f;
            } else {
              Ba[q] = __builtin_fmaf(-fac[q], D[q], Bb[q]);
#pragma unroll
              for (int c = 0; c < CH; ++c) vc[c] = __builtin_fmaf(fac[q], vrq[c], vc[c]);
            }
          }
          row16_sum4(Ba, Bb);
          if (ri == 15) {
#pragma unroll
            for (int q = 0; q < 4; ++q) out[(q >> 1) + 32 * (q & 1)] = make_float2(Tn[q], Ba[q]);
          }
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            float vs[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int q = 2 * p + h;
              const float v_alpha = __builtin_fmaf(Tn[q], D[q], ra[q] * Bb[q]);
              vs[h] = -al[q] * v_alpha;
              if constexpr (kLevel == 1) vs[h] = araw[q] <= kMaxAlpha ? vs[h] : 0.0f;
              if constexpr (kLevel == 2) vs[h] = valid[q] && araw[q] <= kMaxAlpha ? vs[h] : 0.0f;
              S[h] += vs[h];
              Hx[h] = __builtin_fmaf(vs[h], dx[p], Hx[h]);
            }
            if constexpr (kCareful) {  // the means may lie so far that dx dx overflows, with vs 0
              Hxx = __builtin_fmaf((vs[0] + vs[1]) * dx[p], dx[p], Hxx);
            } else {
              Hxx = __builtin_fmaf(vs[0] + vs[1], dx[p] * dx[p], Hxx);
            }
          }
        }
      };
      int level = 0;
      if (__ballot(live && (bits & kCappedRecord)) != 0) level = 1;
      if (!wave_tame || __ballot(live && (bits & (kGeneralRecord | kNonFiniteRecord))) != 0) level = 2;
      if (level == 0) {
        walk(std::integral_constant<int, 0>{});
      } else if (level == 1) {
        walk(std::integral_constant<int, 1>{});
      } else {
        walk(std::integral_constant<int, 2>{});
      }
      float v[NV];
#pragma unroll
      for (int c = 0; c < CH; ++c) v[c] = vc[c];
      v[CH + 0] = Hxx;
      v[CH + 1] = __builtin_fmaf(Hx[1], dy[1], Hx[0] * dy[0]);
      const float sy0 = S[0] * dy[0], sy1 = S[1] * dy[1];
      v[CH + 2] = __builtin_fmaf(sy1, dy[1], sy0 * dy[0]);
      v[CH + 3] = Hx[0] + Hx[1];
      v[CH + 4] = sy0 + sy1;
      v[CH + 5] = S[0] + S[1];
      if (level == 2 && (bits & kNonFiniteRecord) && !(fabsf(xc.x) <= 3.402823466e38f && fabsf(xc.y) <= 3.402823466e38f)) {
        // no pixel has a geometry term under a non-finite mean
#pragma unroll
        for (int i = CH; i < NV; ++i) v[i] = 0.0f;
      }
      // sums over the four rows: after the two exchanges a lane with bits
      // h = lane[5], r = lane[4] holds component 4 m + 2 r + h in y[m]
      constexpr int NA = (NV + 1) / 2, NB = (NA + 1) / 2;
      float w[NA], y[NB];
      unsigned spare = 0u;
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        const unsigned b = (2 * i + 1 < NV) ? ubits(v[2 * i + 1]) : spare;
        const auto sw = __builtin_amdgcn_permlane32_swap(ubits(v[2 * i]), b, false, false);
        w[i] = fbits(sw[0]) + fbits(sw[1]);
        spare = sw[1];
      }
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const unsigned b = (2 * i + 1 < NA) ? ubits(w[2 * i + 1]) : spare;
        const auto sw = __builtin_amdgcn_permlane16_swap(ubits(w[2 * i]), b, false, false);
        y[i] = fbits(sw[0]) + fbits(sw[1]);
        spare = sw[1];
      }
      if (live) {
        const int comp0 = 2 * (rk & 1) + (rk >> 1);
        double* acc = s_acc + slot * NS + comp0;
#pragma unroll
        for (int m = 0; m < NB; ++m) {
          const int c = 4 * m + comp0;
          if (4 * m + 3 < NV || c < NV)
            __hip_atomic_fetch_add(acc + 4 * m, static_cast<double>(y[m]), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
        }
      }
      if (g0 == 0) load_records(b1n, b0n);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the pixels' state: lane 15 wrote it, lane 0 reads it next
    }
    __syncthreads();
    __builtin_amdgcn_s_waitcnt(kWaitVmemOnly);
    for (int idx = t; idx < advance * kFlushLanes; idx += BS) {
      const int slot = idx / kFlushLanes;
      if (fl_word0 < 0) continue;  // lanes past the slot's components
      float v = static_cast<float>(s_acc[slot * NS + fl_word0]);
      const int64_t gg = s_g(slot);
      if (fl_kind == kFlushMean) {
        const float v2 = static_cast<float>(s_acc[slot * NS + fl_word1]);
        if (v == 0.0f && v2 == 0.0f) continue;
        const float4 co = *reinterpret_cast<const float4*>(s_rec + slot * RW);
        v = fl_comp == 0 ? (co.x + co.x) * v + co.y * v2 : co.y * v + (co.z + co.z) * v2;
      } else if (fl_kind == kFlushOpacity) {
        if (v == 0.0f) continue;
        v = -v / s_rec[slot * RW + 3];
      } else {
        v *= fl_scale;
      }
      if (v != 0.0f) unsafeAtomicAdd(fl_base + gg * fl_stride + fl_comp, v);
    }
    b1 = b1n;
  }
}

// Heavy-first tile schedule for the backward. A tile's cost is the number of
// list entries its pixels replay (largest last_id - start + 1, 0 when masked
// or empty). The backward launches one block per tile in descending cost
// order, so the longest tiles start first and the end of the launch is made
// of short ones (greedy longest-processing-time scheduling).
//
// The same pass over the tile's pixels also forms the tile's share of the
// background gradient, v_backgrounds[i, c] = sum over the unmasked pixels of
// image i of (1 - render_alpha) * v_render_colors[c] (gsplat_rasterize.cpp:
// 459-464; the background enters each pixel as T_final * bg): one partial
// per (tile, channel), summed per image by the order kernel's extra blocks.
// No atomics: every partial has one writer.
constexpr int kCostBuckets = 4096;  // costs >= 4095 share the heaviest bucket

template <int CH>
__global__ void __launch_bounds__(256) tile_cost_kernel(RasterArgs a, const int32_t* __restrict__ last_ids,
                                                        const float* __restrict__ render_alphas,
                                                        const float* __restrict__ v_render_colors,
                                                        int32_t* __restrict__ cost, float* __restrict__ bg_part,
                                                        ZeroSpans zero) {
  constexpr int LC = CH > 0 ? CH : 1;
  __shared__ int s_best[256 / kWave];
  __shared__ float s_sum[256 / kWave][LC];
  const int tx = blockIdx.x, ty = blockIdx.y;
  const int64_t image = blockIdx.z;
  const int tile = ty * a.tw + tx;
  const int64_t n_tiles = static_cast<int64_t>(a.tw) * a.th;
  const int64_t unit = image * n_tiles + tile;
  const int t = threadIdx.x;
  const int channels = CH > 0 ? CH : a.channels;
  // the backward's accumulated outputs start at zero: cleared here, one
  // launch ahead of the kernel that accumulates into them
  zero_spans_share(zero, unit * 256 + t, static_cast<int64_t>(a.I) * n_tiles * 256);
  int64_t start, end;
  tile_range(a, image, tile, &start, &end);
  const bool live = !(a.masks && !a.masks[unit]);
  int best = 0;
  float acc[LC];
#pragma unroll
  for (int c = 0; c < LC; ++c) acc[c] = 0.0f;
  if (live) {
    for (int q = t; q < a.ts * a.ts; q += 256) {
      const int x = tx * a.ts + q % a.ts;
      const int y = ty * a.ts + q / a.ts;
      if (x >= a.W || y >= a.H) continue;
      const int64_t pix = (image * a.H + y) * static_cast<int64_t>(a.W) + x;
      const int64_t last = min<int64_t>(end - 1, last_ids[pix]);
      best = max(best, static_cast<int>(min<int64_t>(max<int64_t>(last - start + 1, 0), INT32_MAX)));
      if constexpr (CH > 0) {
        if (bg_part) {
          const float T_final = 1.0f - render_alphas[pix];
#pragma unroll
          for (int c = 0; c < CH; ++c) acc[c] += T_final * v_render_colors[pix * CH + c];
        }
      }
    }
  }
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) best = max(best, __shfl_xor(best, off, kWave));
  if (t % kWave == 0) s_best[t / kWave] = best;
  if (bg_part && CH > 0) {
#pragma unroll
    for (int c = 0; c < LC; ++c) {
      const float w = wave_sum_uniform(acc[c]);
      if (t % kWave == 0) s_sum[t / kWave][c] = w;
    }
  }
  __syncthreads();
  if (t == 0) {
    for (int w = 1; w < 256 / kWave; ++w) best = max(best, s_best[w]);
    cost[unit] = best;
  }
  if (!bg_part) return;
  if constexpr (CH > 0) {
    if (t < CH) {
      float sum = 0.0f;
      for (int w = 0; w < 256 / kWave; ++w) sum += s_sum[w][t];
      bg_part[unit * CH + t] = sum;
    }
  } else {
    // any channel count: one channel at a time
    for (int c = 0; c < channels; ++c) {
      float v = 0.0f;
      if (live) {
        for (int q = t; q < a.ts * a.ts; q += 256) {
          const int x = tx * a.ts + q % a.ts;
          const int y = ty * a.ts + q / a.ts;
          if (x >= a.W || y >= a.H) continue;
          const int64_t pix = (image * a.H + y) * static_cast<int64_t>(a.W) + x;
          v += (1.0f - render_alphas[pix]) * v_render_colors[pix * channels + c];
        }
      }
      const float w = wave_sum_uniform(v);
      __syncthreads();  // the previous channel's partials have been read
      if (t % kWave == 0) s_sum[t / kWave][0] = w;
      __syncthreads();
      if (t == 0) {
        float sum = 0.0f;
        for (int k = 0; k < 256 / kWave; ++k) sum += s_sum[k][0];
        bg_part[unit * channels + c] = sum;
      }
    }
  }
}

// The same for 16-pixel tiles with a block per strip of kStripTiles tiles of
// one tile row: lane c of each wave takes pixel column c of the strip (so a
// wave reads 64 consecutive pixels of a row, 256-768 bytes, instead of four
// 16-pixel pieces), waves take rows w, w + 4, ...; each tile's values are
// reduced over its 16 lanes by DPP row shifts (one 16-lane row is one tile),
// then over the waves in LDS in a fixed order.
constexpr int kStripTiles = 4;

__device__ __forceinline__ float row16_sum(float v) {  // lane 15 of each 16-lane row: the row's sum
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x111, 0xf, 0xf, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x112, 0xf, 0xf, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x114, 0xf, 0xf, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x118, 0xf, 0xf, false));
  return v;
}

__device__ __forceinline__ int row16_max(int v) {  // lane 15 of each 16-lane row: the row's maximum (v >= 0)
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));
  return v;
}

template <int CH>
__global__ void __launch_bounds__(256) tile_cost_strip_kernel(RasterArgs a, const int32_t* __restrict__ last_ids,
                                                              const float* __restrict__ render_alphas,
                                                              const float* __restrict__ v_render_colors,
                                                              int32_t* __restrict__ cost, float* __restrict__ bg_part,
                                                              ZeroSpans zero) {
  static_assert(CH >= 1 && CH <= 4, "staged channel counts");
  constexpr int TS = 16, NW = 4;
  __shared__ int s_best[NW][kStripTiles];
  __shared__ float s_sum[NW][kStripTiles][CH];
  const int t = threadIdx.x, col = t % kWave, wave = t / kWave;
  const int64_t image = blockIdx.z;
  const int ty = blockIdx.y;
  const int k = col / TS;                        // tile of the strip
  const int tx = blockIdx.x * kStripTiles + k;   // its column in the tile grid
  const int64_t n_tiles = static_cast<int64_t>(a.tw) * a.th;
  const int64_t block = (image * gridDim.y + ty) * gridDim.x + blockIdx.x;
  zero_spans_share(zero, block * 256 + t, static_cast<int64_t>(gridDim.x) * gridDim.y * gridDim.z * 256);
  const bool tile_ok = tx < a.tw;
  const int64_t unit = image * n_tiles + static_cast<int64_t>(ty) * a.tw + tx;
  int64_t start = 0, end = 0;
  if (tile_ok) tile_range(a, image, ty * a.tw + tx, &start, &end);
  const bool live = tile_ok && !(a.masks && !a.masks[unit]);
  const int x = tx * TS + col % TS;
  int best = 0;
  float acc[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) acc[c] = 0.0f;
  if (live && x < a.W) {
#pragma unroll
    for (int r = 0; r < TS / NW; ++r) {
      const int y = ty * TS + wave + NW * r;
      if (y >= a.H) break;
      const int64_t pix = (image * a.H + y) * static_cast<int64_t>(a.W) + x;
      const int64_t last = min<int64_t>(end - 1, last_ids[pix]);
      best = max(best, static_cast<int>(min<int64_t>(max<int64_t>(last - start + 1, 0), INT32_MAX)));
      if (bg_part) {
        const float T_final = 1.0f - render_alphas[pix];
#pragma unroll
        for (int c = 0; c < CH; ++c) acc[c] += T_final * v_render_colors[pix * CH + c];
      }
    }
  }
  best = row16_max(best);
#pragma unroll
  for (int c = 0; c < CH; ++c) acc[c] = row16_sum(acc[c]);
  if (col % TS == TS - 1) {
    s_best[wave][k] = best;
#pragma unroll
    for (int c = 0; c < CH; ++c) s_sum[wave][k][c] = acc[c];
  }
  __syncthreads();
  if (t < kStripTiles) {
    const int txo = blockIdx.x * kStripTiles + t;
    if (txo < a.tw) {
      const int64_t u = image * n_tiles + static_cast<int64_t>(ty) * a.tw + txo;
      int b = 0;
      float sum[CH];
#pragma unroll
      for (int c = 0; c < CH; ++c) sum[c] = 0.0f;
      for (int w = 0; w < NW; ++w) {
        b = max(b, s_best[w][t]);
#pragma unroll
        for (int c = 0; c < CH; ++c) sum[c] += s_sum[w][t][c];
      }
      cost[u] = b;
      if (bg_part) {
#pragma unroll
        for (int c = 0; c < CH; ++c) bg_part[u * CH + c] = sum[c];
      }
    }
  }
}

// Block 0: counting sort of the n tile costs into descending order. Blocks
// 1 .. I * channels (when bg_part is set): v_backgrounds[i][c] as the sum of
// image i's per-tile partials of channel c, in tile order (deterministic).
// Up to kOrderItems costs per thread are loaded at once and kept in registers
// for the second pass (n <= 8192 tiles); larger n loop over global memory.
constexpr int kOrderBlock = 1024;
constexpr int kOrderItems = 8;

__global__ void __launch_bounds__(kOrderBlock) tile_order_kernel(const int32_t* __restrict__ cost, int64_t n,
                                                                 int32_t* __restrict__ order,
                                                                 const float* __restrict__ bg_part, int64_t n_tiles,
                                                                 int channels, float* __restrict__ v_backgrounds) {
  static_assert(kCostBuckets % kOrderBlock == 0, "buckets per thread");
  constexpr int PER = kCostBuckets / kOrderBlock;
  constexpr int W = kOrderBlock / kWave;
  __shared__ int hist[kCostBuckets];
  __shared__ int s_w[W];
  const int t = threadIdx.x, lane = t % kWave, wave = t / kWave;
  if (blockIdx.x > 0) {
    const int64_t ic = blockIdx.x - 1;  // image * channels + c
    const int64_t image = ic / channels;
    const int c = static_cast<int>(ic % channels);
    const float* part = bg_part + image * n_tiles * channels + c;
    float v = 0.0f;
    for (int64_t j = t; j < n_tiles; j += kOrderBlock) v += part[j * channels];
    float* s_sum = reinterpret_cast<float*>(hist);
    const float w = wave_sum_uniform(v);
    if (lane == 0) s_sum[wave] = w;
    __syncthreads();
    if (t == 0) {
      float sum = 0.0f;
      for (int k = 0; k < W; ++k) sum += s_sum[k];
      v_backgrounds[ic] = sum;
    }
    return;
  }
  auto bucket = [](int32_t c) { return kCostBuckets - 1 - min(c, kCostBuckets - 1); };
  const bool in_regs = n <= static_cast<int64_t>(kOrderBlock) * kOrderItems;  // uniform
  int32_t b[kOrderItems];
  if (in_regs) {
#pragma unroll
    for (int k = 0; k < kOrderItems; ++k) {
      const int64_t i = t + static_cast<int64_t>(k) * kOrderBlock;
      b[k] = i < n ? bucket(cost[i]) : -1;
    }
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) hist[t * PER + j] = 0;
  __syncthreads();
  if (in_regs) {
#pragma unroll
    for (int k = 0; k < kOrderItems; ++k)
      if (b[k] >= 0) atomicAdd(&hist[b[k]], 1);
  } else {
    for (int64_t i = t; i < n; i += kOrderBlock) atomicAdd(&hist[bucket(cost[i])], 1);
  }
  __syncthreads();
  int h[PER], sum = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    h[j] = hist[t * PER + j];
    sum += h[j];
  }
  const int inc = wave_inclusive_scan(sum);
  if (lane == kWave - 1) s_w[wave] = inc;
  __syncthreads();
  int running = inc - sum;
#pragma unroll
  for (int w = 0; w < W; ++w) running += w < wave ? s_w[w] : 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    hist[t * PER + j] = running;
    running += h[j];
  }
  __syncthreads();
  if (in_regs) {
#pragma unroll
    for (int k = 0; k < kOrderItems; ++k)
      if (b[k] >= 0) order[atomicAdd(&hist[b[k]], 1)] = t + k * kOrderBlock;
  } else {
    for (int64_t i = t; i < n; i += kOrderBlock) order[atomicAdd(&hist[bucket(cost[i])], 1)] = static_cast<int32_t>(i);
  }
}

size_t align256(size_t b) { return (b + 255) / 256 * 256; }
// cost [n] int32, order [n] int32, background partials [n][channels] float
size_t bwd_workspace_bytes(int64_t n_tiles_total, int channels) {
  return 2 * align256(static_cast<size_t>(n_tiles_total) * 4) +
         align256(static_cast<size_t>(n_tiles_total) * channels * 4);
}

// records: mean 2, conic+opacity 4, colours (CH > 0), Gaussian id, touch mask
// plus one float4 wave rectangle per wave
size_t fwd_smem(int ch, int bs) {
  return static_cast<size_t>(bs) * (fwd_record_words(ch) + 1) * 4 + static_cast<size_t>(bs / kWave) * 16;
}
// Backward block: one pixel per lane, the whole tile in one block (measured
// fastest on gfx950 for 16x16 tiles against 2 or 4 pixels per lane and
// against splitting a tile over several blocks: the lower register count
// keeps six waves per SIMD resident). Batch length: 128 entries for blocks of
// up to 256 lanes, 64 above (bounds the per-wave accumulators to 52 KiB at
// 1024 lanes, 4 channels, absgrad); never more than the block, so one lane
// loads one record.
int bwd_block(int ts) { return (ts * ts + kWave - 1) / kWave * kWave; }
int bwd_batch(int bs) { return bs <= 128 ? bs : (bs <= 256 ? 128 : 64); }
// one record (bwd_record_words) per batch slot plus NV + 1 accumulator words
// per (wave, slot)
size_t bwd_smem(int ch, int bs, int bb, bool absgrad) {
  const int cc = ch > 0 ? ch : 0;
  const int ns = cc + (absgrad ? 8 : 6) + 1;
  return static_cast<size_t>(bb) * (bwd_record_words(ch) + (bs / kWave) * ns) * 4 + static_cast<size_t>(bs / kWave) * 16;
}

// The kernels with records in lanes take tiles of whole 8x8 pixel blocks whose
// LDS stays below 64 KiB, in images whose pixel centres are exact floats under
// + 1 steps.
bool rows_kernels_apply(int ts, int width, int height) {
  return (ts == 8 || ts == 16 || ts == 24) && width <= (1 << 22) && height <= (1 << 22);
}

// Where the forward with records in lanes is the faster one (the results are
// the same bits). A group costs the same for one record as for 16, so short
// lists are better off in the kernel with pixels in lanes, whose smaller LDS also
// keeps more blocks resident: the lines lie higher once the tiles come in more
// than one round of resident blocks. Times of the kernel with pixels in lanes over
// this one's, three channels, scenes of 1000 to 1,000,000 Gaussians:
// - side 16, 475 tiles: 0.95 at 4 entries per tile, 1.00-1.01 at 8 to 14, 1.2
//   at 20 to 40. 784 tiles (two blocks each, more than are resident): 0.85 at
//   19, 0.94-0.97 at 30 to 38, 1.13 at 62.
// - 960 to 1200 tiles: 0.96-1.00 at 16 to 18, 1.0-1.06 at 22 to 30. 1900 to 18,900
//   tiles: 0.8-0.9 up to 35, 0.91-1.09 at 40 to 55, 0.97-1.07 at 65 to 95, 1.0-1.2
//   beyond (evenly spread lists of about 145 entries, a batch and a bit: 0.93-0.97).
// - four channels (colours and entries in separate words): 0.97-1.06 at 1024
//   tiles and 17 to 169 entries, 1.10-1.14 beyond; 0.95-1.05 on larger grids.
// - side 8 (a wave per block): 1.04-1.4 up to 1900 tiles, 1.1-1.25 at 4096 from
//   34 on (0.94 at 4), 0.64-1.0 on most larger grids (1.05-1.14 on two). Side 24
//   (9 waves, 3 blocks per CU by LDS): 0.7-1.0 nearly everywhere.
bool fwd_rows_faster(int ts, int ch, int64_t n_tiles, int64_t per_tile) {
  if (ts == 24) return false;
  if (ts == 8) return n_tiles <= 4096 && per_tile >= (n_tiles <= 2048 ? 8 : 32);
  if (n_tiles <= 800) return per_tile >= (n_tiles <= 512 ? 12 : 48);
  if (n_tiles <= 1536) return per_tile >= (ch < 4 ? 24 : 128);  // 6 blocks on each of 256 CUs
  return ch < 4 && per_tile >= 64;
}

// The same for the backward (also by the block's registers: 4 blocks per CU of
// side 16, one of side 24, against 6 and 2):
// - side 16, 475 tiles: 0.87-0.95 at 4 to 8 entries per tile, 0.95-1.27 at 12 to
//   21. 960 and 1024 tiles: 0.87-0.95 up to 18, 0.99-1.06 at 25, 1.06-1.08 at 35.
//   1125 to 18,900 tiles: 0.55-0.9 up to 30, 0.92-1.2 at 55 to 70, 0.95-1.12 at 72
//   to 82, 1.1-1.35 beyond.
// - side 8: 1.0-1.25 up to 3072 tiles, 1.06-1.18 at 4096 from 34 on (0.85 at 4),
//   on larger grids 0.9-1.0 up to 96 and 1.0-1.1 beyond; four channels, which
//   spill, 0.7-1.06 from 4096 tiles on.
// - side 24: 1.04-1.5 up to 663 tiles from 33 on (0.6-0.75 at 12 to 22); from 850
//   tiles on 0.5-1.0 up to 180 and 1.0-1.3 beyond, with four channels 1.02-1.7
//   from 40 on.
bool bwd_rows_faster(int ts, int ch, int64_t n_tiles, int64_t per_tile) {
  if (ts == 24) return per_tile >= (n_tiles <= 768 || ch == 4 ? 32 : 256);
  if (ts == 8) {
    if (n_tiles <= 2048) return per_tile >= (ch < 4 ? 8 : 32);
    return ch < 4 && per_tile >= (n_tiles <= 4096 ? 32 : 128);
  }
  if (n_tiles <= 1024) return per_tile >= (n_tiles <= 512 ? 16 : 32);
  return per_tile >= 80;
}

// raster_fwd_rows_kernel: records, alphas, colours, wave rectangles, entries and
// record lists.
size_t fwd_rows_smem(int ch, int n_waves, int pixels, int bb) {
  const size_t words = static_cast<size_t>(bb) * fwd_rows_record_words(ch) +
                       static_cast<size_t>(n_waves) * (16 * (pixels + 4) + 64 + 4 + (ch == 4 ? 16 : 0));
  return words * 4 + static_cast<size_t>(n_waves) * bb;
}

// raster_bwd_rows_kernel: accumulators, pixel cotangents and state, records, wave
// rectangles and record lists, in the kernel's order.
// Batches: 256 entries leave the fewest barriers and flushes (1M Gaussians, 4346
// tiles of 1245 entries: 232 us against 242 at 128). Of side 16, 128 keep as many
// blocks resident (by registers, 4 on each of 256 CUs) and suit shorter lists, the
// more the fewer rounds of resident blocks there are. Time of 256 over that of
// 128: 1.0-1.18 at 1900 to 5700 tiles and 70 to 260 entries per tile (one scene
// 0.9), 0.93-1.1 at 320; at 7500 to 41,000 tiles 0.98-1.1 at 70 to 110, 0.93-1.05 at
// 140 to 180, 0.92-1.0 beyond. With four channels LDS admits 3 blocks of 256
// entries or 4 of 128: 1.0-1.2.
// Up to 1024 tiles 128, though 256 are 1.0 to 1.3 times as fast there (side 24
// up to 1.4): tiles add to a Gaussian by float atomics, in no fixed order, and
// with 256 entries this showed more. 10,000 Gaussians at 256x256: three quaternion
// gradients of one Gaussian, all cancellation, differed by 3e-4 between a third
// of 120 runs; with 128 none by 1e-4.
int bwd_rows_batch(int ts, int bs, int ch, int64_t n_tiles, int64_t per_tile) {
  const bool small = n_tiles <= 1024 || (ts == 16 && (ch == 4 || per_tile < (n_tiles <= 6144 ? 256 : 160)));
  return std::min(bs, small ? kRowsSmallBatch : kRowsBatch);
}
size_t bwd_rows_smem(int ch, int bs, int bb) {
  const size_t ns = static_cast<size_t>(ch + 6) | 1;
  const size_t acc = (static_cast<size_t>(bb) * ns + 1) / 2 * 16;
  const size_t words = static_cast<size_t>(bs) * (ch == 4 ? 7 : 6) + 2 * kNeutral +
                       static_cast<size_t>(bb) * bwd_record_words(ch) + 5 * (bs / kWave);
  return acc + words * 4 + static_cast<size_t>(bs / kWave) * bb * 2;
}

int check_args(const RasterArgs& a, const char* what) {
  if (a.I < 0 || a.N < 0 || a.channels <= 0 || a.W < 0 || a.H < 0 || a.ts <= 0 || a.tw < 0 || a.th < 0 ||
      a.n_isects < 0)
    return invalid(std::string(what) + ": invalid sizes.");
  if (a.channels > kMaxChannels)
    return invalid(std::string(what) + ": at most 64 channels are supported.");
  if (a.ts * a.ts > 1024) return invalid(std::string(what) + ": tile_size must be at most 32.");
  if (static_cast<int64_t>(a.tw) * a.ts < a.W || static_cast<int64_t>(a.th) * a.ts < a.H)
    return invalid(std::string(what) + ": tile grid does not cover the image.");
  if (a.I > 65535 || a.th > 65535) return invalid(std::string(what) + ": too many images or tile rows.");
  return GSPLAT_OK;
}

// ---------------------------------------------------------------------------
// Rasterize to indices (upstream gsplat's rasterize_to_indices_in_range,
// note/gsplat_cuda_source_map.md:494-545; the reference's planned
// rasterize_to_indices_3dgs_forward). Per pixel, starting from transmittance
// T0 (1 without a transmittance image), the entries of its tile's list at
// positions [range_start, range_end) that pass the forward's alpha test, in
// list order, until the next transmittance would fall to 1e-4 -- the
// forward's compositing rule with its alpha, threshold and exp, so the
// entries are exactly those the forward composites. One block per tile, one
// lane per pixel, records staged through LDS; pass 1 (WRITE false) counts
// per pixel, pass 2 writes each pixel's entries at its scanned start:
// gaussian id and the pixel's global index image * H * W + y * W + x.
template <bool WRITE>
__global__ void __launch_bounds__(1024) raster_indices_kernel(RasterArgs a, int64_t range_start, int64_t range_end,
                                                              const float* __restrict__ transmittances,
                                                              int32_t* __restrict__ counts,
                                                              const int32_t* __restrict__ starts, int64_t n_out,
                                                              int32_t* __restrict__ out_gauss,
                                                              int64_t* __restrict__ out_index) {
  __shared__ float4 s_co[1024];
  __shared__ float2 s_xy[1024];
  __shared__ int32_t s_g[1024];
  const int tx = blockIdx.x, ty = blockIdx.y;
  const int64_t image = blockIdx.z;
  const int t = threadIdx.x;
  const int bs = blockDim.x;
  const int x = tx * a.ts + t % a.ts, y = ty * a.ts + t / a.ts;
  const bool inside = t < a.ts * a.ts && x < a.W && y < a.H;
  const int64_t pix = image * a.H * a.W + static_cast<int64_t>(y) * a.W + x;
  int64_t s0, e0;
  tile_range(a, image, ty * a.tw + tx, &s0, &e0);
  const int64_t start = min(s0 + max<int64_t>(range_start, 0), e0);
  const int64_t end = min(s0 + max<int64_t>(range_end, 0), e0);
  const float px = static_cast<float>(x) + 0.5f, py = static_cast<float>(y) + 0.5f;
  float T = inside && transmittances ? transmittances[pix] : 1.0f;
  bool done = !inside;
  int32_t cnt = 0;
  int64_t pos = WRITE && inside ? starts[pix] : 0;
  for (int64_t b = start; b < end; b += bs) {
    if (__syncthreads_count(!done) == 0) break;
    const int64_t j = b + t;
    if (j < end) {
      float2 xy;
      float4 co;
      s_g[t] = load_gaussian(a, j, &xy, &co);
      s_xy[t] = xy;
      s_co[t] = co;
    }
    __syncthreads();
    const int n = static_cast<int>(min<int64_t>(bs, end - b));
    for (int k = 0; k < n && !done; ++k) {
      const float4 co = s_co[k];
      const float dx = s_xy[k].x - px;
      const float dy = s_xy[k].y - py;
      const float sigma = 0.5f * (co.x * dx * dx + co.z * dy * dy) + co.y * dx * dy;
      const float alpha = fminf(kMaxAlpha, co.w * exp_alpha(-sigma));
      if (sigma < 0.0f || alpha < kAlphaThreshold) continue;
      const float next_T = T * (1.0f - alpha);
      if (next_T <= kTransmittanceThreshold) {
        done = true;
        break;
      }
      if constexpr (WRITE) {
        if (pos < n_out) {
          out_gauss[pos] = s_g[k];
          out_index[pos] = pix;
        }
        ++pos;
      }
      ++cnt;
      T = next_T;
    }
  }
  if (!WRITE && inside) counts[pix] = cnt;
}

// E_f of the forward, per tile: the (pixel, list entry) evaluations of the
// reference's per-pixel loop (gsplat_rasterize.cpp:291-368) -- every entry of
// the pixel's tile list up to and including the one whose alpha would take
// the transmittance to 1e-4 -- summed over the tile's pixels into
// tile_evals[image, tile] (0 for a masked tile). The falloff, exp and
// thresholds are the forward's. This measures the work the rasterizer's
// roofline is priced on; the forward itself skips records that cannot touch a
// wave's pixels and stops at the block's last saturated pixel.
__global__ void __launch_bounds__(1024) raster_count_kernel(RasterArgs a, int64_t* __restrict__ tile_evals) {
  __shared__ float4 s_co[1024];
  __shared__ float2 s_xy[1024];
  __shared__ int64_t s_sum[1024 / kWave];
  const int tx = blockIdx.x, ty = blockIdx.y;
  const int64_t image = blockIdx.z;
  const int t = threadIdx.x;
  const int bs = blockDim.x;
  const int tile = ty * a.tw + tx;
  const int64_t n_tiles = static_cast<int64_t>(a.tw) * a.th;
  const int x = tx * a.ts + t % a.ts, y = ty * a.ts + t / a.ts;
  const bool inside = t < a.ts * a.ts && x < a.W && y < a.H;
  const bool masked = a.masks && !a.masks[image * n_tiles + tile];
  int64_t start, end;
  tile_range(a, image, tile, &start, &end);
  const float px = static_cast<float>(x) + 0.5f, py = static_cast<float>(y) + 0.5f;
  float T = 1.0f;
  bool done = !inside || masked;
  int64_t cnt = 0;
  for (int64_t b = start; b < end; b += bs) {
    if (__syncthreads_count(!done) == 0) break;
    const int64_t j = b + t;
    if (j < end) {
      float2 xy;
      float4 co;
      load_gaussian(a, j, &xy, &co);
      s_xy[t] = xy;
      s_co[t] = co;
    }
    __syncthreads();
    const int n = static_cast<int>(min<int64_t>(bs, end - b));
    for (int k = 0; k < n && !done; ++k) {
      ++cnt;
      const float4 co = s_co[k];
      const float dx = s_xy[k].x - px;
      const float dy = s_xy[k].y - py;
      const float sigma = 0.5f * (co.x * dx * dx + co.z * dy * dy) + co.y * dx * dy;
      const float alpha = fminf(kMaxAlpha, co.w * exp_alpha(-sigma));
      if (sigma < 0.0f || alpha < kAlphaThreshold) continue;
      const float next_T = T * (1.0f - alpha);
      if (next_T <= kTransmittanceThreshold) done = true;
      T = next_T;
    }
  }
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) cnt += __shfl_xor(cnt, off, kWave);
  if (t % kWave == 0) s_sum[t / kWave] = cnt;
  __syncthreads();
  if (t == 0) {
    int64_t sum = 0;
    for (int w = 0; w < bs / kWave; ++w) sum += s_sum[w];
    tile_evals[image * n_tiles + tile] = sum;
  }
}

// out[i] = exp_alpha(y[i]) (the rasterizer's exp, for unit tests).
__global__ void __launch_bounds__(256) exp_alpha_kernel(const float* __restrict__ y, int64_t n,
                                                        float* __restrict__ out) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i < n) out[i] = exp_alpha(y[i]);
}

}  // namespace
}  // namespace gsplat_hip

using namespace gsplat_hip;

extern "C" int gsplat_hip_rasterize_count_evals(const float* means2d, const float* conics, const float* opacities,
                                                const uint8_t* masks, const int32_t* tile_offsets,
                                                const int32_t* flatten_ids, int64_t I, int64_t G,
                                                int32_t image_width, int32_t image_height, int32_t tile_size,
                                                int32_t tile_width, int32_t tile_height, int64_t n_isects,
                                                int64_t* tile_evals, void* stream) {
  RasterArgs a{means2d, conics, nullptr, opacities, nullptr, masks, tile_offsets, flatten_ids, G, 1,
               image_width, image_height, tile_size, tile_width, tile_height, I, n_isects, G};
  int rc = check_args(a, "rasterize_count_evals");
  if (rc) return rc;
  if (G < 0) return invalid("rasterize_count_evals: invalid sizes.");
  if (I == 0 || tile_width == 0 || tile_height == 0) return GSPLAT_OK;
  if (!tile_offsets || !tile_evals || (n_isects > 0 && (!flatten_ids || !means2d || !conics || !opacities)))
    return invalid("rasterize_count_evals: null pointer.");
  const dim3 grid(tile_width, tile_height, static_cast<unsigned>(I));
  const int bs = (tile_size * tile_size + kWave - 1) / kWave * kWave;
  raster_count_kernel<<<grid, bs, 0, as_stream(stream)>>>(a, tile_evals);
  return check_launch("rasterize_count_evals");
}

extern "C" int gsplat_hip_exp_alpha_eval(const float* y, int64_t n, float* out, void* stream) {
  if (n < 0) return invalid("exp_alpha_eval: negative size.");
  if (n == 0) return GSPLAT_OK;
  if (!y || !out) return invalid("exp_alpha_eval: null pointer.");
  exp_alpha_kernel<<<grid_for(n, 256), 256, 0, as_stream(stream)>>>(y, n, out);
  return check_launch("exp_alpha_eval");
}

static int rasterize_fwd_impl(const float* means2d, const float* conics, const float* colors,
                              const float* opacities, const float* backgrounds, const uint8_t* masks,
                              const int32_t* tile_offsets, const int32_t* flatten_ids, int64_t I, int64_t N,
                              int64_t G, int32_t channels, int32_t image_width, int32_t image_height,
                              int32_t tile_size, int32_t tile_width, int32_t tile_height, int64_t n_isects,
                              float* render_colors, float* render_alphas, int32_t* last_ids, void* stream) {
  RasterArgs a{means2d, conics, colors, opacities, backgrounds, masks, tile_offsets, flatten_ids, N, channels,
               image_width, image_height, tile_size, tile_width, tile_height, I, n_isects, G};
  if (G < 0) return invalid("rasterize_to_pixels_3dgs_forward: invalid sizes.");
  int rc = check_args(a, "rasterize_to_pixels_3dgs_forward");
  if (rc) return rc;
  if (I == 0 || tile_width == 0 || tile_height == 0) return GSPLAT_OK;
  if (!tile_offsets || !render_colors || !render_alphas || !last_ids || (n_isects > 0 && !flatten_ids))
    return invalid("rasterize_to_pixels_3dgs_forward: null pointer.");
  if (n_isects > 0 && (!means2d || !conics || !colors || !opacities))
    return invalid("rasterize_to_pixels_3dgs_forward: null pointer.");
  const dim3 grid(tile_width, tile_height, static_cast<unsigned>(I));
  const int bs = (tile_size * tile_size + kWave - 1) / kWave * kWave;
  hipStream_t s = as_stream(stream);
  const int ch = channels <= 4 ? channels : 0;
  const size_t sm = fwd_smem(ch, bs);
  KernelTimer timer("raster_fwd", s);
  // records in lanes where that kernel applies and is the faster one, with
  // smaller pixel blocks on small grids
  const int64_t n_total = I * tile_width * static_cast<int64_t>(tile_height);
  if (ch >= 1 && rows_kernels_apply(tile_size, image_width, image_height) &&
      fwd_rows_faster(tile_size, ch, n_total, n_isects / n_total)) {
    const int pixels = tile_size != 16 || n_total > 800 ? 64 : (n_total > 320 ? 32 : 16);
    const int split = 64 / pixels;
    const int n_waves = tile_size * tile_size / 64;
    const int bb = std::min(n_waves * kWave, pixels == 64 ? kRowsSmallBatch : kRowsBatch);
    const size_t rsm = fwd_rows_smem(ch, n_waves, pixels, bb);
    const dim3 rgrid(static_cast<unsigned>(tile_width) * split, tile_height, static_cast<unsigned>(I));
#define GSPLAT_FWD_ROWS(C, P)                                                                             \
  raster_fwd_rows_kernel<C, P><<<rgrid, n_waves * kWave, rsm, s>>>(a, bb, split, render_colors, render_alphas, \
                                                                   last_ids)
#define GSPLAT_FWD_ROWS_P(C)      \
  if (pixels == 64) {             \
    GSPLAT_FWD_ROWS(C, 64);       \
  } else if (pixels == 32) {      \
    GSPLAT_FWD_ROWS(C, 32);       \
  } else {                        \
    GSPLAT_FWD_ROWS(C, 16);       \
  }
    switch (ch) {
      case 1: GSPLAT_FWD_ROWS_P(1); break;
      case 2: GSPLAT_FWD_ROWS_P(2); break;
      case 3: GSPLAT_FWD_ROWS_P(3); break;
      default: GSPLAT_FWD_ROWS_P(4); break;
    }
#undef GSPLAT_FWD_ROWS_P
#undef GSPLAT_FWD_ROWS
    return check_launch("rasterize_to_pixels_3dgs_forward");
  }
  switch (ch) {
    case 1: raster_fwd_kernel<1><<<grid, bs, sm, s>>>(a, render_colors, render_alphas, last_ids); break;
    case 2: raster_fwd_kernel<2><<<grid, bs, sm, s>>>(a, render_colors, render_alphas, last_ids); break;
    case 3: raster_fwd_kernel<3><<<grid, bs, sm, s>>>(a, render_colors, render_alphas, last_ids); break;
    case 4: raster_fwd_kernel<4><<<grid, bs, sm, s>>>(a, render_colors, render_alphas, last_ids); break;
    default: raster_fwd_kernel<0><<<grid, bs, sm, s>>>(a, render_colors, render_alphas, last_ids); break;
  }
  return check_launch("rasterize_to_pixels_3dgs_forward");
}

static int rasterize_bwd_impl(const float* means2d, const float* conics, const float* colors,
                              const float* opacities, const float* backgrounds, const uint8_t* masks,
                              const int32_t* tile_offsets, const int32_t* flatten_ids, int64_t I, int64_t N,
                              int64_t G, int32_t channels, int32_t image_width, int32_t image_height,
                              int32_t tile_size, int32_t tile_width, int32_t tile_height, int64_t n_isects,
                              const float* render_alphas, const int32_t* last_ids, const float* v_render_colors,
                              const float* v_render_alphas, float* v_means2d_abs, float* v_means2d,
                              float* v_conics, float* v_colors, float* v_opacities, float* v_backgrounds,
                              void* workspace, size_t workspace_bytes, void* stream) {
  RasterArgs a{means2d, conics, colors, opacities, backgrounds, masks, tile_offsets, flatten_ids, N, channels,
               image_width, image_height, tile_size, tile_width, tile_height, I, n_isects, G};
  int rc = check_args(a, "rasterize_to_pixels_3dgs_backward");
  if (rc) return rc;
  if (G < 0) return invalid("rasterize_to_pixels_3dgs_backward: invalid sizes.");
  if (!v_means2d || !v_conics || !v_colors || !v_opacities)
    return invalid("rasterize_to_pixels_3dgs_backward: null pointer.");
  if (backgrounds && !v_backgrounds) return invalid("rasterize_to_pixels_3dgs_backward: null v_backgrounds.");
  hipStream_t s = as_stream(stream);
  // outputs are accumulated from zero; the schedule kernel clears them
  // (v_backgrounds is written whole by the order kernel)
  const ZeroSpan spans[] = {{v_means2d, G * 2},
                            {v_conics, G * 3},
                            {v_colors, G * channels},
                            {v_opacities, G},
                            {v_means2d_abs, v_means2d_abs ? G * 2 : 0},
                            {v_backgrounds, backgrounds ? I * channels : 0}};
  if (I == 0 || tile_width == 0 || tile_height == 0) return fill_zero_spans(spans, 6, s);
  const ZeroSpans zero = pack_zero_spans(spans, 5);
  const dim3 grid(tile_width, tile_height, static_cast<unsigned>(I));
  if (!tile_offsets || !render_alphas || !last_ids || !v_render_colors ||
      (n_isects > 0 && (!flatten_ids || !means2d || !conics || !colors || !opacities)))
    return invalid("rasterize_to_pixels_3dgs_backward: null pointer.");
  const int ch = channels <= 4 ? channels : 0;
  const int bs = bwd_block(tile_size);
  const int64_t n_total = I * tile_width * static_cast<int64_t>(tile_height);
  if (n_total > INT32_MAX) return invalid("rasterize_to_pixels_3dgs_backward: too many tiles.");
  if (!workspace || workspace_bytes < bwd_workspace_bytes(n_total, channels)) {
    set_error("rasterize_to_pixels_3dgs_backward: workspace too small.");
    return GSPLAT_ERR_WORKSPACE_TOO_SMALL;
  }
  int32_t* cost = static_cast<int32_t*>(workspace);
  int32_t* order = reinterpret_cast<int32_t*>(static_cast<char*>(workspace) + align256(n_total * 4));
  float* bg_part =
      backgrounds ? reinterpret_cast<float*>(static_cast<char*>(workspace) + 2 * align256(n_total * 4)) : nullptr;
  {
    KernelTimer timer("raster_bwd_schedule", s);
    const dim3 sgrid((tile_width + kStripTiles - 1) / kStripTiles, tile_height, static_cast<unsigned>(I));
    if (tile_size == 16 && ch >= 1) {  // strips of 16-pixel tiles
      switch (ch) {
        case 1: tile_cost_strip_kernel<1><<<sgrid, 256, 0, s>>>(a, last_ids, render_alphas, v_render_colors, cost, bg_part, zero); break;
        case 2: tile_cost_strip_kernel<2><<<sgrid, 256, 0, s>>>(a, last_ids, render_alphas, v_render_colors, cost, bg_part, zero); break;
        case 3: tile_cost_strip_kernel<3><<<sgrid, 256, 0, s>>>(a, last_ids, render_alphas, v_render_colors, cost, bg_part, zero); break;
        default: tile_cost_strip_kernel<4><<<sgrid, 256, 0, s>>>(a, last_ids, render_alphas, v_render_colors, cost, bg_part, zero); break;
      }
    } else {
      switch (ch) {
        case 1: tile_cost_kernel<1><<<grid, 256, 0, s>>>(a, last_ids, render_alphas, v_render_colors, cost, bg_part, zero); break;
        case 2: tile_cost_kernel<2><<<grid, 256, 0, s>>>(a, last_ids, render_alphas, v_render_colors, cost, bg_part, zero); break;
        case 3: tile_cost_kernel<3><<<grid, 256, 0, s>>>(a, last_ids, render_alphas, v_render_colors, cost, bg_part, zero); break;
        case 4: tile_cost_kernel<4><<<grid, 256, 0, s>>>(a, last_ids, render_alphas, v_render_colors, cost, bg_part, zero); break;
        default: tile_cost_kernel<0><<<grid, 256, 0, s>>>(a, last_ids, render_alphas, v_render_colors, cost, bg_part, zero); break;
      }
    }
    // block 0 orders the tiles; one more block per (image, channel) sums the background partials
    const unsigned order_blocks = 1 + (backgrounds ? static_cast<unsigned>(I * channels) : 0u);
    tile_order_kernel<<<order_blocks, kOrderBlock, 0, s>>>(cost, n_total, order, bg_part,
                                                          tile_width * static_cast<int64_t>(tile_height), channels,
                                                          v_backgrounds);
  }
  if ((rc = check_launch("rasterize_to_pixels_3dgs_backward"))) return rc;
  KernelTimer timer("raster_bwd", s);
  const unsigned nb = static_cast<unsigned>(n_total);
  // one block per tile (block b: the tile of rank b in the heavy-first order)
  //
  // Records in lanes where that kernel applies (staged colours, sums of signed
  // gradients only) and is the faster one
  const int64_t per_tile = n_isects / n_total;
  if (ch >= 1 && !v_means2d_abs && rows_kernels_apply(tile_size, image_width, image_height) &&
      bwd_rows_faster(tile_size, ch, n_total, per_tile)) {
    const int bb = bwd_rows_batch(tile_size, bs, ch, n_total, per_tile);
    const size_t sm = bwd_rows_smem(ch, bs, bb);
#define GSPLAT_BWD_ROWS(C)                                                                                     \
  raster_bwd_rows_kernel<C><<<nb, bs, sm, s>>>(a, bb, n_total, order, cost, render_alphas, last_ids,           \
                                               v_render_colors, v_render_alphas, v_means2d, v_conics, v_colors, \
                                               v_opacities)
    switch (ch) {
      case 1: GSPLAT_BWD_ROWS(1); break;
      case 2: GSPLAT_BWD_ROWS(2); break;
      case 3: GSPLAT_BWD_ROWS(3); break;
      default: GSPLAT_BWD_ROWS(4); break;
    }
#undef GSPLAT_BWD_ROWS
    return check_launch("rasterize_to_pixels_3dgs_backward");
  }
  const int bb = bwd_batch(bs);
  const size_t sm = bwd_smem(ch, bs, bb, v_means2d_abs != nullptr);
#define GSPLAT_BWD_LAUNCH(C, ABS_, VABS)                                                                       \
  {                                                                                                            \
    raster_bwd_kernel<C, ABS_><<<nb, bs, sm, s>>>(a, bb, n_total, order, cost, render_alphas, last_ids,       \
                                                  v_render_colors, v_render_alphas, VABS, v_means2d, v_conics, \
                                                  v_colors, v_opacities, v_backgrounds);                        \
  }
#define GSPLAT_BWD_ABS(C)                            \
  if (v_means2d_abs) {                               \
    GSPLAT_BWD_LAUNCH(C, true, v_means2d_abs)        \
  } else {                                           \
    GSPLAT_BWD_LAUNCH(C, false, nullptr)             \
  }
  switch (ch) {
    case 1: GSPLAT_BWD_ABS(1); break;
    case 2: GSPLAT_BWD_ABS(2); break;
    case 3: GSPLAT_BWD_ABS(3); break;
    case 4: GSPLAT_BWD_ABS(4); break;
    default: GSPLAT_BWD_ABS(0); break;
  }
#undef GSPLAT_BWD_ABS
#undef GSPLAT_BWD_LAUNCH
  return check_launch("rasterize_to_pixels_3dgs_backward");
}

extern "C" int gsplat_hip_rasterize_fwd(const float* means2d, const float* conics, const float* colors,
                                        const float* opacities, const float* backgrounds, const uint8_t* masks,
                                        const int32_t* tile_offsets, const int32_t* flatten_ids, int64_t I, int64_t N,
                                        int32_t channels, int32_t image_width, int32_t image_height, int32_t tile_size,
                                        int32_t tile_width, int32_t tile_height, int64_t n_isects,
                                        float* render_colors, float* render_alphas, int32_t* last_ids, void* stream) {
  return rasterize_fwd_impl(means2d, conics, colors, opacities, backgrounds, masks, tile_offsets, flatten_ids, I, N,
                            I * N, channels, image_width, image_height, tile_size, tile_width, tile_height, n_isects,
                            render_colors, render_alphas, last_ids, stream);
}

extern "C" int gsplat_hip_rasterize_fwd_packed(const float* means2d, const float* conics, const float* colors,
                                               const float* opacities, const float* backgrounds,
                                               const uint8_t* masks, const int32_t* tile_offsets,
                                               const int32_t* flatten_ids, int64_t I, int64_t nnz, int32_t channels,
                                               int32_t image_width, int32_t image_height, int32_t tile_size,
                                               int32_t tile_width, int32_t tile_height, int64_t n_isects,
                                               float* render_colors, float* render_alphas, int32_t* last_ids,
                                               void* stream) {
  return rasterize_fwd_impl(means2d, conics, colors, opacities, backgrounds, masks, tile_offsets, flatten_ids, I, nnz,
                            nnz, channels, image_width, image_height, tile_size, tile_width, tile_height, n_isects,
                            render_colors, render_alphas, last_ids, stream);
}

extern "C" int gsplat_hip_rasterize_bwd(const float* means2d, const float* conics, const float* colors,
                                        const float* opacities, const float* backgrounds, const uint8_t* masks,
                                        const int32_t* tile_offsets, const int32_t* flatten_ids, int64_t I, int64_t N,
                                        int32_t channels, int32_t image_width, int32_t image_height, int32_t tile_size,
                                        int32_t tile_width, int32_t tile_height, int64_t n_isects,
                                        const float* render_alphas, const int32_t* last_ids,
                                        const float* v_render_colors, const float* v_render_alphas,
                                        float* v_means2d_abs, float* v_means2d, float* v_conics, float* v_colors,
                                        float* v_opacities, float* v_backgrounds, void* workspace,
                                        size_t workspace_bytes, void* stream) {
  return rasterize_bwd_impl(means2d, conics, colors, opacities, backgrounds, masks, tile_offsets, flatten_ids, I, N,
                            I * N, channels, image_width, image_height, tile_size, tile_width, tile_height, n_isects,
                            render_alphas, last_ids, v_render_colors, v_render_alphas, v_means2d_abs, v_means2d,
                            v_conics, v_colors, v_opacities, v_backgrounds, workspace, workspace_bytes, stream);
}

extern "C" int gsplat_hip_rasterize_bwd_packed(const float* means2d, const float* conics, const float* colors,
                                               const float* opacities, const float* backgrounds,
                                               const uint8_t* masks, const int32_t* tile_offsets,
                                               const int32_t* flatten_ids, int64_t I, int64_t nnz, int32_t channels,
                                               int32_t image_width, int32_t image_height, int32_t tile_size,
                                               int32_t tile_width, int32_t tile_height, int64_t n_isects,
                                               const float* render_alphas, const int32_t* last_ids,
                                               const float* v_render_colors, const float* v_render_alphas,
                                               float* v_means2d_abs, float* v_means2d, float* v_conics,
                                               float* v_colors, float* v_opacities, float* v_backgrounds,
                                               void* workspace, size_t workspace_bytes, void* stream) {
  return rasterize_bwd_impl(means2d, conics, colors, opacities, backgrounds, masks, tile_offsets, flatten_ids, I, nnz,
                            nnz, channels, image_width, image_height, tile_size, tile_width, tile_height, n_isects,
                            render_alphas, last_ids, v_render_colors, v_render_alphas, v_means2d_abs, v_means2d,
                            v_conics, v_colors, v_opacities, v_backgrounds, workspace, workspace_bytes, stream);
}

// Device address of `scratch` on the current device, looked up once per
// device (hipGetSymbolAddress with that device current) and kept.
static int noalloc_scratch(void** ptr, const char* what) {
  constexpr int kMaxDevices = 64;
  static std::atomic<void*> cache[kMaxDevices];
  static std::mutex mu;
  int dev = 0;
  int rc = check_hip(hipGetDevice(&dev), what);
  if (rc) return rc;
  if (dev < 0 || dev >= kMaxDevices) return invalid(std::string(what) + ": device index out of range.");
  void* p = cache[dev].load(std::memory_order_acquire);
  if (!p) {
    std::lock_guard<std::mutex> lock(mu);
    p = cache[dev].load(std::memory_order_relaxed);
    if (!p) {
      if ((rc = check_hip(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), what))) return rc;
      if (!p) return invalid(std::string(what) + ": no scratch address.");
      cache[dev].store(p, std::memory_order_release);
    }
  }
  *ptr = p;
  return GSPLAT_OK;
}

extern "C" size_t gsplat_hip_rasterize_bwd_noalloc_max_scratch(void) { return kNoAllocScratchBytes; }

extern "C" int gsplat_hip_rasterize_bwd_noalloc(const float* means2d, const float* conics, const float* colors,
                                                const float* opacities, const float* backgrounds,
                                                const uint8_t* masks, const int32_t* tile_offsets,
                                                const int32_t* flatten_ids, int64_t I, int64_t N, int32_t channels,
                                                int32_t image_width, int32_t image_height, int32_t tile_size,
                                                int32_t tile_width, int32_t tile_height, int64_t n_isects,
                                                const float* render_alphas, const int32_t* last_ids,
                                                const float* v_render_colors, const float* v_render_alphas,
                                                float* v_means2d_abs, float* v_means2d, float* v_conics,
                                                float* v_colors, float* v_opacities, float* v_backgrounds,
                                                void* stream) {
  const char* what = "rasterize_to_pixels_3dgs_backward_noalloc";
  RasterArgs a{means2d, conics, colors, opacities, backgrounds, masks, tile_offsets, flatten_ids, N, channels,
               image_width, image_height, tile_size, tile_width, tile_height, I, n_isects, I * N};
  int rc = check_args(a, what);
  if (rc) return rc;
  const int64_t n_total = I * tile_width * static_cast<int64_t>(tile_height);
  // every schedule word and background partial the kernels read is written
  // earlier in the same call, so nothing in the scratch needs clearing
  if (n_total > 0 && bwd_workspace_bytes(n_total, channels) > kNoAllocScratchBytes)
    return invalid(std::string(what) + ": the tile schedule needs " +
                   std::to_string(bwd_workspace_bytes(n_total, channels)) + " bytes (images * tiles * (8 + 4 * " +
                   "channels), rounded), more than the " + std::to_string(kNoAllocScratchBytes) +
                   "-byte static scratch; use gsplat_hip_rasterize_bwd with a workspace.");
  void* ws = nullptr;
  if ((rc = noalloc_scratch(&ws, what))) return rc;
  return rasterize_bwd_impl(means2d, conics, colors, opacities, backgrounds, masks, tile_offsets, flatten_ids, I, N,
                            I * N, channels, image_width, image_height, tile_size, tile_width, tile_height, n_isects,
                            render_alphas, last_ids, v_render_colors, v_render_alphas, v_means2d_abs, v_means2d,
                            v_conics, v_colors, v_opacities, v_backgrounds, ws, kNoAllocScratchBytes, stream);
}

static int raster_indices_args(const char* what, const RasterArgs& a) {
  int rc = check_args(a, what);
  if (rc) return rc;
  if (a.ts * a.ts > 1024) return invalid(std::string(what) + ": tile_size must be at most 32.");
  if (a.I > 0 && a.tw > 0 && a.th > 0 && (!a.tile_offsets || (a.n_isects > 0 && !a.flatten_ids)))
    return invalid(std::string(what) + ": null pointer.");
  if (a.n_isects > 0 && (!a.means2d || !a.conics || !a.opacities)) return invalid(std::string(what) + ": null pointer.");
  return GSPLAT_OK;
}

extern "C" size_t gsplat_hip_rasterize_to_indices_workspace_size(int64_t I, int32_t image_width,
                                                                 int32_t image_height) {
  return scan_workspace_bytes(I * image_width * static_cast<int64_t>(image_height));
}

extern "C" int gsplat_hip_rasterize_to_indices_count(int64_t range_start, int64_t range_end,
                                                     const float* transmittances, const float* means2d,
                                                     const float* conics, const float* opacities,
                                                     const int32_t* tile_offsets, const int32_t* flatten_ids,
                                                     int64_t I, int64_t n_rows, int32_t image_width,
                                                     int32_t image_height, int32_t tile_size, int32_t tile_width,
                                                     int32_t tile_height, int64_t n_isects, int32_t* starts,
                                                     int64_t* total_dev, void* workspace, size_t workspace_bytes,
                                                     void* stream) {
  const char* what = "rasterize_to_indices_3dgs";
  RasterArgs a{means2d, conics, nullptr, opacities, nullptr, nullptr, tile_offsets, flatten_ids, n_rows, 1,
               image_width, image_height, tile_size, tile_width, tile_height, I, n_isects, n_rows};
  int rc = raster_indices_args(what, a);
  if (rc) return rc;
  if (!total_dev) return invalid(std::string(what) + ": null total.");
  hipStream_t s = as_stream(stream);
  const int64_t n_pix = I * image_width * static_cast<int64_t>(image_height);
  if (n_pix == 0 || tile_width == 0 || tile_height == 0) return fill_zero(total_dev, sizeof(int64_t), s);
  if (!starts) return invalid(std::string(what) + ": null pointer.");
  if (!workspace || workspace_bytes < scan_workspace_bytes(n_pix)) {
    set_error(std::string(what) + ": workspace too small.");
    return GSPLAT_ERR_WORKSPACE_TOO_SMALL;
  }
  const int bs = (tile_size * tile_size + kWave - 1) / kWave * kWave;
  {
    KernelTimer timer("raster_indices", s);
    raster_indices_kernel<false><<<dim3(tile_width, tile_height, static_cast<unsigned>(I)), bs, 0, s>>>(
        a, range_start, range_end, transmittances, starts, nullptr, 0, nullptr, nullptr);
  }
  if ((rc = check_launch(what))) return rc;
  return scan_exclusive_i32(starts, starts, n_pix, total_dev, workspace, s);
}

extern "C" int gsplat_hip_rasterize_to_indices_write(int64_t range_start, int64_t range_end,
                                                     const float* transmittances, const float* means2d,
                                                     const float* conics, const float* opacities,
                                                     const int32_t* tile_offsets, const int32_t* flatten_ids,
                                                     int64_t I, int64_t n_rows, int32_t image_width,
                                                     int32_t image_height, int32_t tile_size, int32_t tile_width,
                                                     int32_t tile_height, int64_t n_isects, const int32_t* starts,
                                                     int64_t n_out, int32_t* out_gauss_ids, int64_t* out_indices,
                                                     void* stream) {
  const char* what = "rasterize_to_indices_3dgs";
  RasterArgs a{means2d, conics, nullptr, opacities, nullptr, nullptr, tile_offsets, flatten_ids, n_rows, 1,
               image_width, image_height, tile_size, tile_width, tile_height, I, n_isects, n_rows};
  int rc = raster_indices_args(what, a);
  if (rc) return rc;
  if (n_out < 0) return invalid(std::string(what) + ": negative output size.");
  const int64_t n_pix = I * image_width * static_cast<int64_t>(image_height);
  if (n_pix == 0 || tile_width == 0 || tile_height == 0 || n_out == 0) return GSPLAT_OK;
  if (!starts || !out_gauss_ids || !out_indices) return invalid(std::string(what) + ": null pointer.");
  hipStream_t s = as_stream(stream);
  const int bs = (tile_size * tile_size + kWave - 1) / kWave * kWave;
  {
    KernelTimer timer("raster_indices", s);
    raster_indices_kernel<true><<<dim3(tile_width, tile_height, static_cast<unsigned>(I)), bs, 0, s>>>(
        a, range_start, range_end, transmittances, nullptr, starts, n_out, out_gauss_ids, out_indices);
  }
  return check_launch(what);
}

extern "C" size_t gsplat_hip_rasterize_bwd_workspace_size(int64_t I, int32_t channels, int32_t tile_width,
                                                          int32_t tile_height) {
  if (I <= 0 || tile_width <= 0 || tile_height <= 0 || channels <= 0) return 0;
  return bwd_workspace_bytes(I * tile_width * static_cast<int64_t>(tile_height), channels);
}
