// render.hip -- the render path the reference delegates to its external
// instant-ngp renderer (src/server.cpp:161-194 sends a FrameRequest and waits
// for RGB + depth): ray generation, occupancy-grid march, 16-level hash-grid
// encoding, density/colour MLPs and volume compositing.
//
// Pipeline per pass (a pass covers a window of march steps; one pass of 128
// steps is the default):
//   march_emit    one thread per ray slot (march_emit_split: four, for few
//                 rays): camera ray, box clip, occupied steps; one atomic per
//                 workgroup reserves a contiguous segment of the sample list
//                 on the device, one part per wavefront's tile
//   encode_parts  16-level hash-grid encoding, XCD-partitioned: workgroups on
//                 XCD p encode levels p and 15-p, so each XCD's L2 caches two
//                 levels of the table
//   MLPs          density + colour MLPs over the dense sample list:
//                   FP32:  mlp_f32 (train.hip), FP32 features on
//                          v_mfma_f32_16x16x4_f32
//                   mixed: mlp_mixed, FP16 features on
//                          v_mfma_f32_16x16x32_f16, FP32 accumulation
//   composite     one thread per ray (composite_split: four, for few rays):
//                 front-to-back alpha compositing in FP32, stops at T < 1e-4,
//                 writes RGB24 / depth / float RGB
// frame_begin clears the frame's counters, frame_end stores them, and outputs
// wanted in pinned memory, on the host's side.
// Both precisions share every kernel except the table type in encode_parts,
// the MLP kernel and the width of the MLP output, so their throughput ratio
// isolates those; both MLPs run on matrix cores.  The sample
// total stays on the device (no host round trip inside a render).
//
// Sample geometry (ray, box clip, step positions, occupancy cell) is defined
// in FP32 with explicit fused multiply-adds and correctly rounded division and
// square root, so every implementation visits the same samples.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "device_common.h"

namespace nes {

// ----------------------------------------------------------- march kernel
// One kernel for both march walks: count this ray's occupied steps, reserve
// the workgroup's range of the sample list (one atomic per workgroup on a
// device-side cursor), then write the records in rank-major order.  The
// sample total never leaves the device: later kernels read it from the
// cursor, and writes beyond `capacity` are dropped (the host re-renders with a
// larger buffer when the final total exceeds it).  counts[slot] receives the
// ray's sample count, flags and resume step (see kCountMask), offsets[wavefront]
// the wavefront's range start.  A ray emits at most `cap` samples per pass;
// with `resume` it starts where its previous pass stopped.
//
// Bound by VALU in frames (a wavefront whose rays cross the cube runs about
// 50 to 100 steps and then its longest ray's samples) and by the chain of
// dependent steps in small ones, so: tiles that cannot see the cube are left
// after a test of a few instructions; positions are scaled by powers of two
// inside the fused multiply-add (exact) instead of after it; kStepUnroll
// occupancy words are in flight at once.  One atomic per workgroup: the cursor
// is a single address and takes about 1e8 atomics per second.  Rays without
// samples store nothing but their count.  Stereo 1080p (4.1 M rays, 10.3 M
// samples): 102 -> 75 us; 64x48: 33 -> 25 us.
enum MarchMode : int {
  kMarchFirst,     // rays from the views
  kMarchNext,      // a later pass over rays the first one stored
  kMarchPrepared,  // rays prepared by the caller (training)
};
struct MarchArgs {
  const ViewDesc *views;
  uint32_t n_views, n_slots;
  const uint32_t *occ;
  RayData *rays;
  uint32_t *counts, *offsets, *samples;
  float *t_start;
  float4 *pos;
  uint32_t *cursor;  // the pass's sample cursor (a word of RenderWork::total)
  uint32_t capacity, cap;
  int k_begin, k_end, mode, packed;
  int resume;      // kMarchNext: every ray with samples left has kRayState, go on at its step
  int store_rays;  // kMarchFirst: 0 none (single pass), 1 rays with samples, 2 every ray
  uint2 *ray_sh;
  uint32_t *tile_n;  // kMarchFirst: samples per wavefront
  uint64_t *stamp;  // device clock at the kernel's start (optional)
};

// The device's 100 MHz clock at the start of a kernel, from its first
// workgroup.  Stage times come from these stamps: hipEventRecord between the
// kernels costs about 5 us of idle device time each (six of them in a chain of
// five empty launches: 20 -> 52 us).
__device__ __forceinline__ void stamp_start(uint64_t *stamp) {
  if (stamp && blockIdx.x == 0 && threadIdx.x == 0) *stamp = wall_clock64();
}

// The view of a wavefront's ray slots (views start on tile boundaries).
__device__ __forceinline__ uint32_t view_of(const ViewDesc *views, uint32_t n_views, uint32_t slot) {
  uint32_t vi = 0;
  for (uint32_t i = 1; i < n_views; ++i)
    if (slot >= views[i].slot_base) vi = i;
  return vi;
}

// Whether no ray of the 8x8 tile at pixel (px, py) can come near the cube.  A
// pixel's direction is dc + e with dc the tile centre's and |e| <= tile_reach;
// a sphere around the cube of radius R, c away from the eye, is missed by all
// of them if |t dc - c| > R + t |e| for every t >= 0.  R is 0.4 % above the
// cube's, far above the rounding of the ray arithmetic at these distances;
// farther eyes and non-finite cameras are never left out.
__device__ __forceinline__ bool tile_misses(const ViewDesc &v, uint32_t px, uint32_t py) {
  constexpr float kR = 0.87f;
  const float u = ((float)px + 4.0f - 0.5f * (float)v.width) * v.inv_focal;
  const float w = ((float)py + 4.0f - 0.5f * (float)v.height) * v.inv_focal;
  float s = 0.0f, len2 = 0.0f, c2 = 0.0f;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const float d = fmaf(v.c2w[4 * i + 0], u, fmaf(v.c2w[4 * i + 1], w, v.c2w[4 * i + 2]));
    const float c = 0.5f - v.c2w[4 * i + 3];
    s = fmaf(d, c, s);
    len2 = fmaf(d, d, len2);
    c2 = fmaf(c, c, c2);
  }
  const float a = 0.9999f * len2 - v.tile_reach * v.tile_reach;
  const float k = c2 - kR * kR, b = s + kR * v.tile_reach;
  return k > 0.01f && c2 < 1e6f && len2 < 1e30f && a > 0.0f && (b <= 0.0f || b * b < a * k);
}

constexpr int kStepUnroll = 8;
static_assert(32 % kStepUnroll == 0, "a group's bits lie in one word");

__global__ __launch_bounds__(256) void march_emit(MarchArgs m) {
  stamp_start(m.stamp);
  __shared__ uint32_t wave_n[4];
  __shared__ uint32_t block_base;
  const uint32_t slot = blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = lane_id();
  const uint32_t wave = threadIdx.x >> 6;
  uint32_t cnt = 0;
  uint32_t state = 0;
  uint32_t knext = kMaxSteps;           // where a later pass resumes this ray
  uint32_t bits[4] = {0u, 0u, 0u, 0u};  // occupied steps of this pass
  RayData r;
  r.n_steps = 0;
  int k = m.k_begin;
  if (slot < m.n_slots) {
    if (m.mode == kMarchFirst) {
      const uint32_t wslot = __builtin_amdgcn_readfirstlane(slot);
      const ViewDesc &v = m.views[view_of(m.views, m.n_views, wslot)];
      const uint32_t tile = (wslot - v.slot_base) >> 6;
      const uint32_t px0 = (tile % v.tiles_x) * 8, py0 = (tile / v.tiles_x) * 8;
      const uint32_t px = px0 + (lane & 7), py = py0 + (lane >> 3);
      if (!tile_misses(v, px0, py0) && px < v.width && py < v.height) {
        make_ray(v, px, py, r.o, r.d);
        r.n_steps = ray_box(r.o, r.d, &r.t_start);
      } else {
        r.o[0] = r.o[1] = r.o[2] = 0.0f;
        r.d[0] = r.d[1] = r.d[2] = 0.0f;
        r.t_start = 0.0f;
      }
      if (m.store_rays == 2) m.rays[slot] = r;
    } else if (m.mode == kMarchPrepared) {
      r = load_ray(m.rays, slot);
    } else {
      const uint32_t prev = m.counts[slot];
      state = prev & (kRayState | kRayDone);
      if (!(prev & kRayDone) && (!m.resume || (prev & kRayState))) r = load_ray(m.rays, slot);
      if (m.resume) k = max(k, (int)(prev >> 16));
    }
    const int kend = min(m.k_end, (int)r.n_steps);
    if (k < kend) {
      // positions times 128, as the occupancy cells need them: scaling by a
      // power of two commutes with the rounding of the fused multiply-add
      float o128[3], d128[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        o128[a] = 128.0f * r.o[a];
        d128[a] = 128.0f * r.d[a];
      }
      knext = (uint32_t)kend;
      const int k0 = k;
      // groups of kStepUnroll steps: the occupancy words are loaded together
      // (unconditionally: the clamped cell index is inside the bitfield
      // before k0 and past kend too), then taken in order
      for (k &= ~(kStepUnroll - 1); k < kend; k += kStepUnroll) {
        uint32_t word[kStepUnroll], cell[kStepUnroll];
        const float kf = (float)k + 0.5f;
#pragma unroll
        for (int u = 0; u < kStepUnroll; ++u) {
          const float t = fmaf(kf + (float)u, kDelta, r.t_start);
          float x[3];
#pragma unroll
          for (int a = 0; a < 3; ++a) x[a] = fmaf(t, d128[a], o128[a]);
          cell[u] = occ_cell(x);
          word[u] = __ldg(m.occ + (cell[u] >> 5));
        }
        uint32_t hit = 0;
#pragma unroll
        for (int u = 0; u < kStepUnroll; ++u) hit |= ((word[u] >> (cell[u] & 31u)) & 1u) << u;
        if (k < k0) hit &= ~0u << (k0 - k);
        if (kend - k < kStepUnroll) hit &= (1u << (kend - k)) - 1u;
        cnt += (uint32_t)__popc(hit);
        if (cnt >= m.cap) {  // drop what lies behind the cap-th sample
          for (; cnt > m.cap; --cnt) hit &= ~(0x80000000u >> __clz(hit));
          knext = (uint32_t)(k + 32 - __clz(hit));
        }
        const uint32_t at = hit << (k & 31);
        const int wd = k >> 5;
#pragma unroll
        for (int i = 0; i < 4; ++i) bits[i] |= wd == i ? at : 0u;
        if (cnt >= m.cap) break;
      }
    } else {
      knext = (uint32_t)max(kend, k);
    }
    m.counts[slot] = cnt | state | (knext << 16);
    if (cnt) {
      m.t_start[slot] = r.t_start;
      if (m.store_rays == 1) m.rays[slot] = r;
    }
  }
  if (m.ray_sh && cnt) {
    // the colour MLP's SH input of this ray, in FP16 (mixed path); written by
    // every pass in which the ray has samples
    float sh[16];
    sh4(r.d, sh);
    uint32_t hw[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      half2v h;
      h[0] = (_Float16)sh[2 * i];
      h[1] = (_Float16)sh[2 * i + 1];
      hw[i] = __builtin_bit_cast(uint32_t, h);
    }
    uint4 *dst = reinterpret_cast<uint4 *>(m.ray_sh + (size_t)slot * 4);
    dst[0] = make_uint4(hw[0], hw[1], hw[2], hw[3]);
    dst[1] = make_uint4(hw[4], hw[5], hw[6], hw[7]);
  }
  // the workgroup's range of the sample list, one part per wavefront
  const uint32_t wave_total = wave_sum(cnt);
  if (lane == 0) {
    wave_n[wave] = wave_total;
    if (m.mode == kMarchFirst && slot < m.n_slots) m.tile_n[slot >> 6] = wave_total;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t n = wave_n[0] + wave_n[1] + wave_n[2] + wave_n[3];
    block_base = n ? atomicAdd(m.cursor, n) : 0u;
  }
  __syncthreads();
  if (wave_total == 0) return;
  uint32_t base = block_base;
  for (uint32_t i = 0; i < wave; ++i) base += wave_n[i];
  if (lane == 0) m.offsets[slot >> 6] = base;
  const uint32_t mx = wave_max(cnt);
  // packed positions are multiples of 2^-21 (the scaling is exact as above)
  const float scale = m.packed ? 2097152.0f : 1.0f;
  float os[3], ds[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    os[a] = scale * r.o[a];
    ds[a] = scale * r.d[a];
  }
  uint32_t at0 = base;  // start of the current rank
  int wd = 0;
  uint32_t b = bits[0];
  for (uint32_t i = 0; i < mx; ++i) {  // wavefront-uniform
    const uint64_t has = __ballot(cnt > i);
    if (cnt > i) {
      while (b == 0) {
        ++wd;
        b = wd == 1 ? bits[1] : wd == 2 ? bits[2] : bits[3];
      }
      const int ks = 32 * wd + __builtin_ctz(b);
      b &= b - 1;
      const uint32_t at =
          at0 + __builtin_amdgcn_mbcnt_hi((uint32_t)(has >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)has, 0u));
      if (at < m.capacity) {
        const float t = step_t(ks, r.t_start);
        float x[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) x[a] = fmaf(t, ds[a], os[a]);
        if (m.packed)
          reinterpret_cast<uint2 *>(m.pos)[at] = pack_pos21(x);
        else
          m.pos[at] = make_float4(fminf(fmaxf(x[0], 0.0f), 1.0f), fminf(fmaxf(x[1], 0.0f), 1.0f),
                                  fminf(fmaxf(x[2], 0.0f), 1.0f), __uint_as_float(slot));
        m.samples[at] = (slot << 7) | (uint32_t)ks;
      }
    }
    at0 += (uint32_t)__popcll(has);
  }
}


// The same for few rays, which leave the chip idle while each wavefront works
// through its chain of steps and samples: one workgroup per tile, four lanes
// per ray, each testing a quarter of the ray's steps and emitting what it
// found.  The list is laid out as march_emit lays it out: rank r of ray l at
// start[r] + |{rays < l with more than r samples}|, from the ranks' ray masks.
// 64x48: 24.0 -> 11.4 us, 320x240: 24.6 -> 14.5 us, 4096 rays of a batch:
// 29 -> 14 us.
__global__ __launch_bounds__(256) void march_emit_split(MarchArgs m) {
  stamp_start(m.stamp);
  __shared__ uint32_t ray_n[64];
  __shared__ uint64_t rank_rays[kMaxSteps];
  __shared__ uint32_t rank_at[kMaxSteps];
  __shared__ uint32_t block_base;
  const int lane = lane_id();
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t ray = threadIdx.x >> 2, seg = threadIdx.x & 3u;
  const uint32_t slot = blockIdx.x * 64 + ray;
  const bool valid = slot < m.n_slots;
  RayData r;
  r.n_steps = 0;
  uint32_t state = 0;
  int k = m.k_begin;
  if (m.mode == kMarchFirst) {
    const uint32_t tslot = blockIdx.x * 64;
    const ViewDesc &v = m.views[view_of(m.views, m.n_views, tslot)];
    const uint32_t tile = (tslot - v.slot_base) >> 6;
    const uint32_t px0 = (tile % v.tiles_x) * 8, py0 = (tile / v.tiles_x) * 8;
    const uint32_t px = px0 + (ray & 7), py = py0 + (ray >> 3);
    if (!tile_misses(v, px0, py0) && px < v.width && py < v.height) {
      make_ray(v, px, py, r.o, r.d);
      r.n_steps = ray_box(r.o, r.d, &r.t_start);
    } else {
      r.o[0] = r.o[1] = r.o[2] = 0.0f;
      r.d[0] = r.d[1] = r.d[2] = 0.0f;
      r.t_start = 0.0f;
    }
    if (m.store_rays == 2 && seg == 0) m.rays[slot] = r;
  } else if (valid) {
    if (m.mode == kMarchPrepared) {
      r = load_ray(m.rays, slot);
    } else {
      const uint32_t prev = m.counts[slot];
      state = prev & (kRayState | kRayDone);
      if (!(prev & kRayDone) && (!m.resume || (prev & kRayState))) r = load_ray(m.rays, slot);
      if (m.resume) k = max(k, (int)(prev >> 16));
    }
  }
  // this lane's quarter of the ray's steps
  const int kend = min(m.k_end, (int)r.n_steps);
  const int quarter = (max(kend - k, 0) + 3) >> 2;
  const int k0 = k + (int)seg * quarter, k1 = min(k0 + quarter, kend);
  uint32_t hits = 0;  // occupied steps, from k0 on
  if (k0 < k1) {
    float o128[3], d128[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      o128[a] = 128.0f * r.o[a];
      d128[a] = 128.0f * r.d[a];
    }
    for (int g = k0; g < k1; g += kStepUnroll) {
      uint32_t word[kStepUnroll], cell[kStepUnroll];
      const float kf = (float)g + 0.5f;
#pragma unroll
      for (int u = 0; u < kStepUnroll; ++u) {
        const float t = fmaf(kf + (float)u, kDelta, r.t_start);
        float x[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) x[a] = fmaf(t, d128[a], o128[a]);
        cell[u] = occ_cell(x);
        word[u] = __ldg(m.occ + (cell[u] >> 5));
      }
      uint32_t hit = 0;
#pragma unroll
      for (int u = 0; u < kStepUnroll; ++u) hit |= ((word[u] >> (cell[u] & 31u)) & 1u) << u;
      if (k1 - g < kStepUnroll) hit &= (1u << (k1 - g)) - 1u;
      hits |= hit << (g - k0);
    }
  }
  // samples of the ray's earlier quarters and of all of them, cut at the cap
  uint32_t n = (uint32_t)__popc(hits), before = 0, all = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint32_t c = (uint32_t)__shfl((int)n, (lane & ~3) + q);
    if (q < (int)seg) before += c;
    all += c;
  }
  uint32_t knext = (uint32_t)max(kend, k);
  if (all >= m.cap) {
    const uint32_t keep = before < m.cap ? min(n, m.cap - before) : 0u;
    for (; n > keep; --n) hits &= ~(0x80000000u >> __clz(hits));
    // one step past the cap-th sample, which one lane of the ray holds
    uint32_t past = n && before + n == m.cap ? (uint32_t)(k0 + 32 - __clz(hits)) : 0u;
    past = max(past, (uint32_t)__shfl_xor((int)past, 1));
    past = max(past, (uint32_t)__shfl_xor((int)past, 2));
    knext = past;
    all = m.cap;
  }
  if (valid && seg == 0) {
    m.counts[slot] = all | state | (knext << 16);
    if (all) {
      m.t_start[slot] = r.t_start;
      if (m.store_rays == 1) m.rays[slot] = r;
    }
  }
  if (seg == 0) ray_n[ray] = all;
  if (m.ray_sh && all) {
    // the colour MLP's SH input of this ray, a quarter per lane
    float sh[16];
    sh4(r.d, sh);
    uint32_t hw[2] = {0u, 0u};
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (q == (int)seg)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          half2v h;
          h[0] = (_Float16)sh[4 * q + 2 * i];
          h[1] = (_Float16)sh[4 * q + 2 * i + 1];
          hw[i] = __builtin_bit_cast(uint32_t, h);
        }
    m.ray_sh[(size_t)slot * 4 + seg] = make_uint2(hw[0], hw[1]);
  }
  __syncthreads();
  // every wavefront sees the 64 counts; the ranks' masks are dealt to them
  const uint32_t c = ray_n[lane];
  const uint32_t mx = wave_max(c);
  if (wave == 0) {
    const uint32_t total = wave_sum(c);
    if (lane == 0) {
      block_base = total ? atomicAdd(m.cursor, total) : 0u;
      if (m.mode == kMarchFirst) m.tile_n[blockIdx.x] = total;
      if (total) m.offsets[blockIdx.x] = block_base;
    }
  }
  if (mx == 0) return;  // the same in every wavefront
  index_ranks(c, mx, rank_rays, rank_at);
  const uint32_t base = block_base;
  const uint64_t below = lanes_below((int)ray);
  const float scale = m.packed ? 2097152.0f : 1.0f;
  float os[3], ds[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    os[a] = scale * r.o[a];
    ds[a] = scale * r.d[a];
  }
  for (uint32_t rank = before; hits; ++rank) {
    const int ks = k0 + __builtin_ctz(hits);
    hits &= hits - 1;
    const uint32_t at = base + rank_at[rank] + (uint32_t)__popcll(rank_rays[rank] & below);
    if (at >= m.capacity) continue;
    const float t = step_t(ks, r.t_start);
    float x[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) x[a] = fmaf(t, ds[a], os[a]);
    if (m.packed)
      reinterpret_cast<uint2 *>(m.pos)[at] = pack_pos21(x);
    else
      m.pos[at] = make_float4(fminf(fmaxf(x[0], 0.0f), 1.0f), fminf(fmaxf(x[1], 0.0f), 1.0f),
                              fminf(fmaxf(x[2], 0.0f), 1.0f), __uint_as_float(slot));
    m.samples[at] = (slot << 7) | (uint32_t)ks;
  }
}

// Ray slots up to which the march runs four lanes per ray.  Past that the chip
// is full either way and a ray's set-up, done by all four, costs more than the
// shorter chains give (march_emit -> march_emit_split, us): 173k slots
// 24.6 -> 16.5, 307k 25.9 -> 24.3, 614k 29.7 -> 29.9, 1.0M 39.6 -> 45.2,
// 4.1M 73 -> 135.
constexpr uint32_t kSplitSlots = 1u << 19;
// The same for a batch of rays, whose tiles all have rays that cross the cube,
// where a frame's mostly miss it: 16k rays 25.1 -> 14.8, 65k 23.8 -> 25.0,
// 131k 27 -> 38.
constexpr uint32_t kSplitBatchRays = 1u << 15;

static int launch_march(const MarchArgs &m, hipStream_t stream) {
  if (m.n_slots <= (m.mode == kMarchPrepared ? kSplitBatchRays : kSplitSlots))
    march_emit_split<<<(unsigned)((m.n_slots + 63) / 64), 256, 0, stream>>>(m);
  else
    march_emit<<<(unsigned)((m.n_slots + 255) / 256), 256, 0, stream>>>(m);
  NES_HIP_TRY(hipGetLastError());
  return NES_OK;
}

constexpr int kEvalWaves = 4;

// ------------------------------------------------------ FP32 VALU eval
// The plain FP32 path: FP32 table features, one lane per sample, every MAC a
// VALU FMA with the weights in LDS (wave-uniform broadcasts).
template <int NI, int NO, bool kRelu>
__device__ __forceinline__ void dense_f32(const float *w, const float *in, float *out) {
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    float acc = 0.0f;
#pragma unroll
    for (int i = 0; i < NI; ++i) acc = fmaf(w[o * NI + i], in[i], acc);
    out[o] = kRelu ? fmaxf(acc, 0.0f) : acc;
    // keep the scheduler from hoisting every weight read of the layer
    if ((o & 3) == 3) __asm__ volatile("" ::: "memory");
  }
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void mlp_fp32_valu(
    const float4 *__restrict__ pos, const float4 *__restrict__ feat,
    const uint32_t *__restrict__ n_ptr, uint32_t stride, const RayData *__restrict__ rays,
    const float *__restrict__ Wg, float4 *__restrict__ out, uint64_t *stamp) {
  stamp_start(stamp);
  const uint32_t n = min(*n_ptr, stride);
  __shared__ __attribute__((aligned(16))) float W[kWeights];
  for (int i = (int)threadIdx.x; i < kWeights / 4; i += (int)blockDim.x)
    reinterpret_cast<float4 *>(W)[i] = reinterpret_cast<const float4 *>(Wg)[i];
  __syncthreads();
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    float f[32];
#pragma unroll
    for (int p = 0; p < kParts; ++p) {
      const float4 v = feat[(size_t)p * stride + i];
      f[part_feature(p, 0)] = v.x;
      f[part_feature(p, 1)] = v.y;
      f[part_feature(p, 2)] = v.z;
      f[part_feature(p, 3)] = v.w;
    }
    const RayData r = load_ray(rays, __float_as_uint(pos[i].w));
    float h1[64], o2[16], in3[31], h3[64], h4[64], o5[3], sh[16];
    dense_f32<32, 64, true>(W + kW1, f, h1);
    dense_f32<64, 16, false>(W + kW2, h1, o2);
    sh4(r.d, sh);
#pragma unroll
    for (int k = 0; k < 16; ++k) in3[k] = sh[k];
#pragma unroll
    for (int k = 0; k < 15; ++k) in3[16 + k] = o2[1 + k];
    dense_f32<31, 64, true>(W + kW3, in3, h3);
    dense_f32<64, 64, true>(W + kW4, h3, h4);
    dense_f32<64, 3, false>(W + kW5, h4, o5);
    out[i] = make_float4(expf(o2[0]), sigmoidf_(o5[0]), sigmoidf_(o5[1]), sigmoidf_(o5[2]));
  }
}

// ----------------------------------------------------------- mixed eval
// MFMA tile: v_mfma_f32_16x16x32_f16, D[16x16] += A[16x32] B[32x16].
// Rows (M) are output neurons, columns (N) are 16 samples, K is the input.
// Lane l holds B column l%16 at K-slots (l/16, s = 0..7); D rows 4(l/16)+r.
// A neuron block's D therefore already sits where the next layer's B needs it
// once the K index of slot (g, s) is taken to be
//   s < 4 : block 2c   neuron 4g + s        s >= 4 : block 2c+1 neuron 4g + s-4
// which the host bakes into the weight fragments (build_mlp_fragments).  The
// level-split encode delivers layer 1's B operand straight from the gathers.
__device__ __forceinline__ float4v mfma(half8 a, half8 b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// ReLU of eight FP32 accumulators as the next layer's FP16 B operand: round
// pairs to FP16 (v_cvt_pk_f16_f32, round to nearest even) and clamp at zero
// in FP16 (v_pk_max_f16); rounding is monotonic and keeps the sign, so this
// equals rounding the clamped values.
__device__ __forceinline__ half8 pack_relu(float4v lo, float4v hi) {
  typedef float float2v_ __attribute__((ext_vector_type(2)));
  const half2v z = {(_Float16)0.0f, (_Float16)0.0f};
  const half2v a = __builtin_elementwise_max(__builtin_convertvector((float2v_){lo[0], lo[1]}, half2v), z);
  const half2v b = __builtin_elementwise_max(__builtin_convertvector((float2v_){lo[2], lo[3]}, half2v), z);
  const half2v c = __builtin_elementwise_max(__builtin_convertvector((float2v_){hi[0], hi[1]}, half2v), z);
  const half2v d = __builtin_elementwise_max(__builtin_convertvector((float2v_){hi[2], hi[3]}, half2v), z);
  half8 r;
  r[0] = a[0]; r[1] = a[1]; r[2] = b[0]; r[3] = b[1];
  r[4] = c[0]; r[5] = c[1]; r[6] = d[0]; r[7] = d[1];
  return r;
}

// Mixed-path sigmoid: hardware exp and reciprocal (about 1 ulp each, far
// below the FP16 network's own rounding).
__device__ __forceinline__ float sigmoid_fast(float v) {
  return __builtin_amdgcn_rcpf(1.0f + __expf(-v));
}

// ------------------------------------------------- outputs to host memory
// A frame whose outputs go to pinned host memory is bound by the link for a
// quarter of its time (stereo 1080p RGB24 and depth: 29 MB, 0.52 ms at 56
// GB/s, against 1.4 ms of kernels).  Pixels of tiles without samples are final
// (zero) once the march is done, so they are stored during the encode, by a
// few extra workgroups of its launch; the rest follow the composite.  The
// split is by 128-byte line of each output array: a line is background if all
// of its pixels lie in tiles without samples.
//
// Everything goes out in 16-byte units that are aligned on the host's side (a
// PCIe write of less costs a packet of its own), whatever the destination's
// alignment: the source is read at any byte offset, and the bytes in front of
// the first unit and behind the last one follow one by one.  Stereo 1080p into
// arrays at odd addresses 2017 -> 1379 us, at multiples of 4 bytes 1874 -> 1379
// (before: single-byte and 4-byte stores, all after the composite); aligned
// arrays 1385 either way.
constexpr uint32_t kUnit = 16;

__device__ __forceinline__ uint32_t whole_units(const HostArray &h) { return (uint32_t)((h.bytes - h.head) / kUnit); }

// Whether the 16 bytes of unit `unit` of the array are background.
__device__ __forceinline__ bool unit_is_background(const HostArray &h, const ViewDesc &v,
                                                   const uint32_t *__restrict__ tile_n, uint32_t unit) {
  const uint32_t at = h.head + unit * kUnit;
  const uint32_t p0 = at / h.bpp, p1 = (at + kUnit - 1) / h.bpp;
  const uint32_t *tn = tile_n + (v.slot_base >> 6);
  uint32_t y = p0 / v.width, x = p0 - y * v.width;
  uint32_t n = 0;
  // the tiles of the first pixel and of every pixel that starts a tile or row
  for (uint32_t p = p0;;) {
    n |= tn[(y >> 3) * v.tiles_x + (x >> 3)];
    const uint32_t step = min(8u - (x & 7u), v.width - x);
    p += step;
    x += step;
    if (p > p1) break;
    if (x == v.width) {
      x = 0;
      ++y;
    }
  }
  return n == 0;
}

// The same for the 128-byte line of this lane's unit; lanes hold consecutive
// units from a multiple of 64 on.
__device__ __forceinline__ bool line_is_background(const HostArray &h, const ViewDesc &v,
                                                   const uint32_t *__restrict__ tile_n, uint32_t unit,
                                                   uint32_t n_units) {
  const uint64_t b = __ballot(unit < n_units && unit_is_background(h, v, tile_n, unit));
  return ((b >> (lane_id() & ~7)) & 0xffu) == 0xffu;
}

struct BackgroundArgs {
  const HostArray *arrays;
  const ViewDesc *views;
  const uint32_t *tile_n;
  uint32_t n_arrays, groups;  // groups: workgroups that store, 0 = none
};

// One store of 1 KB per wavefront in flight: with kBackgroundGroups x 4 waves
// that covers the link's bandwidth times its latency, and no more queues up
// in the memory pipeline that the encode's gathers share.
__device__ __forceinline__ void store_background(const BackgroundArgs &a, uint32_t grp) {
  const uint32_t wave = grp * 4 + (threadIdx.x >> 6), n_waves = a.groups * 4;
  for (uint32_t i = 0; i < a.n_arrays; ++i) {
    const HostArray h = a.arrays[i];
    const ViewDesc v = a.views[h.view];
    const uint32_t n_units = whole_units(h);
    for (uint32_t at = wave * 64; at < n_units; at += n_waves * 64) {
      const uint32_t unit = at + (uint32_t)lane_id();
      if (line_is_background(h, v, a.tile_n, unit, n_units))
        reinterpret_cast<uint4 *>(h.dst + h.head)[unit] = make_uint4(0u, 0u, 0u, 0u);
      __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
  }
}

// ------------------------------------------------- XCD-partitioned encode
// MI355X dispatches workgroup b to XCD b % 8, and each XCD has its own 4 MB
// L2.  Part p = b % 8 encodes only levels p and 15 - p for every sample, so
// an XCD's L2 holds one coarse level plus one (2 MB in FP16) hashed level and
// the corner gathers hit in L2 instead of streaming 64-byte lines from the
// Infinity Cache.  (In FP32 a hashed level alone is 4 MB.)  Features go to
// feat[p][sample] as {level p f0, f1, level 15-p f0, f1}.
//
// Parts 0, 1 and 2 take longer than the others where neighbouring rays lie
// several cells of the finest levels apart: level 15's four L2 requests per
// sample fill XCD 0's request rate, while XCD 7 is done in two thirds of the
// time.  So XCD 7 - p encodes the last share[p] of part p's samples (in 1 /
// 65536) once its own part is done: in turn, so that its L2 holds two levels
// at a time.  Stereo 1080p, times of the parts alone, us:
//   996 951 844 775 779 714 700 659, together 1040; with shares 950
// (1440x1600 at 75 degrees 1229 -> 1064, 2064x2208 2263 -> 1995).  A batch of
// random rays in FP32 is the other way round (see kScatteredShare).
constexpr int kHelpedParts = 3;
struct PartShares {
  uint32_t share[kHelpedParts];
  uint32_t reverse;  // parts 7, 6, 5 are helped by XCDs 0, 1, 2 instead (FP32 only)
};

// Samples of part P beyond its own XCD's share start here (a multiple of the
// workgroup size, so that a workgroup works on one part at a time).
__device__ __forceinline__ uint32_t part_end(uint32_t n, uint32_t share) {
  return (n - (uint32_t)((uint64_t)n * share >> 16)) & ~255u;
}

// Samples [from + i, to) of part P for i, i + step, ...; returns the first i
// past them.
template <class Tab, int P>
__device__ __forceinline__ uint32_t encode_part_loop(const typename PosIn<Tab>::type *__restrict__ pos,
                                                     uint32_t from, uint32_t to, uint32_t stride,
                                                     const Tab *table,
                                                     typename PartOut<Tab>::type *__restrict__ feat,
                                                     uint32_t i, uint32_t step, uint32_t *xch) {
  constexpr int LA = P, LB = 15 - P;
  const char *base_a = level_base<Tab, LA>(table), *base_b = level_base<Tab, LB>(table);
  typename PartOut<Tab>::type *dst = feat + (size_t)P * stride;
  const uint32_t count = to - from;
  for (; i < count; i += step) {
    const uint32_t s = from + i;
    float xc[3];
    PosIn<Tab>::get(pos[s], xc);
    float2 fa, fb;
    encode_two<Tab, LA, LB>(base_a, base_b, xc, fa, fb, xch);
    dst[s] = PartOut<Tab>::pack(fa, fb);
  }
  return i - count;
}

// Each part is its own instantiation, so level resolutions, offsets and the
// dense/hashed choice are compile-time constants.
template <class Tab>
__global__ __launch_bounds__(256) void encode_parts(const typename PosIn<Tab>::type *__restrict__ pos,
                                                    const uint32_t *__restrict__ n_ptr,
                                                    uint32_t stride, const Tab *__restrict__ table,
                                                    typename PartOut<Tab>::type *__restrict__ feat,
                                                    uint32_t blocks_per_part, PartShares shares,
                                                    BackgroundArgs bg, uint64_t *stamp) {
  stamp_start(stamp);
  __shared__ uint32_t xch_all[4][256];  // per-wavefront gather exchange (FP16 hashed levels)
  // the first workgroups (a multiple of kParts of them) store background pixels
  // (nothing of a pass that overflowed: the host may not be able to run it again)
  if (blockIdx.x < bg.groups) {
    if (*n_ptr <= stride) store_background(bg, blockIdx.x);
    return;
  }
  uint32_t *xch = xch_all[threadIdx.x >> 6];
  const uint32_t n = min(*n_ptr, stride);
  uint32_t i = (blockIdx.x - bg.groups) / kParts * blockDim.x + threadIdx.x;
  const uint32_t step = blocks_per_part * blockDim.x;
#define NES_PART(P, FROM, TO) i = encode_part_loop<Tab, P>(pos, FROM, TO, stride, table, feat, i, step, xch)
  // part P and its helper's turn at part 7 - P, or the other way round
  const bool rev = sizeof(Tab) == 4 && shares.reverse;
#define NES_PART_PAIR(P)                                                \
  case P:                                                               \
    NES_PART(P, 0u, rev ? n : part_end(n, shares.share[P]));            \
    if (rev) NES_PART(7 - P, part_end(n, shares.share[P]), n);          \
    break;                                                              \
  case 7 - P:                                                           \
    NES_PART(7 - P, 0u, rev ? part_end(n, shares.share[P]) : n);        \
    if (!rev) NES_PART(P, part_end(n, shares.share[P]), n);             \
    break;
  switch (blockIdx.x % kParts) {
    NES_PART_PAIR(0)
    NES_PART_PAIR(1)
    NES_PART_PAIR(2)
    case 3: NES_PART(3, 0u, n); break;
    default: NES_PART(4, 0u, n); break;
  }
#undef NES_PART_PAIR
#undef NES_PART
}

// FP16 MFMA MLPs: lane (g, j) of a 16-sample tile loads parts 2g and 2g+1 of
// sample j -- the layer-1 B operand with K-slot s of group g holding feature
// part_feature(2g + s/4, s%4) (baked into the W1 fragments).  Each wave keeps
// the 20 weight fragments in registers for all its tiles: re-reading them
// from LDS per tile moves 20 KB of LDS data per 16 samples, and the frame is
// power-limited, so that energy costs clock in every kernel.
__global__ __launch_bounds__(256) void mlp_mixed(const uint32_t *__restrict__ samples,
                                                 const uint2 *__restrict__ feat,
                                                 const uint32_t *__restrict__ n_ptr,
                                                 uint32_t stride,
                                                 const uint2 *__restrict__ ray_sh,
                                                 const half8 *__restrict__ wfrag,
                                                 uint2 *__restrict__ out, uint64_t *stamp) {
  stamp_start(stamp);
  const uint32_t n = min(*n_ptr, stride);
  if (blockIdx.x * kEvalWaves * 16 >= n) return;  // no tile for any wave of this workgroup
  __shared__ half8 wl[20 * 64];
  for (int i = (int)threadIdx.x; i < 20 * 64; i += (int)blockDim.x) wl[i] = wfrag[i];
  __syncthreads();
  const int lane = lane_id(), wave = (int)(threadIdx.x >> 6);
  const int j = lane & 15, g = lane >> 4;
  half8 wf[20];
#pragma unroll
  for (int i = 0; i < 20; ++i) wf[i] = wl[64 * i + lane];
  const float4v zero = {0.0f, 0.0f, 0.0f, 0.0f};
  const uint32_t n_tiles = (n + 15) / 16;
  const uint32_t tile_step = gridDim.x * kEvalWaves;
  uint32_t tile = blockIdx.x * kEvalWaves + wave;
  if (tile >= n_tiles) return;
  // Software pipeline: the sample record and features of the next tile are
  // loaded while this tile's MFMAs run, its SH (which needs the record) at
  // the end of the iteration.  The loads are unconditional (indices clamped
  // to the last sample) so that each wait covers only what it needs.
  uint32_t sc = min(tile * 16 + (uint32_t)j, n - 1);
  uint2 fa = feat[(size_t)(2 * g) * stride + sc];
  uint2 fb = feat[(size_t)(2 * g + 1) * stride + sc];
  uint2 shw = ray_sh[(size_t)(samples[sc] >> 7) * 4 + g];
  while (true) {
    const uint32_t s = tile * 16 + (uint32_t)j;
    const uint32_t next = tile + tile_step;
    const bool more = next < n_tiles;
    const uint32_t nsc = min(next * 16 + (uint32_t)j, n - 1);
    const uint32_t nrec = samples[nsc];
    const uint2 nfa = feat[(size_t)(2 * g) * stride + nsc];
    const uint2 nfb = feat[(size_t)(2 * g + 1) * stride + nsc];
    __builtin_amdgcn_sched_barrier(0);  // keep the prefetch ahead of the MFMAs
    const uint32_t words[4] = {fa.x, fa.y, fb.x, fb.y};
    half8 b1;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const half2v h = __builtin_bit_cast(half2v, words[k]);
      b1[2 * k] = h.x;
      b1[2 * k + 1] = h.y;
    }
    float4v d1[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) d1[m] = mfma(wf[m], b1, zero);
    float4v d2 = mfma(wf[4], pack_relu(d1[0], d1[1]), zero);
    d2 = mfma(wf[5], pack_relu(d1[2], d1[3]), d2);
    const half2v sh01 = __builtin_bit_cast(half2v, shw.x), sh23 = __builtin_bit_cast(half2v, shw.y);
    half8 b3;
    b3[0] = (_Float16)d2[0]; b3[1] = (_Float16)d2[1];
    b3[2] = (_Float16)d2[2]; b3[3] = (_Float16)d2[3];
    b3[4] = sh01[0]; b3[5] = sh01[1]; b3[6] = sh23[0]; b3[7] = sh23[1];
    float4v d3[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) d3[m] = mfma(wf[6 + m], b3, zero);
    const half8 b4a = pack_relu(d3[0], d3[1]), b4b = pack_relu(d3[2], d3[3]);
    float4v d4[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      d4[m] = mfma(wf[10 + 2 * m], b4a, zero);
      d4[m] = mfma(wf[11 + 2 * m], b4b, d4[m]);
    }
    float4v d5 = mfma(wf[18], pack_relu(d4[0], d4[1]), zero);
    d5 = mfma(wf[19], pack_relu(d4[2], d4[3]), d5);
    if (g == 0 && s < n) {
      // (log sigma, r, g, b) as FP16; the FP32 composite takes the exp
      half2v lo, hi;
      lo.x = (_Float16)d2[0];
      lo.y = (_Float16)sigmoid_fast(d5[0]);
      hi.x = (_Float16)sigmoid_fast(d5[1]);
      hi.y = (_Float16)sigmoid_fast(d5[2]);
      out[s] = make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
    }
    if (!more) break;
    __builtin_amdgcn_sched_barrier(0);
    shw = ray_sh[(size_t)(nrec >> 7) * 4 + g];
    __builtin_amdgcn_sched_barrier(0);  // and the SH load at the end of the iteration
    tile = next;
    fa = nfa;
    fb = nfb;
  }
}

// ------------------------------------------------------------- composite
struct OutPtrs {
  uint8_t *rgb24;
  float *depth;
  float *rgbf;
  uint16_t *nsamp;
};

// Per-sample MLP output as the composite reads it: FP32 (sigma, r, g, b), or
// the mixed path's FP16 (log sigma, r, g, b).
__device__ __forceinline__ float4 sample_value(const float4 &v) { return v; }
__device__ __forceinline__ float4 sample_value(const uint2 &v) {
  const half2v lo = __builtin_bit_cast(half2v, v.x), hi = __builtin_bit_cast(half2v, v.y);
  return make_float4(__expf((float)lo.x), (float)lo.y, (float)hi.x, (float)hi.y);
}

// One lane per ray slot, walking the wavefront's rank-major sample range
// eight ranks at a time (positions from ballots, loads issued together, then
// composited in order).
struct CompositeArgs {
  const ViewDesc *views;  // null: output index = ray slot (training)
  uint32_t n_views, n_slots;
  const RayData *rays;
  RayAcc *acc;
  uint32_t *counts;
  const uint32_t *offsets, *samples;
  const float *t_start;
  const uint32_t *n_ptr;
  uint32_t capacity;
  int first;  // no state from an earlier pass
  int last;   // write the outputs
  int keep;   // store the state after the last pass too
  OutPtrs o;
  uint32_t *stats;
  uint64_t *stamp;
};

template <class SampleOut>
__global__ __launch_bounds__(256) void composite(CompositeArgs c, const SampleOut *__restrict__ sout) {
  stamp_start(c.stamp);
  if (*c.n_ptr > c.capacity) return;  // overflowed pass: the host re-renders
  const uint32_t slot = blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = lane_id();
  const bool valid = slot < c.n_slots;
  RayAcc a{};
  a.T = 1.0f;
  const uint32_t flags = valid ? c.counts[slot] : 0u;
  const uint32_t cnt = flags & kCountMask;
  if (!c.first && (flags & kRayState)) {
    a = c.acc[slot];  // an earlier pass composited samples of this ray
  }
  const bool live = cnt != 0 && !a.done;
  const uint32_t n_before = a.n_samples;
  const uint32_t mx = wave_max(cnt);
  if (mx) {
    const uint32_t base = c.offsets[__builtin_amdgcn_readfirstlane(slot >> 6)];
    const float ts = live ? c.t_start[slot] : 0.0f;
    uint32_t at0 = base;
    for (uint32_t i0 = 0; i0 < mx; i0 += 8) {  // wavefront-uniform
      if (__ballot(live && !a.done && i0 < cnt) == 0) break;
      SampleOut sb[8];
      uint32_t kb[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const uint32_t i = i0 + (uint32_t)u;
        const uint64_t has = __ballot(cnt > i);
        const uint32_t at =
            at0 + __builtin_amdgcn_mbcnt_hi((uint32_t)(has >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)has, 0u));
        at0 += (uint32_t)__popcll(has);
        sb[u] = SampleOut{};
        kb[u] = 0u;
        if (live && cnt > i && !a.done) {
          sb[u] = sout[at];
          kb[u] = c.samples[at];
        }
      }
      if (live) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          if (i0 + (uint32_t)u >= cnt || a.done) break;
          const float4 sm = sample_value(sb[u]);
          const float t = step_t((int)(kb[u] & 127u), ts);
          const float sd = sm.x * kDelta;
          const float alpha = -expm1f(-sd);
          const float w = a.T * alpha;
          a.r = fmaf(w, sm.y, a.r);
          a.g = fmaf(w, sm.z, a.g);
          a.b = fmaf(w, sm.w, a.b);
          a.depth = fmaf(w, t, a.depth);
          a.T *= expf(-sd);
          a.n_samples++;
          if (a.T < kTStop) a.done = 1;
        }
      }
    }
  }
  if (c.stats) {
    // Termination counters, touched only by wavefronts with a ray that
    // reached T < 1e-4 in this pass (none in a scene that never does), on
    // one of kTotTermSlots lines so that such wavefronts rarely share one.
    const bool term = live && a.done;
    const uint64_t tb = __ballot(term);
    if (tb) {
      const uint32_t here = a.n_samples - n_before;  // composited in this pass
      bool saved = false;
      if (term && !c.last) saved = (flags >> 16) < c.rays[slot].n_steps;
      const uint32_t ts_sum = wave_sum(term ? a.n_samples : 0u);
      const uint32_t waste = wave_sum(term ? cnt - here : 0u);
      const uint32_t ns = (uint32_t)__popcll(__ballot(saved));
      if (lane == 0) {
        uint32_t *st = c.stats + kTotTermBase + kTotTermStride * ((slot >> 6) % kTotTermSlots);
        atomicAdd(st + 0, (uint32_t)__popcll(tb));
        atomicAdd(st + 1, ts_sum);
        if (waste) atomicAdd(st + 2, waste);
        if (ns) atomicAdd(st + 3, ns);
      }
    }
    // every pass adds its sample total once
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(c.stats + kTotEvaluated, *c.n_ptr);
  }
  if (!valid) return;
  // the state carries into the next pass; after the last pass only a caller
  // that reads it again (keep: the training backward) stores it
  if (live && (!c.last || c.keep)) c.acc[slot] = a;
  if (!c.last) {
    if (live) c.counts[slot] = flags | kRayState | (a.done ? kRayDone : 0u);
    return;
  }
  uint32_t p = slot;
  if (c.views) {
    const uint32_t wslot = __builtin_amdgcn_readfirstlane(slot);
    const ViewDesc &v = c.views[view_of(c.views, c.n_views, wslot)];
    const uint32_t tile = (wslot - v.slot_base) >> 6;
    const uint32_t px = (tile % v.tiles_x) * 8 + (lane & 7), py = (tile / v.tiles_x) * 8 + (lane >> 3);
    if (px >= v.width || py >= v.height) return;
    p = v.px_base + py * v.width + px;
  }
  const float col[3] = {a.r, a.g, a.b};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float q = floorf(fmaf(col[k], 255.0f, 0.5f));
    c.o.rgb24[3 * (size_t)p + k] = (uint8_t)fminf(fmaxf(q, 0.0f), 255.0f);
    c.o.rgbf[3 * (size_t)p + k] = col[k];
  }
  c.o.depth[p] = a.depth;
  c.o.nsamp[p] = (uint16_t)a.n_samples;
}

// The ray's next sample, held by lane q of its four lanes, added to the
// front-to-back sums that all four keep.
template <int q>
__device__ __forceinline__ void add_sample(RayAcc &a, bool more, const float4 &sm, float t, float alpha, float e) {
  const float aq = quad_value<q>(alpha), eq = quad_value<q>(e);
  const float y = quad_value<q>(sm.y), z = quad_value<q>(sm.z), x = quad_value<q>(sm.w), tq = quad_value<q>(t);
  if (more && !a.done) {
    const float w = a.T * aq;
    a.r = fmaf(w, y, a.r);
    a.g = fmaf(w, z, a.g);
    a.b = fmaf(w, x, a.b);
    a.depth = fmaf(w, tq, a.depth);
    a.T *= eq;
    a.n_samples++;
    if (a.T < kTStop) a.done = 1;
  }
}

// The same with one workgroup per tile and four lanes per ray, as
// march_emit_split: of 32 ranks in turn every lane loads eight (while the 32
// before are summed) and computes their opacities, then all four lanes take the
// 32 in order.  64x48: 17.2 -> 12.2 us, 4096 rays of a batch: 26.6 -> 11.6 us;
// without the loads ahead 15.0 and 14.2.
template <class SampleOut>
__global__ __launch_bounds__(256) void composite_split(CompositeArgs c, const SampleOut *__restrict__ sout) {
  stamp_start(c.stamp);
  __shared__ uint64_t rank_rays[kMaxSteps];
  __shared__ uint32_t rank_at[kMaxSteps];
  const int lane = lane_id();
  const uint32_t ray = threadIdx.x >> 2, seg = threadIdx.x & 3u;
  const uint32_t slot0 = blockIdx.x * 64, slot = slot0 + ray;
  const bool valid = slot < c.n_slots;
  const uint32_t tile_flags = slot0 + (uint32_t)lane < c.n_slots ? c.counts[slot0 + (uint32_t)lane] : 0u;
  // (neither is written, nor used, where there are no samples)
  const uint32_t base = c.offsets[blockIdx.x];
  const float ts = valid ? c.t_start[slot] : 0.0f;
  if (*c.n_ptr > c.capacity) return;  // overflowed pass: the host re-renders
  const uint32_t flags = (uint32_t)__shfl((int)tile_flags, (int)ray);
  const uint32_t cnt = flags & kCountMask;
  RayAcc a{};
  a.T = 1.0f;
  if (!c.first && (flags & kRayState)) a = c.acc[slot];
  const bool live = cnt != 0 && !a.done;
  const uint32_t n_before = a.n_samples;
  const uint32_t tile_mx = wave_max(tile_flags & kCountMask);
  if (tile_mx) {  // the same in every wavefront
    index_ranks(tile_flags & kCountMask, tile_mx, rank_rays, rank_at);
    const uint64_t below = lanes_below((int)ray);
    const uint32_t mx = wave_max(cnt);
    SampleOut sb[8];
    uint32_t kb[8];
    const auto load = [&](uint32_t i0) {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const uint32_t i = i0 + 4u * (uint32_t)u + seg;
        sb[u] = SampleOut{};
        kb[u] = 0u;
        if (live && i < cnt) {
          const uint32_t at = base + rank_at[i] + (uint32_t)__popcll(rank_rays[i] & below);
          sb[u] = sout[at];
          kb[u] = c.samples[at];
        }
      }
    };
    load(0);
    for (uint32_t i0 = 0; i0 < mx; i0 += 32) {  // wavefront-uniform
      if (__ballot(live && !a.done && i0 < cnt) == 0) break;
      SampleOut sv[8];
      uint32_t kv[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        sv[u] = sb[u];
        kv[u] = kb[u];
      }
      load(i0 + 32);  // in flight while these are summed
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const uint32_t i = i0 + 4u * (uint32_t)u;
        if (i >= mx) break;  // wavefront-uniform
        const float4 sm = sample_value(sv[u]);
        const float t = step_t((int)(kv[u] & 127u), ts);
        const float sd = sm.x * kDelta;
        const float alpha = -expm1f(-sd);
        const float e = expf(-sd);
        add_sample<0>(a, live && i < cnt, sm, t, alpha, e);
        add_sample<1>(a, live && i + 1 < cnt, sm, t, alpha, e);
        add_sample<2>(a, live && i + 2 < cnt, sm, t, alpha, e);
        add_sample<3>(a, live && i + 3 < cnt, sm, t, alpha, e);
      }
    }
  }
  if (c.stats) {  // as in composite
    const bool term = live && a.done && seg == 0;
    const uint64_t tb = __ballot(term);
    if (tb) {
      const uint32_t here = a.n_samples - n_before;
      bool saved = false;
      if (term && !c.last) saved = (flags >> 16) < c.rays[slot].n_steps;
      const uint32_t ts_sum = wave_sum(term ? a.n_samples : 0u);
      const uint32_t waste = wave_sum(term ? cnt - here : 0u);
      const uint32_t ns = (uint32_t)__popcll(__ballot(saved));
      if (lane == 0) {
        uint32_t *st = c.stats + kTotTermBase + kTotTermStride * (blockIdx.x % kTotTermSlots);
        atomicAdd(st + 0, (uint32_t)__popcll(tb));
        atomicAdd(st + 1, ts_sum);
        if (waste) atomicAdd(st + 2, waste);
        if (ns) atomicAdd(st + 3, ns);
      }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(c.stats + kTotEvaluated, *c.n_ptr);
  }
  if (!valid) return;
  if (seg == 0 && live && (!c.last || c.keep)) c.acc[slot] = a;
  if (!c.last) {
    if (seg == 0 && live) c.counts[slot] = flags | kRayState | (a.done ? kRayDone : 0u);
    return;
  }
  uint32_t p = slot;
  if (c.views) {
    const ViewDesc &v = c.views[view_of(c.views, c.n_views, slot0)];
    const uint32_t tile = (slot0 - v.slot_base) >> 6;
    const uint32_t px = (tile % v.tiles_x) * 8 + (ray & 7), py = (tile / v.tiles_x) * 8 + (ray >> 3);
    if (px >= v.width || py >= v.height) return;
    p = v.px_base + py * v.width + px;
  }
  if (seg == 3) {
    c.o.depth[p] = a.depth;
    c.o.nsamp[p] = (uint16_t)a.n_samples;
  } else {  // one colour channel per lane
    const float col = seg == 0 ? a.r : seg == 1 ? a.g : a.b;
    const float q = floorf(fmaf(col, 255.0f, 0.5f));
    c.o.rgb24[3 * (size_t)p + seg] = (uint8_t)fminf(fmaxf(q, 0.0f), 255.0f);
    c.o.rgbf[3 * (size_t)p + seg] = col;
  }
}

// Ray slots up to which the composite runs four lanes per ray, by the same
// reasoning as the march but with more work per sample to do four times
// (composite -> composite_split, us): frames of 77k slots 18.4 -> 14.4, 173k
// 19.2 -> 17.9, 307k 20.0 -> 22.3, 614k 23.9 -> 31.9; batches of 16k rays
// 24.6 -> 11.5, 65k 17.0 -> 17.9.
constexpr uint32_t kSplitComposite = 1u << 17;

template <class SampleOut>
static int composite_pass(const CompositeArgs &c, const SampleOut *sout, hipStream_t stream) {
  if (c.n_slots <= (c.views ? kSplitComposite : kSplitBatchRays))
    composite_split<SampleOut><<<(unsigned)((c.n_slots + 63) / 64), 256, 0, stream>>>(c, sout);
  else
    composite<SampleOut><<<(unsigned)((c.n_slots + 255) / 256), 256, 0, stream>>>(c, sout);
  NES_HIP_TRY(hipGetLastError());
  return NES_OK;
}

__global__ void zero_u32(uint32_t *p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// The start of a frame: every counter cleared and up to kArgViews view
// descriptors stored from the kernel's arguments (a copy from host memory
// costs 14 us before the first kernel of a small frame).
constexpr uint32_t kArgViews = 8;
struct ArgViews {
  ViewDesc v[kArgViews];
};
struct ArgArrays {
  HostArray a[kHostArrays];
};
constexpr int kViewWords = (int)(sizeof(ViewDesc) / sizeof(uint32_t));
constexpr int kArrayWords = (int)(sizeof(HostArray) / sizeof(uint32_t));
static_assert(sizeof(ViewDesc) % sizeof(uint32_t) == 0 && sizeof(HostArray) % sizeof(uint32_t) == 0, "whole words");
constexpr int kFrameThreads = 1024;

__global__ __launch_bounds__(kFrameThreads) void frame_begin(uint32_t *total, ArgViews views, uint32_t n_views,
                                                             ViewDesc *dst, ArgArrays arrays,
                                                             uint32_t n_arrays, HostArray *array_dst) {
  const int t = (int)threadIdx.x;
  for (int i = t; i < kTotWords; i += kFrameThreads)
    if (i != kTotStamps + 2 * kStampBegin && i != kTotStamps + 2 * kStampBegin + 1) total[i] = 0u;
  for (int i = t; i < (int)n_views * kViewWords; i += kFrameThreads)
    reinterpret_cast<uint32_t *>(dst)[i] = reinterpret_cast<const uint32_t *>(&views)[i];
  for (int i = t; i < (int)n_arrays * kArrayWords; i += kFrameThreads)
    reinterpret_cast<uint32_t *>(array_dst)[i] = reinterpret_cast<const uint32_t *>(&arrays)[i];
  if (t == 0) reinterpret_cast<uint64_t *>(total + kTotStamps)[kStampBegin] = wall_clock64();
}

// Byte `at` of the array.
__device__ __forceinline__ uint8_t output_byte(const HostArray &h, uint32_t at) {
  // (the scale may have any value: 0 for an infinite far distance)
  return h.bpp == 1 ? depth_gray8(reinterpret_cast<const float *>(h.src)[at], h.gray_scale) : h.src[at];
}

typedef uint32_t Unit __attribute__((ext_vector_type(4), aligned(1)));

__device__ __forceinline__ void store_unit(const HostArray &h, uint32_t unit) {
  const uint32_t at = h.head + unit * kUnit;
  uint4 v;
  if (h.bpp == 1) {
    const float *d = reinterpret_cast<const float *>(h.src) + at;
    uint8_t g[kUnit];
#pragma unroll
    for (uint32_t i = 0; i < kUnit; ++i) g[i] = depth_gray8(d[i], h.gray_scale);
    __builtin_memcpy(&v, g, kUnit);
  } else {
    const Unit u = *reinterpret_cast<const Unit *>(h.src + at);
    v = make_uint4(u.x, u.y, u.z, u.w);
  }
  *reinterpret_cast<uint4 *>(h.dst + at) = v;
}

// An output array into host memory (one per blockIdx.y); with `bg`, only what
// store_background left.
__device__ __forceinline__ void store_outputs(const HostArray &array, const BackgroundArgs *bg) {
  const HostArray h = array;
  ViewDesc v;
  if (bg) v = bg->views[h.view];
  const uint32_t n_units = whole_units(h);
  for (uint32_t at = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 64; at < n_units; at += gridDim.x * 256) {
    const uint32_t unit = at + (uint32_t)lane_id();
    const bool done = bg && line_is_background(h, v, bg->tile_n, unit, n_units);
    if (unit < n_units && !done) store_unit(h, unit);
  }
  const uint32_t behind = h.head + n_units * kUnit;  // the bytes beside the units
  if (blockIdx.x == 0) {
    if (threadIdx.x < h.head) h.dst[threadIdx.x] = output_byte(h, threadIdx.x);
    if (behind + threadIdx.x < h.bytes) h.dst[behind + threadIdx.x] = output_byte(h, behind + threadIdx.x);
  }
}

// The end of a frame: the counters and stamps and, if its samples fitted, the
// output arrays into pinned host memory.
__global__ __launch_bounds__(256) void frame_end(const uint32_t *total, uint32_t *host, BackgroundArgs a,
                                                 uint32_t capacity) {
  constexpr int kEnd = kTotStamps + 2 * kStampEnd;
  if (blockIdx.x == 0 && blockIdx.y == 0) {
    for (int i = (int)threadIdx.x; i < kTotWords; i += (int)blockDim.x)
      if (i != kEnd && i != kEnd + 1) host[i] = total[i];
    if (threadIdx.x == 0) reinterpret_cast<uint64_t *>(host + kTotStamps)[kStampEnd] = wall_clock64();
  }
  if (max(total[kTotCursor], total[kTotCursorLater]) > capacity) return;  // the host re-renders
  if (blockIdx.y < a.n_arrays) store_outputs(a.arrays[blockIdx.y], a.groups ? &a : nullptr);
}

// The same for arrays of a finished frame (nes_render_fetch).
__global__ __launch_bounds__(256) void store_arrays(ArgArrays arrays) {
  store_outputs(arrays.a[blockIdx.y], nullptr);
}

// FP32 expected depth -> the GRAY8 depth plane of the response.
__global__ void depth_gray8_kernel(const float *__restrict__ depth, size_t n, float scale,
                                   uint8_t *__restrict__ gray) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i < n) gray[i] = depth_gray8(depth[i], scale);
}

// ----------------------------------------------------------------- host
void build_mlp_fragments(const float *w, _Float16 *frag) {
  // slot (g, s) of K-chunk c -> input neuron of a 64-wide hidden layer
  auto hid = [](int c, int g, int s) { return s < 4 ? 32 * c + 4 * g + s : 32 * c + 16 + 4 * g + (s - 4); };
  auto put = [&](int mf, int lane, int s, float v) { frag[((size_t)mf * 64 + lane) * 8 + s] = (_Float16)v; };
  for (int lane = 0; lane < 64; ++lane) {
    const int i = lane & 15, g = lane >> 4;
    for (int s = 0; s < 8; ++s) {
      // layer 1: 32 features -> 64; K-slot (g, s) holds feature
      // part_feature(2g + s/4, s%4) as delivered by encode_parts
      for (int m = 0; m < 4; ++m)
        put(m, lane, s, w[kW1 + (16 * m + i) * 32 + part_feature(2 * g + s / 4, s % 4)]);
      // layer 2: 64 -> 16, two K-chunks
      for (int c = 0; c < 2; ++c) put(4 + c, lane, s, w[kW2 + i * 64 + hid(c, g, s)]);
      // layer 3: [density outputs 4g..4g+3 | SH 4g..4g+3] -> 64; density
      // output 0 is log-sigma and gets no weight; outputs 1..15 are inputs
      // 16..30 of W3, SH are inputs 0..15
      for (int m = 0; m < 4; ++m) {
        float v;
        if (s < 4) {
          const int o2 = 4 * g + s;
          v = o2 == 0 ? 0.0f : w[kW3 + (16 * m + i) * 31 + 16 + (o2 - 1)];
        } else {
          v = w[kW3 + (16 * m + i) * 31 + 4 * g + (s - 4)];
        }
        put(6 + m, lane, s, v);
      }
      // layer 4: 64 -> 64
      for (int m = 0; m < 4; ++m)
        for (int c = 0; c < 2; ++c) put(10 + 2 * m + c, lane, s, w[kW4 + (16 * m + i) * 64 + hid(c, g, s)]);
      // layer 5: 64 -> 3 (rows 3..15 zero)
      for (int c = 0; c < 2; ++c) put(18 + c, lane, s, i < 3 ? w[kW5 + i * 64 + hid(c, g, s)] : 0.0f);
    }
  }
}

int scene_upload(SceneDev &s, const nes_scene_desc *desc) {
  if (!desc || !desc->table || !desc->weights || !desc->occupancy) return NES_EINVAL;
  const size_t nt = (size_t)kTableEntries * 2, ndev = (size_t)kDevTableEntries * 2;
  if (!s.table_f32) {
    NES_HIP_TRY(hipMalloc(&s.table_f32, ndev * sizeof(float)));
    NES_HIP_TRY(hipMalloc(&s.table_f16, ndev * sizeof(_Float16)));
    NES_HIP_TRY(hipMalloc(&s.weights_f32, kWeights * sizeof(float)));
    NES_HIP_TRY(hipMalloc(&s.wfrag, 20 * 64 * 8 * sizeof(_Float16)));
    NES_HIP_TRY(hipMalloc(&s.occ, NES_OCC_WORDS * sizeof(uint32_t)));
    // the padding between levels (device layout) is never read; keep it zero
    NES_HIP_TRY(hipMemset(s.table_f32, 0, ndev * sizeof(float)));
    NES_HIP_TRY(hipMemset(s.table_f16, 0, ndev * sizeof(_Float16)));
  }
  std::vector<_Float16> t16(nt);
  for (size_t i = 0; i < nt; ++i) t16[i] = (_Float16)desc->table[i];
  std::vector<_Float16> frag(20 * 64 * 8);
  build_mlp_fragments(desc->weights, frag.data());
  NES_TRY(table_copy(s.table_f32, true, desc->table, false, sizeof(float), hipMemcpyHostToDevice, nullptr));
  NES_TRY(table_copy(s.table_f16, true, t16.data(), false, sizeof(_Float16), hipMemcpyHostToDevice, nullptr));
  NES_HIP_TRY(hipMemcpy(s.weights_f32, desc->weights, kWeights * sizeof(float), hipMemcpyHostToDevice));
  NES_HIP_TRY(hipMemcpy(s.wfrag, frag.data(), frag.size() * sizeof(_Float16), hipMemcpyHostToDevice));
  NES_HIP_TRY(hipMemcpy(s.occ, desc->occupancy, NES_OCC_WORDS * sizeof(uint32_t), hipMemcpyHostToDevice));
  return NES_OK;
}

void scene_free(SceneDev &s) {
  hipFree(s.table_f32);
  hipFree(s.table_f16);
  hipFree(s.weights_f32);
  hipFree(s.wfrag);
  hipFree(s.occ);
  s = SceneDev();
}

void render_work_free(RenderWork &w) {
  for (DevBuf *b : {&w.views, &w.rays, &w.acc, &w.counts, &w.offsets, &w.ray_sh, &w.t_start, &w.gray, &w.tile_n, &w.host_arrays, &w.samples,
                    &w.sample_out, &w.sample_pos, &w.feat, &w.out, &w.total})
    b->release();
  if (w.total_host) hipHostFree(w.total_host);
  w.total_host = nullptr;
  if (w.ev_views) {
    hipEventSynchronize(w.ev_views);
    hipEventDestroy(w.ev_views);
    w.ev_views = nullptr;
  }
  if (w.views_pinned) hipHostFree(w.views_pinned);
  w.views_pinned = nullptr;
  w.views_pinned_cap = 0;
}

static size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

OutLayout out_layout(size_t px) {
  OutLayout l;
  l.rgb24 = 0;
  l.depth = align_up(3 * px, 256);
  l.rgbf = align_up(l.depth + 4 * px, 256);
  l.nsamp = align_up(l.rgbf + 12 * px, 256);
  l.total = align_up(l.nsamp + 2 * px, 256);
  return l;
}

static OutPtrs out_ptrs(RenderWork &w) {
  const OutLayout L = out_layout(w.out_px);
  OutPtrs op;
  op.rgb24 = w.out.as<uint8_t>() + L.rgb24;
  op.depth = reinterpret_cast<float *>(w.out.as<uint8_t>() + L.depth);
  op.rgbf = reinterpret_cast<float *>(w.out.as<uint8_t>() + L.rgbf);
  op.nsamp = reinterpret_cast<uint16_t *>(w.out.as<uint8_t>() + L.nsamp);
  return op;
}

int render_setup(RenderWork &w, const nes_camera *views, int n_views, hipStream_t stream) {
  // Until this render completes, the work area describes no views: a fetch
  // after a failed setup or pass is refused instead of reading stale layouts.
  w.n_views = 0;
  w.out_px = 0;
  w.n_host_out = 0;
  w.store_background = false;
  if (!views || n_views < 1) return NES_EINVAL;
  w.host_views.resize((size_t)n_views);
  uint64_t slots = 0, px = 0, pixels = 0;
  for (int i = 0; i < n_views; ++i) {
    const nes_camera &c = views[i];
    if (c.width < 1 || c.height < 1 || c.width > 16384 || c.height > 16384 ||
        !(c.fov_y_deg > 0.0f && c.fov_y_deg < 180.0f)) {
      set_last_error("bad view size or field of view");
      return NES_EINVAL;
    }
    ViewDesc &v = w.host_views[(size_t)i];
    std::memcpy(v.c2w, c.c2w, sizeof(v.c2w));
    v.focal = (float)(0.5 * (double)c.height /
                      std::tan(0.5 * (double)c.fov_y_deg * 3.14159265358979323846 / 180.0));
    v.width = c.width;
    v.height = c.height;
    v.tiles_x = (c.width + 7) / 8;
    const uint32_t tiles_y = (c.height + 7) / 8;
    v.slot_base = (uint32_t)slots;
    v.slot_count = v.tiles_x * tiles_y * 64;
    v.px_base = (uint32_t)px;
    v.inv_focal = 1.0f / v.focal;
    // half a tile from its centre along the camera's right and down axes
    const double right = std::sqrt((double)c.c2w[0] * c.c2w[0] + (double)c.c2w[4] * c.c2w[4] + (double)c.c2w[8] * c.c2w[8]);
    const double down = std::sqrt((double)c.c2w[1] * c.c2w[1] + (double)c.c2w[5] * c.c2w[5] + (double)c.c2w[9] * c.c2w[9]);
    v.tile_reach = (float)(1.01 * 3.5 * (right + down) / (double)v.focal);
    slots += v.slot_count;
    px = align_up(px + (uint64_t)c.width * c.height, kViewAlign);
    pixels += (uint64_t)c.width * c.height;
    if (slots > kMaxSlots) {
      set_last_error("render batch exceeds 2^25 ray slots");
      return NES_ERANGE;
    }
  }
  w.n_views = (uint32_t)n_views;
  w.n_slots = (uint32_t)slots;
  w.out_px = px;
  w.pixels = pixels;
  NES_TRY(w.views.reserve(sizeof(ViewDesc) * n_views));
  NES_TRY(w.rays.reserve(sizeof(RayData) * slots));
  NES_TRY(w.acc.reserve(sizeof(RayAcc) * slots));
  NES_TRY(w.counts.reserve(sizeof(uint32_t) * slots));
  NES_TRY(w.offsets.reserve(sizeof(uint32_t) * wavefronts(slots)));
  NES_TRY(w.ray_sh.reserve(32 * slots));
  NES_TRY(w.t_start.reserve(sizeof(float) * slots));
  NES_TRY(w.tile_n.reserve(sizeof(uint32_t) * wavefronts(slots)));
  NES_TRY(w.host_arrays.reserve(sizeof(HostArray) * kHostArrays));
  NES_TRY(w.out.reserve(out_layout(px).total));
  NES_TRY(w.total.reserve(kTotBytes));
  if (!w.total_host) NES_HIP_TRY(hipHostMalloc((void **)&w.total_host, kTotBytes));
  if ((uint32_t)n_views <= kArgViews) return NES_OK;  // uploaded by frame_begin
  if (!w.ev_views) NES_HIP_TRY(hipEventCreateWithFlags(&w.ev_views, hipEventDisableTiming));
  NES_HIP_TRY(hipEventSynchronize(w.ev_views));  // the previous upload has read the staging
  if ((uint32_t)n_views > w.views_pinned_cap) {
    if (w.views_pinned) NES_HIP_TRY(hipHostFree(w.views_pinned));
    w.views_pinned = nullptr;
    w.views_pinned_cap = 0;
    const uint32_t cap = std::max<uint32_t>((uint32_t)n_views, kPinnedViews);
    NES_HIP_TRY(hipHostMalloc((void **)&w.views_pinned, sizeof(ViewDesc) * cap));
    w.views_pinned_cap = cap;
  }
  std::memcpy(w.views_pinned, w.host_views.data(), sizeof(ViewDesc) * n_views);
  NES_HIP_TRY(hipMemcpyAsync(w.views.ptr, w.views_pinned, sizeof(ViewDesc) * n_views,
                             hipMemcpyHostToDevice, stream));
  NES_HIP_TRY(hipEventRecord(w.ev_views, stream));
  return NES_OK;
}

int render_work_reserve(RenderWork &w, uint64_t max_slots, uint64_t max_px, uint32_t max_views,
                        int precision) {
  if (max_slots > kMaxSlots) return NES_ERANGE;
  NES_TRY(w.views.reserve(sizeof(ViewDesc) * std::max<uint32_t>(max_views, kPinnedViews)));
  NES_TRY(w.rays.reserve(sizeof(RayData) * max_slots));
  NES_TRY(w.acc.reserve(sizeof(RayAcc) * max_slots));
  NES_TRY(w.counts.reserve(sizeof(uint32_t) * max_slots));
  NES_TRY(w.offsets.reserve(sizeof(uint32_t) * wavefronts(max_slots)));
  NES_TRY(w.ray_sh.reserve(32 * max_slots));
  NES_TRY(w.t_start.reserve(sizeof(float) * max_slots));
  NES_TRY(w.tile_n.reserve(sizeof(uint32_t) * wavefronts(max_slots)));
  NES_TRY(w.host_arrays.reserve(sizeof(HostArray) * kHostArrays));
  NES_TRY(w.out.reserve(out_layout(max_px + kViewAlign * max_views).total));
  NES_TRY(w.total.reserve(kTotBytes));
  return render_reserve_samples(w, precision, std::max<size_t>(max_slots * 4, (size_t)1 << 20));
}

int render_reserve_samples(RenderWork &w, int precision, size_t capacity) {
  if (capacity > 0xffffffffull) capacity = 0xffffffffull;
  const size_t fbytes = precision != NES_PRECISION_MIXED ? sizeof(float4) : sizeof(uint2);
  w.capacity = 0;  // a buffer that cannot be had leaves the work area without any
  NES_TRY(w.samples.reserve(sizeof(uint32_t) * (capacity + 1)));
  NES_TRY(w.sample_out.reserve(sizeof(float4) * (capacity + 1)));
  NES_TRY(w.sample_pos.reserve(sizeof(float4) * (capacity + 1)));
  NES_TRY(w.feat.reserve(fbytes * kParts * (capacity + 1)));
  w.capacity = (uint32_t)capacity;
  w.capacity_precision = precision;
  return NES_OK;
}

static MarchArgs march_args(RenderWork &w, const uint32_t *occ, int k0, int k1, MarchMode mode,
                            uint32_t ray_cap) {
  MarchArgs m{};
  m.views = w.views.as<ViewDesc>();
  m.n_views = w.n_views;
  m.n_slots = w.n_slots;
  m.occ = occ;
  m.rays = w.rays.as<RayData>();
  m.counts = w.counts.as<uint32_t>();
  m.offsets = w.offsets.as<uint32_t>();
  m.samples = w.samples.as<uint32_t>();
  m.t_start = w.t_start.as<float>();
  m.tile_n = w.tile_n.as<uint32_t>();
  m.pos = w.sample_pos.as<float4>();
  m.cursor = w.total.as<uint32_t>();
  m.capacity = w.capacity;
  m.cap = ray_cap;
  m.k_begin = k0;
  m.k_end = k1;
  m.mode = mode;
  return m;
}

static CompositeArgs composite_args(RenderWork &w) {
  CompositeArgs c{};
  c.n_slots = w.n_slots;
  c.rays = w.rays.as<RayData>();
  c.acc = w.acc.as<RayAcc>();
  c.counts = w.counts.as<uint32_t>();
  c.offsets = w.offsets.as<uint32_t>();
  c.samples = w.samples.as<uint32_t>();
  c.t_start = w.t_start.as<float>();
  c.capacity = w.capacity;
  c.o = out_ptrs(w);
  return c;
}

int render_begin(RenderWork &w, hipStream_t stream) {
  ArgViews av{};
  const uint32_t n = w.n_views <= kArgViews ? w.n_views : 0u;
  std::copy(w.host_views.begin(), w.host_views.begin() + n, av.v);
  ArgArrays aa{};
  std::copy(w.host_out, w.host_out + w.n_host_out, aa.a);
  frame_begin<<<1, kFrameThreads, 0, stream>>>(w.total.as<uint32_t>(), av, n, w.views.as<ViewDesc>(), aa,
                                               w.n_host_out, w.host_arrays.as<HostArray>());
  NES_HIP_TRY(hipGetLastError());
  return NES_OK;
}

// Workgroups that store background during the encode: enough in flight for
// the link, and not so much that the encode's loads queue behind it.  Frame
// times with 0 (everything after the composite), 8, 16, 24, 32, 64 of them:
//   stereo 1080p           2170 1790 1721 1896 1972 2042 us
//   solid stereo 1440x1600 2012 1987 1640 1727 1804 1886 us
constexpr uint32_t kBackgroundGroups = 16;
static_assert(kBackgroundGroups % kParts == 0, "the encode's parts follow blockIdx % kParts");

static BackgroundArgs background_args(const RenderWork &w) {
  return BackgroundArgs{w.host_arrays.as<HostArray>(), w.views.as<ViewDesc>(), w.tile_n.as<uint32_t>(),
                        w.n_host_out, w.store_background ? kBackgroundGroups : 0u};
}

// Workgroups per array for stores over the link: a few dozen keep it busy.
static unsigned store_blocks(uint64_t most_bytes) {
  return (unsigned)std::min<uint64_t>(32, std::max<uint64_t>(1, (most_bytes + 4095) / 4096));
}

int render_end(RenderWork &w, hipStream_t stream) {
  uint64_t most = 0;
  for (uint32_t i = 0; i < w.n_host_out; ++i) most = std::max(most, w.host_out[i].bytes);
  frame_end<<<dim3(store_blocks(most), std::max(w.n_host_out, 1u)), 256, 0, stream>>>(
      w.total.as<uint32_t>(), w.total_host, background_args(w), w.capacity);
  NES_HIP_TRY(hipGetLastError());
  return NES_OK;
}

// The requested arrays of one view; false if any of them is not pinned.
static bool host_arrays_of_view(const RenderWork &w, uint32_t view, const nes_view_out &o, HostArray *a, uint32_t *n) {
  const ViewDesc &v = w.host_views[view];
  const size_t px = (size_t)v.width * v.height, base = v.px_base;
  const OutLayout L = out_layout(w.out_px);
  const uint8_t *d = w.out.as<uint8_t>();
  const struct {
    void *dst;
    size_t at;
    uint32_t bpp;
    float scale;
  } all[5] = {{o.rgb24, L.rgb24 + 3 * base, 3, 0.0f},
              {o.depth, L.depth + 4 * base, 4, 0.0f},
              {o.rgb_f32, L.rgbf + 12 * base, 12, 0.0f},
              {o.n_samples, L.nsamp + 2 * base, 2, 0.0f},
              {o.depth_gray8, L.depth + 4 * base, 1, depth_scale(o.depth_far)}};
  for (const auto &x : all) {
    if (!x.dst) continue;
    if (*n == kHostArrays || !device_writable(x.dst, px * x.bpp)) return false;
    const size_t bytes = px * x.bpp, head = (16 - (uintptr_t)x.dst % 16) % 16;
    a[(*n)++] = HostArray{d + x.at, static_cast<uint8_t *>(x.dst), bytes, x.bpp, view,
                          (uint32_t)std::min(head, bytes), x.scale};
  }
  return true;
}

// Outputs below this are stored after the composite in one go: 1 MiB takes
// the link 19 us, about what the march and an encode of such a frame leave.
// At 640x480 (2.1 MB) the split gains 279 -> 247 us.
constexpr uint64_t kBackgroundMinBytes = 1u << 20;

void plan_host_outputs(RenderWork &w, const nes_view_out *outs) {
  uint32_t n = 0;
  for (uint32_t i = 0; i < w.n_views; ++i)
    if (!host_arrays_of_view(w, i, outs[i], w.host_out, &n)) return;
  w.n_host_out = n;
  uint64_t bytes = 0;
  for (uint32_t i = 0; i < n; ++i) bytes += w.host_out[i].bytes;
  w.store_background = bytes >= kBackgroundMinBytes;
}

// Samples a pass is expected to have: a little more than the work area's last
// frame had, at least one per other ray (a view that comes back into sight
// must not run on a handful of workgroups), and about three per ray slot when
// nothing is known.  Only launch sizes follow it.
static size_t expected_samples(const RenderWork &w, int pass) {
  const size_t last = w.last_total[pass];
  const size_t est = last ? std::max<size_t>(last + last / 8, w.n_slots / 2) : (size_t)w.n_slots * 3;
  return std::min<size_t>(est, w.capacity);
}

// Shares of the encode's first parts (see encode_parts) by how far apart
// neighbouring samples lie: distance over focal length, written as the focal
// length in pixels of a view with the same spacing from 2 units off the cube's
// centre.  (From inside, a ray's samples are 0.3 away in the mean.)  Encode
// times below: two eyes (views of up to 10 degrees one), without shares -> with
// them, us, frame after frame.
//
// Mixed: part 0 costs 12 % more than part 7 at 416 (640x480 at 60 degrees), 52 %
// at 935 (1080p) and 75 % at 1439 (2064x2208 at 75 degrees), until neighbours
// share the finest level's cells too.  The shares start at 500 (720p at 620:
// 619 -> 610; 1440x1600 from 6 off at 348: 213 without, 240 with the shares of
// 2 off), reach 12, 9 and 4 % at 935 (1293 -> 1234), stay at 21, 15 and 6 % from
// 1250 to 3600 (1440x1600 from 1 off 7200 -> 5700, 2064x2208 from 0.8 off 18900 ->
// 15600) and end at 9600 (2064x2208 from 0.6 off, 4797: 31700 -> 27600; 1080p
// from 0.3 off, 6233: 15900 -> 14000, with 21 % 15300; 640x480 at 5 degrees
// from 0.6 off, 18300: 1080, with 21 % 1200).
//
// FP32: a hashed level fills an XCD's L2 by itself; shares of 15, 10 and 5 %
// gain from 485 on (at 425 1800x1700 loses, 433 -> 456; 900x800 at 521 632 ->
// 618, 720p 879 -> 818, 1080p 1857 -> 1680, 640x480 of one eye from 0.3 off,
// 2773, 1964 -> 1650), up to about 5000 (640x480 at 10 degrees: 3918 2020 -> 2009,
// 5486 1690, with 15 % 1733, 9143 1396 -> 1666).
// Between limits: of 1 M samples the helpers' extra 4 MB of table cost more
// than they take off part 0 (640x480: 201 -> 204, the frame 535 -> 546); and
// where the samples are more than twice the grid's threads its passes mix the
// parts' turns and four such levels take turns in one L2 (26.7 M samples
// 2690 -> 3100, 50.8 M 4280 -> 5460).
constexpr size_t kF32ShareMin = 3u << 19, kF32ShareMax = 2 * 256 * (size_t)kMaxPartBlocks;
constexpr double kShareEnd = 9600.0;

static double spacing_focal(const ViewDesc &v) {
  double d2 = 0.0;
  for (int i = 0; i < 3; ++i) d2 += ((double)v.c2w[4 * i + 3] - 0.5) * ((double)v.c2w[4 * i + 3] - 0.5);
  return 2.0 * v.focal / std::max(std::sqrt(d2), 0.3);
}

static PartShares part_shares(const RenderWork &w, bool f32, size_t expect) {
  double focal = 0.0;
  for (uint32_t i = 0; i < w.n_views; ++i)
    focal += spacing_focal(w.host_views[i]) * w.host_views[i].slot_count / w.n_slots;
  if (!(focal < kShareEnd)) return PartShares{};  // (nor for a camera that is not finite)
  const auto q = [](double v) { return (uint32_t)(std::max(v, 0.0) * 65536); };
  if (f32) {
    if (expect < kF32ShareMin || expect > kF32ShareMax) return PartShares{};
    const double s = 0.15 * std::min({(focal - 470.0) / 130.0, (6000.0 - focal) / 2000.0, 1.0});
    return PartShares{{q(s), q(s - 0.05), q(s - 0.10)}, 0u};
  }
  const double f = std::min({std::max((focal - 500.0) / 600.0, 0.0), (kShareEnd - focal) / 4800.0, 1.25});
  return PartShares{{q(0.17 * f), q(0.12 * f), q(0.05 * f)}, 0u};
}

int render_launch_pass(const SceneDev &scene, RenderWork &w, int precision, int k0, int k1,
                       bool first, bool last, hipStream_t stream, uint32_t ray_cap, bool resume) {
  uint32_t *const total = w.total.as<uint32_t>();
  uint32_t *cursor = total + (first ? kTotCursor : kTotCursorLater);
  const uint32_t cap = w.capacity;
  uint64_t *stamp = reinterpret_cast<uint64_t *>(total + kTotStamps) + kStampPass + (first ? 0 : kStampStages);
  const bool f32 = precision != NES_PRECISION_MIXED;
  MarchArgs m = march_args(w, scene.occ, k0, k1, first ? kMarchFirst : kMarchNext, ray_cap);
  m.cursor = cursor;
  m.packed = f32 ? 0 : 1;
  m.resume = resume ? 1 : 0;
  // the ray itself is read by later passes (by passes over windows of steps
  // also where this one found no samples) and by the FP32 MLP; the mixed MLP
  // reads ray_sh
  m.store_rays = !first ? 0 : k1 < kMaxSteps ? 2 : !last || f32 ? 1 : 0;
  m.ray_sh = f32 ? nullptr : w.ray_sh.as<uint2>();
  m.stamp = stamp;
  NES_TRY(launch_march(m, stream));
  // grids for the expected samples, with grid-stride loops: the sample count
  // stays on the device
  const size_t expect = expected_samples(w, first ? 0 : 1);
  const PartShares shares = part_shares(w, f32, expect);
  const uint32_t bpp = part_blocks(expect + (expect * shares.share[0] >> 16));
  BackgroundArgs bg = background_args(w);
  if (!first) bg.groups = 0;
  if (f32) {
    encode_parts<float><<<bpp * kParts + bg.groups, 256, 0, stream>>>(w.sample_pos.as<float4>(), cursor, cap,
                                                           scene.table_f32, w.feat.as<float4>(),
                                                           bpp, shares, bg, stamp + 1);
    NES_HIP_TRY(hipGetLastError());
    if (precision == NES_PRECISION_FP32_VALU)
      mlp_fp32_valu<<<256 * 4, 256, 0, stream>>>(w.sample_pos.as<float4>(), w.feat.as<float4>(),
                                                 cursor, cap, w.rays.as<RayData>(),
                                                 scene.weights_f32, w.sample_out.as<float4>(),
                                                 stamp + 2);
    else
      NES_TRY(launch_mlp_f32(scene.weights_f32, w, cursor, stream, stamp + 2));
  } else {
    encode_parts<_Float16><<<bpp * kParts + bg.groups, 256, 0, stream>>>(w.sample_pos.as<uint2>(), cursor,
                                                              cap, scene.table_f16,
                                                              w.feat.as<uint2>(), bpp, shares, bg, stamp + 1);
    NES_HIP_TRY(hipGetLastError());
    const unsigned mlp_blocks =
        (unsigned)std::min<size_t>(256 * 8, std::max<size_t>(expect / (16 * kEvalWaves), 64));
    mlp_mixed<<<mlp_blocks, 256, 0, stream>>>(w.samples.as<uint32_t>(), w.feat.as<uint2>(), cursor,
                                           cap, w.ray_sh.as<uint2>(),
                                           reinterpret_cast<const half8 *>(scene.wfrag),
                                           w.sample_out.as<uint2>(), stamp + 2);
  }
  NES_HIP_TRY(hipGetLastError());
  CompositeArgs c = composite_args(w);
  c.views = w.views.as<ViewDesc>();
  c.n_views = w.n_views;
  c.n_ptr = cursor;
  c.first = first ? 1 : 0;
  c.last = last ? 1 : 0;
  c.stats = total;
  c.stamp = stamp + 3;
  if (f32) return composite_pass(c, w.sample_out.as<float4>(), stream);
  return composite_pass(c, w.sample_out.as<uint2>(), stream);
}

int render_launch_frame(const SceneDev &scene, RenderWork &w, int precision, hipStream_t stream) {
  w.whole_frame = true;
  NES_TRY(render_begin(w, stream));
  const uint32_t cap1 = w.first_pass_cap;
  if (cap1 >= (uint32_t)kMaxSteps) {
    w.frame_passes = 1;
    NES_TRY(render_launch_pass(scene, w, precision, 0, kMaxSteps, true, true, stream));
  } else {
    // two passes, no host round trip between them: the second resumes every
    // ray the first left above T = 1e-4 at the step after its last sample
    w.frame_passes = 2;
    NES_TRY(render_launch_pass(scene, w, precision, 0, kMaxSteps, true, false, stream, cap1, false));
    NES_TRY(render_launch_pass(scene, w, precision, 0, kMaxSteps, false, true, stream, kMaxSteps, true));
  }
  return render_end(w, stream);
}

// A third or later pass counts its samples on the second one's cursor again.
static int clear_later_cursor(RenderWork &w, hipStream_t stream) {
  zero_u32<<<1, 64, 0, stream>>>(w.total.as<uint32_t>() + kTotCursorLater, 1);
  NES_HIP_TRY(hipGetLastError());
  return NES_OK;
}

uint32_t render_frame_max_total(const RenderWork &w) {
  return std::max(w.total_host[0], w.frame_passes > 1 ? w.total_host[1] : 0u);
}

int render_launch_bounded(const SceneDev &scene, RenderWork &w, int precision,
                          hipStream_t stream) {
  if (w.capacity < w.n_slots) {
    set_last_error("sample buffers hold less than one sample per ray");
    return NES_ENOMEM;
  }
  // each pass emits at most n_slots * cap <= capacity samples: no overflow
  const uint32_t cap = std::min<uint32_t>(w.capacity / std::max<uint32_t>(w.n_slots, 1u),
                                          kMaxSteps);
  const int passes = (int)((kMaxSteps + cap - 1) / cap);
  w.frame_passes = (uint32_t)passes;
  w.whole_frame = false;
  NES_TRY(render_begin(w, stream));
  for (int p = 0; p < passes; ++p) {
    if (p > 1) NES_TRY(clear_later_cursor(w, stream));
    NES_TRY(render_launch_pass(scene, w, precision, 0, kMaxSteps, p == 0, p == passes - 1, stream, cap, p > 0));
  }
  return render_end(w, stream);
}

bool render_growth_fits(const RenderWork &w, int precision, size_t capacity) {
  if (!w.budget) return true;
  const size_t cur = w.samples.bytes + w.sample_out.bytes + w.sample_pos.bytes + w.feat.bytes;
  return work_device_bytes(w) - cur + sample_buffer_bytes(capacity, precision) <= w.budget;
}

size_t sample_buffer_bytes(size_t capacity, int precision) {
  const size_t c = capacity + 1, fb = precision != NES_PRECISION_MIXED ? sizeof(float4) : sizeof(uint2);
  size_t t = 0;
  // the buffers of render_reserve_samples, with DevBuf's growth slack
  for (size_t need : {sizeof(uint32_t) * c, sizeof(float4) * c, sizeof(float4) * c, fb * kParts * c})
    t += need + need / 8 + 256;
  return t;
}

// Early-termination policy for the next frame of this work area.  A single
// pass evaluates every occupied sample; when more than 5 % of them lie behind
// the point where T fell below 1e-4, the next frame runs two passes, the first
// giving each ray as many samples as the terminated rays needed on average
// (rounded up).  Multi-pass frames go back to one pass when the first pass
// stopped fewer than 1 % of the pixels with steps still ahead of them.
FrameCounts render_frame_finish(RenderWork &w) {
  FrameCounts c;
  c.passes = w.frame_passes;
  // the passes of other frames (bounded, windows) say nothing about a whole one
  w.last_total[0] = w.whole_frame ? w.total_host[kTotCursor] : 0u;
  w.last_total[1] = w.whole_frame && c.passes == 2 ? w.total_host[kTotCursorLater] : 0u;
  c.evaluated = w.total_host[2];
  for (int s = 0; s < kTotTermSlots; ++s) {
    const uint32_t *t = w.total_host + kTotTermBase + kTotTermStride * s;
    c.terminated += t[0];
    c.term_samples += t[1];
    c.wasted += t[2];
    c.saved_rays += t[3];
  }
  c.composited = c.evaluated - std::min(c.wasted, c.evaluated);
  // one pass: switch to two when more than 5 % of the evaluated samples lay
  // behind T < 1e-4; several passes: keep two while more than 1 % of the
  // pixels stopped early with steps left (the work the first pass saved)
  const bool wasteful = c.wasted * 20 > c.evaluated;
  const bool saving = c.saved_rays * 100 > w.pixels;
  if (c.terminated && ((c.passes == 1 && wasteful) || (c.passes > 1 && saving))) {
    const uint64_t m = (c.term_samples + c.terminated - 1) / c.terminated;
    w.first_pass_cap = (uint32_t)std::min<uint64_t>(std::max<uint64_t>(m, 1), kMaxSteps - 1);
  } else {
    w.first_pass_cap = kMaxSteps;
  }
  return c;
}

// Single-stage launchers reused by the training step (rays prepared and the
// sample cursor cleared by the caller, one output index per ray slot).
int launch_march_emit(const uint32_t *occ, RenderWork &w, int k0, int k1, hipStream_t stream) {
  return launch_march(march_args(w, occ, k0, k1, kMarchPrepared, kMaxSteps), stream);
}

// Rays drawn at random share no cells, and an XCD's time goes with its hashed
// levels' L2 lines (four to five per sample and level): parts 7, 6 and 5 have
// two such levels, parts 0, 1 and 2 one.  Helping the former takes a 2^18-ray
// batch's encode from 424 to 329 us (65536 rays 112 -> 88, 16384 33 -> 28); 20
// or 30 % instead of 25 gained less.  A caller's own rays may be in any order
// and are not shared.
constexpr uint32_t kScatteredShare = 65536 / 4;

int launch_encode_f32(const float *table, RenderWork &w, uint32_t n, bool scattered, hipStream_t stream) {
  PartShares shares{};
  if (scattered) shares = PartShares{{kScatteredShare, kScatteredShare, kScatteredShare}, 1u};
  const uint32_t bpp = part_blocks(n + ((uint64_t)n * shares.share[0] >> 16));
  encode_parts<float><<<bpp * kParts, 256, 0, stream>>>(w.sample_pos.as<float4>(),
                                                         w.total.as<uint32_t>(), w.capacity,
                                                         table, w.feat.as<float4>(), bpp, shares, BackgroundArgs{},
                                                         nullptr);
  NES_HIP_TRY(hipGetLastError());
  return NES_OK;
}

int launch_composite(RenderWork &w, hipStream_t stream) {
  CompositeArgs c = composite_args(w);
  c.n_ptr = w.total.as<uint32_t>();
  c.first = c.last = c.keep = 1;
  return composite_pass(c, w.sample_out.as<float4>(), stream);
}

// Initial sample capacity: four samples per ray slot, or what the last render
// of this work area needed.
int render_prepare_capacity(RenderWork &w, int precision) {
  size_t want = std::max<size_t>((size_t)w.n_slots * 4, 1u << 20);
  if (w.capacity >= want && w.capacity_precision == precision) return NES_OK;
  want = std::max<size_t>(want, w.capacity);
  return render_reserve_samples(w, precision, want);
}

size_t work_device_bytes(const RenderWork &w) {
  size_t b = 0;
  for (const DevBuf *d : {&w.views, &w.rays, &w.acc, &w.counts, &w.offsets, &w.ray_sh, &w.t_start, &w.gray, &w.tile_n, &w.host_arrays, &w.samples,
                          &w.sample_out, &w.sample_pos, &w.feat, &w.out, &w.total})
    b += d->bytes;
  return b;
}

// Over budget: drop every buffer (they only grow) so that a later, smaller
// render starts from nothing, and report NES_ENOMEM.
static int check_budget(RenderWork &w) {
  if (w.budget && work_device_bytes(w) > w.budget) {
    for (DevBuf *d : {&w.views, &w.rays, &w.acc, &w.counts, &w.offsets, &w.ray_sh, &w.t_start, &w.gray, &w.tile_n, &w.host_arrays, &w.samples,
                      &w.sample_out, &w.sample_pos, &w.feat, &w.out, &w.total})
      d->release();
    w.capacity = 0;
    w.capacity_precision = -1;
    w.n_views = 0;
    set_last_error("render buffers exceed the context's HBM budget");
    return NES_ENOMEM;
  }
  return NES_OK;
}

static int render_enqueue_inner(const SceneDev &scene, RenderWork &w, int precision,
                                const nes_camera *views, int n_views, int steps_per_pass,
                                hipStream_t stream, nes_render_stats *stats,
                                const nes_view_out *outs);

int render_enqueue(const SceneDev &scene, RenderWork &w, int precision,
                   const nes_camera *views, int n_views, int steps_per_pass,
                   hipStream_t stream, nes_render_stats *stats, const nes_view_out *outs,
                   bool *delivered) {
  const int rc = render_enqueue_inner(scene, w, precision, views, n_views, steps_per_pass, stream,
                                      stats, outs);
  if (delivered) *delivered = rc == NES_OK && w.n_host_out != 0;
  // the caller's memory is not referred to after this call
  if (rc != NES_OK && w.n_host_out) hipStreamSynchronize(stream);
  w.n_host_out = 0;
  w.store_background = false;
  if (rc != NES_OK) {
    // a failed render leaves nothing to fetch
    w.n_views = 0;
    w.out_px = 0;
  }
  return rc;
}

static bool valid_precision(int p) {
  return p == NES_PRECISION_FP32 || p == NES_PRECISION_MIXED || p == NES_PRECISION_FP32_VALU;
}

// Milliseconds per tick of the device clock.
static double tick_ms() {
  static const double ms = [] {
    int khz = 0;
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, 0) != hipSuccess || khz <= 0) khz = 100000;
    return 1.0 / khz;
  }();
  return ms;
}

double frame_ms(const RenderWork &w) {
  const uint64_t *st = reinterpret_cast<const uint64_t *>(w.total_host + kTotStamps);
  return st[kStampEnd] > st[kStampBegin] ? (double)(st[kStampEnd] - st[kStampBegin]) * tick_ms() : 0.0;
}

// Stage times of `passes` passes from the stamps of the last frame_end:
// t[0..3] += march, encode, MLPs, composite; returns begin to end.
static double add_stage_times(const RenderWork &w, int first_pass, int passes, double t[4]) {
  const uint64_t *st = reinterpret_cast<const uint64_t *>(w.total_host + kTotStamps);
  auto ms = [](uint64_t a, uint64_t b) { return b > a ? (double)(b - a) * tick_ms() : 0.0; };
  for (int p = first_pass; p < first_pass + passes; ++p) {
    const uint64_t *s = st + kStampPass + p * kStampStages;
    const uint64_t next = p + 1 < first_pass + passes ? s[kStampStages] : st[kStampEnd];
    for (int k = 0; k < kStampStages; ++k) t[k] += ms(s[k], k + 1 < kStampStages ? s[k + 1] : next);
  }
  return frame_ms(w);
}

static int render_enqueue_inner(const SceneDev &scene, RenderWork &w, int precision,
                                const nes_camera *views, int n_views, int steps_per_pass,
                                hipStream_t stream, nes_render_stats *stats,
                                const nes_view_out *outs) {
  if (!valid_precision(precision) || steps_per_pass < 0) return NES_EINVAL;
  NES_TRY(render_setup(w, views, n_views, stream));
  NES_TRY(render_prepare_capacity(w, precision));
  NES_TRY(check_budget(w));
  double t[4] = {0, 0, 0, 0};  // march, encode, MLPs, composite
  double total = 0, lost = 0;  // (lost: launches that overflowed)
  FrameCounts fc;
  if (steps_per_pass == 0 || steps_per_pass >= kMaxSteps) {
    // whole frame: one pass, or two when the previous frame of this work area
    // evaluated samples behind terminated rays (steps_per_pass 0)
    if (steps_per_pass) w.first_pass_cap = kMaxSteps;
    if (outs) plan_host_outputs(w, outs);
    bool bounded = false;
    for (int attempt = 0;; ++attempt) {
      if (bounded)
        NES_TRY(render_launch_bounded(scene, w, precision, stream));
      else
        NES_TRY(render_launch_frame(scene, w, precision, stream));
      NES_HIP_TRY(hipStreamSynchronize(stream));
      const uint32_t n = render_frame_max_total(w);
      if (bounded || n <= w.capacity) break;
      if (attempt > 0) {
        set_last_error("sample capacity still exceeded after regrowth");
        return NES_ENOMEM;
      }
      lost += frame_ms(w);
      // grow when the budget and the device allow it, else render within the
      // buffers (the first of two passes has stored background already: the
      // frame is not given up here)
      const size_t want = (size_t)n + n / 8 + 1024, had = w.capacity;
      bounded = !render_growth_fits(w, precision, want);
      if (!bounded && render_reserve_samples(w, precision, want) != NES_OK) {
        NES_TRY(render_reserve_samples(w, precision, had));
        bounded = true;
      }
    }
    if (bounded) {
      double unused[4] = {0, 0, 0, 0};
      total = t[1] = add_stage_times(w, 0, 1, unused);  // no per-stage times over bounded passes
    } else {
      total = add_stage_times(w, 0, (int)w.frame_passes, t);
    }
    fc = render_frame_finish(w);
  } else {
    // fixed windows of steps_per_pass march steps, one host round trip each
    const int spp = steps_per_pass;
    const int passes = (kMaxSteps + spp - 1) / spp;
    w.frame_passes = 1;
    w.whole_frame = false;
    for (int p = 0; p < passes; ++p) {
      const int k0 = p * spp, k1 = std::min(kMaxSteps, k0 + spp);
      uint32_t n = 0;
      for (int attempt = 0;; ++attempt) {
        if (p == 0)
          NES_TRY(render_begin(w, stream));
        else
          NES_TRY(clear_later_cursor(w, stream));
        NES_TRY(render_launch_pass(scene, w, precision, k0, k1, p == 0, p == passes - 1, stream));
        NES_TRY(render_end(w, stream));
        NES_HIP_TRY(hipStreamSynchronize(stream));
        n = w.total_host[p == 0 ? 0 : 1];
        if (n <= w.capacity) break;
        if (attempt > 0) {
          set_last_error("sample capacity still exceeded after regrowth");
          return NES_ENOMEM;
        }
        if (p == 0) lost += frame_ms(w);  // (later passes run on the first one's clock)
        const size_t want = (size_t)n + n / 8 + 1024;
        if (!render_growth_fits(w, precision, want)) {
          set_last_error("a pass's samples exceed the context's HBM budget");
          return NES_ENOMEM;
        }
        NES_TRY(render_reserve_samples(w, precision, want));
      }
      total = add_stage_times(w, p == 0 ? 0 : 1, 1, t);
    }
    w.frame_passes = (uint32_t)passes;
    fc = render_frame_finish(w);
    w.first_pass_cap = kMaxSteps;  // windows are the caller's choice, not learned from
  }
  if (stats) {
    stats->rays = w.pixels;
    stats->samples = fc.evaluated;
    stats->ms_total = total + lost;
    stats->ms_march = t[0];
    stats->ms_encode = t[1];
    stats->ms_mlp = t[2];
    stats->ms_eval = t[1] + t[2];
    stats->ms_composite = t[3];
    stats->composited = fc.composited;
    stats->terminated_rays = fc.terminated;
    stats->passes = fc.passes;
  }
  return NES_OK;
}

int render_fetch(RenderWork &w, int view, const nes_view_out *out, hipStream_t stream) {
  if (!out || view < 0 || (uint32_t)view >= w.n_views) return NES_EINVAL;
  const ViewDesc &v = w.host_views[(size_t)view];
  const size_t px = (size_t)v.width * v.height, base = v.px_base;
  if (base + px > w.out_px) {
    set_last_error("view lies outside the last render's outputs");
    return NES_EINVAL;
  }
  ArgArrays arrays{};
  uint32_t n = 0;
  if (host_arrays_of_view(w, (uint32_t)view, *out, arrays.a, &n)) {
    // pinned memory: every array in one launch
    if (n) store_arrays<<<dim3(store_blocks(12 * px), n), 256, 0, stream>>>(arrays);
    NES_HIP_TRY(hipGetLastError());
    NES_HIP_TRY(hipStreamSynchronize(stream));
    return NES_OK;
  }
  const OutLayout L = out_layout(w.out_px);
  const uint8_t *o = w.out.as<uint8_t>();
  if (out->rgb24)
    NES_HIP_TRY(hipMemcpyAsync(out->rgb24, o + L.rgb24 + 3 * base, 3 * px, hipMemcpyDeviceToHost, stream));
  if (out->depth)
    NES_HIP_TRY(hipMemcpyAsync(out->depth, o + L.depth + 4 * base, 4 * px, hipMemcpyDeviceToHost, stream));
  if (out->rgb_f32)
    NES_HIP_TRY(hipMemcpyAsync(out->rgb_f32, o + L.rgbf + 12 * base, 12 * px, hipMemcpyDeviceToHost, stream));
  if (out->n_samples)
    NES_HIP_TRY(hipMemcpyAsync(out->n_samples, o + L.nsamp + 2 * base, 2 * px, hipMemcpyDeviceToHost, stream));
  if (out->depth_gray8) {
    NES_TRY(w.gray.reserve(px));
    depth_gray8_kernel<<<(unsigned)((px + 255) / 256), 256, 0, stream>>>(
        reinterpret_cast<const float *>(o + L.depth) + base, px, depth_scale(out->depth_far),
        w.gray.as<uint8_t>());
    NES_HIP_TRY(hipGetLastError());
    NES_HIP_TRY(hipMemcpyAsync(out->depth_gray8, w.gray.ptr, px, hipMemcpyDeviceToHost, stream));
  }
  NES_HIP_TRY(hipStreamSynchronize(stream));
  return NES_OK;
}

std::shared_ptr<SceneDev> new_scene() {
  return std::shared_ptr<SceneDev>(new SceneDev(), [](SceneDev *p) {
    scene_free(*p);
    delete p;
  });
}

std::shared_ptr<SceneDev> ctx_scene(nes_ctx *ctx) {
  std::lock_guard<std::mutex> lk(ctx->scene_mu);
  return ctx->scene;
}

}  // namespace nes

using namespace nes;

extern "C" {

int nes_ctx_create(const nes_scene_desc *scene, uint64_t hbm_budget_bytes, nes_ctx **out) {
  if (!scene || !out) return NES_EINVAL;
  NES_TRY(ensure_device());
  nes_ctx *c = new nes_ctx();
  c->budget = hbm_budget_bytes ? hbm_budget_bytes : (16ull << 30);
  c->work.budget = c->budget;
  c->scene = new_scene();
  int rc = scene_upload(*c->scene, scene);
  if (rc == NES_OK && hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) rc = NES_EIO;
  if (rc != NES_OK) {
    delete c;
    return rc;
  }
  *out = c;
  return NES_OK;
}

int nes_ctx_destroy(nes_ctx *ctx) {
  if (!ctx) return NES_EINVAL;
  {
    std::lock_guard<std::mutex> lk(ctx->mu);
    if (ctx->stream) hipStreamSynchronize(ctx->stream);
    render_work_free(ctx->work);
    if (ctx->stream) hipStreamDestroy(ctx->stream);
  }
  delete ctx;  // frees the scene copies (servers on it are destroyed first)
  return NES_OK;
}

int nes_ctx_update_scene(nes_ctx *ctx, const nes_scene_desc *scene) {
  if (!ctx || !scene || !scene->table || !scene->weights || !scene->occupancy) return NES_EINVAL;
  std::shared_ptr<SceneDev> next;
  {
    // reuse the previous copy once no render or batch holds it any more
    std::lock_guard<std::mutex> lk(ctx->scene_mu);
    if (ctx->spare && ctx->spare.use_count() == 1) next = ctx->spare;
    ctx->spare.reset();
  }
  if (!next) next = new_scene();
  // the copy being written is referenced by no launched work
  NES_TRY(scene_upload(*next, scene));
  std::lock_guard<std::mutex> lk(ctx->scene_mu);
  ctx->spare = ctx->scene;
  ctx->scene = next;
  return NES_OK;
}

int nes_render_device(nes_ctx *ctx, int precision, const nes_camera *views, int n_views,
                      int steps_per_pass, nes_render_stats *stats) {
  if (!ctx) return NES_EINVAL;
  std::lock_guard<std::mutex> lk(ctx->mu);
  const std::shared_ptr<SceneDev> sc = ctx_scene(ctx);
  return render_enqueue(*sc, ctx->work, precision, views, n_views, steps_per_pass, ctx->stream,
                        stats);
}

int nes_render_fetch(nes_ctx *ctx, int view, const nes_view_out *out) {
  if (!ctx) return NES_EINVAL;
  std::lock_guard<std::mutex> lk(ctx->mu);
  return render_fetch(ctx->work, view, out, ctx->stream);
}

int nes_render(nes_ctx *ctx, int precision, const nes_camera *views, int n_views,
               const nes_view_out *outs, int steps_per_pass, nes_render_stats *stats) {
  if (!ctx || !outs) return NES_EINVAL;
  std::lock_guard<std::mutex> lk(ctx->mu);
  const std::shared_ptr<SceneDev> sc = ctx_scene(ctx);
  bool delivered = false;
  NES_TRY(render_enqueue(*sc, ctx->work, precision, views, n_views, steps_per_pass, ctx->stream,
                         stats, outs, &delivered));
  for (int i = 0; i < n_views && !delivered; ++i)
    NES_TRY(render_fetch(ctx->work, i, &outs[i], ctx->stream));
  return NES_OK;
}

}  // extern "C"
