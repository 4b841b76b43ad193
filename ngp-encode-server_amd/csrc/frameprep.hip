// frameprep.hip -- nearer-depth composite + RGB24 -> YUV420P (K5).
//
// Replaces RenderedFrame::convert_frame (include/base/video/
// rendered_frame.h:24-33) -> SwsContextManager (src/base/video/
// type_managers.cc:143-155): sws_getContext(W, H, RGB24, W, H, YUV420P,
// flags = 0) + one whole-frame sws_scale.  With flags 0 libswscale 5.5 picks
// its default bicubic scaler and, for an RGB source, the generic path:
//   luma   Y14 = (RY r + GY g + BY b + (16.5 << 15)) >> 9      (rgb24ToY_c)
//          Y15 = 2 * Y14 (1-tap unscaled hScale16To15, shift 13)
//          Y   = clip((Y15 + 64) >> 7)                          (yuv2plane1_8_c)
//   chroma U14 = (RU (r0+r1) + GU (g0+g1) + BU (b0+b1) + (256.03 << 15)) >> 10
//          on horizontally paired pixels (rgb24ToUV_half_c), U15 = 2 * U14,
//          then an 8-tap 2:1 bicubic vertical filter (initFilter, 12-bit
//          coefficients, clamp-to-edge borders) whose arithmetic depends on
//          the build: x86-64 uses yuv2yuvX_sse3 (pmulhw taps) for every output
//          row but the last two luma rows, which use yuv2planeX_8_c.
//
// Kernel layout: one workgroup per tile of one frame (a 256-pixel strip of some
// chroma rows).  Phase 1 streams the tile's source rows (plus the filter's
// 6-row halo) once, composites A/B, writes luma and parks the 15-bit chroma
// intermediates in LDS; phase 2 runs the vertical chroma filter out of LDS.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>

#include "nes_internal.h"

namespace nes {

// ------------------------------------------------------------------ host
// utils.c initFilter() of libswscale 5.5 restated for the bicubic scaler
// (param B = 0, C = 0.6), followed by the x86 filter alignment (2 for a
// vertical filter), the border fix-up and the error-diffusion normalisation.
static int init_filter(int x_inc, int src_w, int dst_w, int filter_align,
                       int one, int src_pos, int dst_pos,
                       std::vector<int16_t> &coef, std::vector<int32_t> &fpos) {
  const int ratio = src_w / dst_w;
  int lg = 0;
  for (unsigned r = (unsigned)(ratio > 0 ? ratio : 1); r >>= 1;) ++lg;
  const int64_t fone = 1ll << (54 - (lg < 8 ? lg : 8));
  std::vector<int64_t> filt;
  std::vector<int32_t> p((size_t)dst_w + 3, 0);
  int size;
  if (std::llabs((long long)x_inc - 0x10000) < 10 && src_pos == dst_pos) {
    size = 1;
    filt.assign((size_t)dst_w, fone);
    for (int i = 0; i < dst_w; ++i) p[i] = i;
  } else {
    size = x_inc <= (1 << 16) ? 5 : 1 + (4 * src_w + dst_w - 1) / dst_w;
    size = std::min(size, src_w - 2);
    size = std::max(size, 1);
    filt.assign((size_t)dst_w * size, 0);
    int64_t xdst = ((dst_pos * (int64_t)x_inc) >> 7) - ((src_pos * 0x10000ll) >> 7);
    const int64_t B = 0, C = (int64_t)(0.6 * (1 << 24));
    for (int i = 0; i < dst_w; ++i) {
      int xx = (int)((xdst - (size - 2) * (1ll << 16)) / (1 << 17));
      p[i] = xx;
      for (int j = 0; j < size; ++j, ++xx) {
        int64_t d = std::llabs((int64_t)xx * (1 << 17) - xdst) << 13;
        if (x_inc > (1 << 16)) d = d * dst_w / src_w;
        int64_t c = 0;
        if (d < (1ll << 31)) {
          int64_t dd = (d * d) >> 30, ddd = (dd * d) >> 30;
          if (d < (1ll << 30))
            c = (12 * (1 << 24) - 9 * B - 6 * C) * ddd +
                (-18 * (1 << 24) + 12 * B + 6 * C) * dd +
                (6 * (1 << 24) - 2 * B) * (1 << 30);
          else
            c = (-B - 6 * C) * ddd + (6 * B + 30 * C) * dd +
                (-12 * B - 48 * C) * d + (8 * B + 24 * C) * (1 << 30);
        }
        c /= (1ll << 54) / fone;
        filt[(size_t)i * size + j] = c;
      }
      xdst += 2 * (int64_t)x_inc;
    }
  }
  // Reduce: drop negligible leading taps (shifting the window right) and
  // measure the widest remaining support.
  const double cutoff = 0.002 * (double)fone;
  int min_size = 0;
  for (int i = dst_w - 1; i >= 0; --i) {
    int64_t *f = &filt[(size_t)i * size];
    int keep = size;
    int64_t acc = 0;
    for (int j = 0; j < size; ++j) {
      acc += std::llabs(f[0]);
      if ((double)acc > cutoff) break;
      if (i < dst_w - 1 && p[i] >= p[i + 1]) break;
      for (int k = 1; k < size; ++k) f[k - 1] = f[k];
      f[size - 1] = 0;
      p[i]++;
    }
    acc = 0;
    for (int j = size - 1; j > 0; --j) {
      acc += std::llabs(f[j]);
      if ((double)acc > cutoff) break;
      keep--;
    }
    min_size = std::max(min_size, keep);
  }
  if (min_size == 1 && filter_align == 2) filter_align = 1;
  const int out = (min_size + filter_align - 1) & ~(filter_align - 1);
  std::vector<int64_t> fr((size_t)dst_w * out, 0);
  for (int i = 0; i < dst_w; ++i)
    for (int j = 0; j < out && j < size; ++j) fr[(size_t)i * out + j] = filt[(size_t)i * size + j];
  // Borders: fold taps that fall outside the source onto the edge sample.
  for (int i = 0; i < dst_w; ++i) {
    int64_t *f = &fr[(size_t)i * out];
    if (p[i] < 0) {
      for (int j = 1; j < out; ++j) {
        int left = std::max(j + p[i], 0);
        f[left] += f[j];
        f[j] = 0;
      }
      p[i] = 0;
    }
    if (p[i] + out > src_w) {
      int shift = p[i] + std::min(out - src_w, 0);
      int64_t acc = 0;
      for (int j = out - 1; j >= 0; --j)
        if (p[i] + j >= src_w) {
          acc += f[j];
          f[j] = 0;
        }
      for (int j = out - 1; j >= 0; --j) f[j] = j < shift ? 0 : f[j - shift];
      p[i] -= shift;
      f[src_w - 1 - p[i]] += acc;
    }
  }
  coef.assign((size_t)dst_w * out, 0);
  fpos.assign((size_t)dst_w, 0);
  for (int i = 0; i < dst_w; ++i) {
    int64_t sum = 0, err = 0;
    for (int j = 0; j < out; ++j) sum += fr[(size_t)i * out + j];
    sum = (sum + one / 2) / one;
    if (!sum) sum = 1;
    for (int j = 0; j < out; ++j) {
      int64_t v = fr[(size_t)i * out + j] + err;
      int64_t iv = (v >= 0 ? v + (sum >> 1) : v - (sum >> 1)) / sum;
      coef[(size_t)i * out + j] = (int16_t)iv;
      err = v - iv * sum;
    }
    fpos[i] = p[i];
  }
  return out;
}

VFilter build_vchroma_filter(int h) {
  // Source chroma is full height (RGB input), destination half height.  Both
  // chroma positions default to -513, i.e. centred: get_local_pos() = 128.
  const int dst_h = (h + 1) >> 1;
  const int inc = (int)((((int64_t)h << 16) + (dst_h >> 1)) / dst_h);
  VFilter f;
  f.taps = init_filter(inc, h, dst_h, 2, 1 << 12, 128, 128, f.coef, f.pos);
  return f;
}

namespace {
std::mutex g_filter_mu;
std::map<int, VRows> g_filters;  // by frame height
constexpr size_t kMaxFilters = 8192;
}  // namespace

int get_vrows(int h, VRows *out) {
  std::lock_guard<std::mutex> lk(g_filter_mu);
  auto it = g_filters.find(h);
  if (it == g_filters.end()) {
    const VFilter f = build_vchroma_filter(h);
    const int ch = (int)f.pos.size();
    VRows r;
    r.taps = f.taps;
    bool ok = f.taps >= 1 && f.taps <= kVTaps && ch == h / 2;
    for (int k = 0; ok && k < ch; ++k) {
      const int c = row_class(k, ch);
      int16_t coef[kVTaps] = {};
      std::copy_n(&f.coef[(size_t)k * f.taps], f.taps, coef);
      if (c != 2) {
        r.pos[c] = f.pos[k];
      } else {
        ok = f.taps == kVTaps && f.pos[k] == 2 * k - 3 && (k == 2 || std::equal(coef, coef + kVTaps, r.coef[2]));
      }
      std::copy_n(coef, kVTaps, r.coef[c]);
    }
    if (!ok) {
      set_last_error("unsupported vertical filter size");
      return NES_ERANGE;
    }
    if (g_filters.size() >= kMaxFilters) g_filters.clear();
    it = g_filters.emplace(h, r).first;
  }
  *out = it->second;
  return NES_OK;
}

// ---------------------------------------------------------------- device
constexpr int kFpQuads = 64;    // 4-pixel quads per tile row, one per lane
constexpr int kFpWaves = 4;
constexpr int kFpXcds = 8;      // workgroup b runs on XCD b % 8
// Workgroups in a row of the grid.  One dimension of a launch holds fewer than
// 2^32 threads; tens of thousands of narrow frames have more tiles than that.
constexpr uint32_t kFpGridRow = 1u << 23;
static_assert(kFpGridRow % kFpXcds == 0, "a row starts on XCD 0");

struct FrameprepArgs {
  const uint8_t *rgb_a;
  const float *depth_a;
  const uint8_t *rgb_b;
  const float *depth_b;
  uint8_t *y;
  uint8_t *u;
  uint8_t *v;
  size_t rgb_fb, depth_fb, y_fb, u_fb, v_fb;  // per-frame byte offsets
  int w, h, y_stride, u_stride, v_stride, mode;
  uint32_t strips, tiles, frames;  // tiles: per strip
  uint32_t run;                    // consecutive tiles per XCD
  VRows flt;
};

// Loads and stores at any byte alignment (gfx950 serves them in one
// instruction), so frame widths and addresses need no case of their own.
typedef uint32_t Word __attribute__((aligned(1)));
typedef uint16_t Half __attribute__((aligned(1)));
typedef uint32_t Word2 __attribute__((ext_vector_type(2), aligned(1)));
typedef float Depth4 __attribute__((ext_vector_type(4), aligned(1)));
typedef float Float __attribute__((aligned(1)));
struct Rgb4 { uint32_t w[3]; };  // four RGB24 pixels
struct RowIn {                   // one quad of a row of both inputs
  Rgb4 a, b;
  Depth4 da, db;
};

template <class T>
__device__ __forceinline__ T load_from(const uint8_t *p) {
  return *reinterpret_cast<const T *>(p);
}
// kStream: past the caches (non-temporal).
template <bool kStream, class T>
__device__ __forceinline__ void store_to(uint8_t *p, T v) {
  if (kStream)
    __builtin_nontemporal_store(v, reinterpret_cast<T *>(p));
  else
    *reinterpret_cast<T *>(p) = v;
}
__device__ __forceinline__ Rgb4 load_rgb4(const uint8_t *p) {
  const Word2 lo = load_from<Word2>(p);
  return Rgb4{{lo.x, lo.y, load_from<Word>(p + 8)}};
}

enum FrameClass {
  kPlain,
  kBulk,    // more data than the Infinity Cache holds
  kNarrow,  // width 2
};

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef short i16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t dot_u(uint32_t a, uint32_t c0, uint32_t c1, uint32_t acc) {
  const u16x2 c = {(unsigned short)c0, (unsigned short)c1};
  return __builtin_amdgcn_udot2(__builtin_bit_cast(u16x2, a), c, acc, false);
}
__device__ __forceinline__ int dot_i(uint32_t a, int c, int acc) {
  const i16x2 cc = {(short)c, (short)c};
  return __builtin_amdgcn_sdot2(__builtin_bit_cast(i16x2, a), cc, acc, false);
}
// Bytes i and j (0..3 of lo, 4..7 of hi) as the halves of a word.
template <int I, int J>
__device__ __forceinline__ uint32_t byte_pair(uint32_t hi, uint32_t lo) {
  return __builtin_amdgcn_perm(hi, lo, 0x0c000c00u | (J << 16) | I);
}

// Depth key order with NaN as +infinity; ties keep A.
__device__ __forceinline__ bool take_b(float da, float db) { return db < fminf(da, INFINITY); }

// Luma of two pixels whose components are the halves of r, g, b.  With
// Y14 = (8414 r + 16519 g + 3208 b + 524544) >> 9 (at most 15040, so neither
// 2 * Y14 nor the result reaches a clamp), (2 * Y14 + 64) >> 7 is the sum
// plus 16384 shifted by 15; the doubled sum has it in its third byte.
__device__ __forceinline__ void luma2(uint32_t r, uint32_t g, uint32_t b, uint32_t y[2]) {
  constexpr uint32_t kR = 2 * 8414, kG = 2 * 16519, kB = 2 * 3208, kC = 2 * (524544 + 16384);
  y[0] = dot_u(r, kR, 0, dot_u(g, kG, 0, dot_u(b, kB, 0, kC)));
  y[1] = dot_u(r, 0, kR, dot_u(g, 0, kG, dot_u(b, 0, kB, kC)));
}
// The 15-bit chroma 2 * (sum >> 10) of a pixel pair and of the next one, as
// the halves of a word (the sums are positive and at most 30720 after it: no
// clamp is reached).
__device__ __forceinline__ uint32_t chroma2(int s0, int s1) {
  const uint32_t lo = (uint32_t)s0 >> 9, hi = (uint32_t)s1 << 7;
  return ((lo & 0xffffu) | (hi & 0xffff0000u)) & 0xfffefffeu;
}
__device__ __forceinline__ int usum(uint32_t r, uint32_t g, uint32_t b) {
  return dot_i(r, -4865, dot_i(g, -9528, dot_i(b, 14392, 8389120)));
}
__device__ __forceinline__ int vsum(uint32_t r, uint32_t g, uint32_t b) {
  return dot_i(r, 14392, dot_i(g, -12061, dot_i(b, -2332, 8389120)));
}

// Frame widths under four: the row's two pixels byte by byte.
__device__ __forceinline__ Rgb4 load_two_pixels(const uint8_t *p) {
  Rgb4 q;
  q.w[0] = (uint32_t)p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16) | ((uint32_t)p[3] << 24);
  q.w[1] = (uint32_t)p[4] | ((uint32_t)p[5] << 8);
  q.w[2] = 0u;
  return q;
}

// One chroma row of a quad: (u0 u1, v0 v1) in bytes.  The x86 rows (all but
// the last) sum the high halves of the products, which no order of taps takes
// out of 16 bits.
template <bool kX86, class Rows>
__device__ __forceinline__ uint2 filter_row(Rows &&rows, const int16_t *cf, int taps) {
  const int init = kX86 ? (64 + 8 * (taps - 1)) >> 4 : 64 << 12;
  int s[4] = {init, init, init, init};  // u0, u1, v0, v1
#pragma unroll
  for (int j = 0; j < kVTaps; ++j) {
    const uint2 q = rows(j);
    const int t[4] = {(int)(q.x & 0xffffu), (int)(q.x >> 16), (int)(q.y & 0xffffu), (int)(q.y >> 16)};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int prod = __mul24((int)cf[j], t[i]);
      s[i] += kX86 ? prod >> 16 : prod;
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) s[i] = min(max(s[i] >> (kX86 ? 3 : 19), 0), 255);
  return make_uint2((uint32_t)(s[0] | (s[1] << 8)), (uint32_t)(s[2] | (s[3] << 8)));
}

template <FrameClass kClass>
struct PlaneRow {
  uint8_t *u, *v;
  __device__ __forceinline__ void store(const FrameprepArgs &a, int k, uint2 s) const {
    uint8_t *ur = u + (size_t)k * a.u_stride, *vr = v + (size_t)k * a.v_stride;
    if (kClass == kNarrow) {
      ur[0] = (uint8_t)s.x;
      vr[0] = (uint8_t)s.y;
    } else {
      store_to<kClass == kBulk, Half>(ur, (uint16_t)s.x);
      store_to<kClass == kBulk, Half>(vr, (uint16_t)s.y);
    }
  }
};

// Bound by HBM in bulk (256 720p pairs: 727 -> 706 us, 5.18 TB/s of inputs and
// outputs, what a device copy reaches) and by its own latency for one frame
// (720p pair with launch and wait: 24.4 -> 16.7 us, 11.1 of them an empty
// launch and wait).  What counted: the filter's rows as kernel arguments (no
// table in memory); byte pairs gathered by v_perm into 16-bit dot products (a
// third fewer instructions); wide loads at any alignment, so that widths of 4k
// + 2 need no per-pixel path (642x360 x 8: 37 -> 17 us); the next row's loads
// ahead of this row's arithmetic.  Tiles are dealt to the XCDs in runs of
// kFpRunRows tile rows, and neighbours meet at the rows they share (bulk: 716
// us with single tiles, 737 with one run per XCD).  Tiles of 32 and 64 chroma
// rows (less halo, 8 and 16 wavefronts) took 721 and 714 us, non-temporal
// loads 820.
template <bool kTwo, int kCRows, FrameClass kClass>
__global__ __launch_bounds__(64 * kFpWaves) void frameprep_kernel(FrameprepArgs a) {
  __shared__ uint2 uv[2 * kCRows + 6][kFpQuads];  // (u0 u1, v0 v1) of each quad
  __shared__ int16_t edge_coef[kVClasses * kVTaps];
  const uint32_t total = a.strips * a.tiles * a.frames;
  // runs of a.run tiles, dealt to the XCDs in turn
  const uint32_t block = blockIdx.y * kFpGridRow + blockIdx.x, turn = block / kFpXcds;
  const uint32_t id = (turn / a.run * kFpXcds + block % kFpXcds) * a.run + turn % a.run;
  if (id >= total) return;
  const uint32_t strip = id % a.strips, tile = id / a.strips % a.tiles, f = id / a.strips / a.tiles;
  const uint8_t *rgb_a = a.rgb_a + f * a.rgb_fb;
  const uint8_t *rgb_b = kTwo ? a.rgb_b + f * a.rgb_fb : nullptr;
  const uint8_t *dep_a = kTwo ? (const uint8_t *)a.depth_a + f * a.depth_fb : nullptr;
  const uint8_t *dep_b = kTwo ? (const uint8_t *)a.depth_b + f * a.depth_fb : nullptr;
  uint8_t *yp = a.y + f * a.y_fb, *up = a.u + f * a.u_fb, *vp = a.v + f * a.v_fb;

  const int ch = a.h >> 1;
  const int k0 = (int)tile * kCRows, k1 = min(k0 + kCRows, ch);
  const int lo = min(row_pos(a.flt, k0, ch), 2 * k0);
  const int hi = min(max(row_pos(a.flt, k1 - 1, ch) + a.flt.taps - 1, 2 * k1 - 1), a.h - 1);
  const int nrows = hi - lo + 1;
  const int lane = (int)(threadIdx.x & 63u);
  const int wave = (int)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // rows are wavefront-uniform
  const int quad = (int)strip * kFpQuads + lane;
  // the last quad of a width that is no multiple of 4 overlaps the one before
  // it (both compute the same values)
  constexpr bool narrow = kClass == kNarrow, stream = kClass == kBulk;
  const int x0 = narrow ? 0 : min(4 * quad, a.w - 4);
  const bool on = 4 * quad < a.w;

  const bool edge = k0 < 2 || k1 > ch - 2;
  if (edge && threadIdx.x < kVClasses * kVTaps)
    edge_coef[threadIdx.x] = reinterpret_cast<const int16_t *>(a.flt.coef)[threadIdx.x];

  // Phase 1: composite, luma out, chroma intermediates into LDS; one row per
  // wavefront and iteration.
  if (on) {
    auto fetch = [&](int rr) {
      const size_t at = (size_t)(lo + rr) * a.w + x0;
      RowIn in;
      if (narrow) {
        in.a = load_two_pixels(rgb_a + 3 * at);
        if (kTwo) {
          in.b = load_two_pixels(rgb_b + 3 * at);
          for (int i = 0; i < 2; ++i) {
            in.da[i] = load_from<Float>(dep_a + 4 * (at + i));
            in.db[i] = load_from<Float>(dep_b + 4 * (at + i));
          }
        }
      } else {
        in.a = load_rgb4(rgb_a + 3 * at);
        if (kTwo) {
          in.b = load_rgb4(rgb_b + 3 * at);
          in.da = load_from<Depth4>(dep_a + 4 * at);
          in.db = load_from<Depth4>(dep_b + 4 * at);
        }
      }
      return in;
    };
    // Every other tile goes from its last row up, so that two neighbours read
    // the rows they share at about the same time.  The next row's loads are in
    // flight while this one is converted.
    const int from = tile & 1 ? nrows - 1 : 0, dir = tile & 1 ? -1 : 1;
    RowIn next = fetch(from + dir * min(wave, nrows - 1));
    for (int it = wave; it < nrows; it += kFpWaves) {
      const RowIn in = next;
      next = fetch(from + dir * min(it + kFpWaves, nrows - 1));
      const int rr = from + dir * it, row = lo + rr;
      Rgb4 p = in.a;
      if (kTwo) {
        uint32_t m[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) m[i] = !narrow || i < 2 ? (take_b(in.da[i], in.db[i]) ? ~0u : 0u) : 0u;
        const uint32_t wm[3] = {(m[0] & 0x00ffffffu) | (m[1] & 0xff000000u),
                                (m[1] & 0x0000ffffu) | (m[2] & 0xffff0000u),
                                (m[2] & 0x000000ffu) | (m[3] & 0xffffff00u)};
#pragma unroll
        for (int i = 0; i < 3; ++i) p.w[i] = (in.b.w[i] & wm[i]) | (p.w[i] & ~wm[i]);
      }
      // [r0 g0 b0 r1] [g1 b1 r2 g2] [b2 r3 g3 b3]
      const uint32_t r01 = byte_pair<0, 3>(p.w[1], p.w[0]), g01 = byte_pair<1, 4>(p.w[1], p.w[0]),
                     b01 = byte_pair<2, 5>(p.w[1], p.w[0]);
      const uint32_t r23 = byte_pair<2, 5>(p.w[2], p.w[1]), g23 = byte_pair<3, 6>(p.w[2], p.w[1]),
                     b23 = byte_pair<0, 3>(0u, p.w[2]);
      if (row >= 2 * k0 && row < 2 * k1) {
        uint32_t y[4];
        luma2(r01, g01, b01, y);
        luma2(r23, g23, b23, y + 2);
        const uint32_t y01 = __builtin_amdgcn_perm(y[1], y[0], 0x0c0c0602u),
                       y23 = __builtin_amdgcn_perm(y[3], y[2], 0x06020c0cu);
        uint8_t *yr = yp + (size_t)row * a.y_stride + x0;
        if (narrow)
          store_to<stream, Half>(yr, (uint16_t)y01);
        else
          store_to<stream, Word>(yr, y01 | y23);
      }
      uv[rr][lane] = make_uint2(chroma2(usum(r01, g01, b01), usum(r23, g23, b23)),
                                chroma2(vsum(r01, g01, b01), vsum(r23, g23, b23)));
    }
  }
  __syncthreads();
  if (!on) return;

  // Phase 2: vertical chroma filter out of LDS, one chroma row per wavefront
  // and iteration, two samples of each plane per lane.  Tiles without the
  // frame's first or last two chroma rows have one filter row and start at a
  // fixed offset; in the x86 mode they hold no row of the other rounding.
  const PlaneRow<kClass> to{up + (x0 >> 1), vp + (x0 >> 1)};
  if (!edge) {
    for (int k = k0 + wave; k < k1; k += kFpWaves) {
      const uint2(*rows)[kFpQuads] = uv + 2 * (k - k0);
      if (a.mode == NES_SWS_X86)
        to.store(a, k, filter_row<true>([&](int j) { return rows[j][lane]; }, a.flt.coef[2], kVTaps));
      else
        to.store(a, k, filter_row<false>([&](int j) { return rows[j][lane]; }, a.flt.coef[2], kVTaps));
    }
  } else {
    for (int k = k0 + wave; k < k1; k += kFpWaves) {
      const int c = row_class(k, ch), p0 = row_pos(a.flt, k, ch) - lo;
      const int16_t *cf = &edge_coef[c * kVTaps];
      // taps past the filter's own have no weight: any row of the tile will do
      auto row = [&](int j) { return uv[min(p0 + j, nrows - 1)][lane]; };
      if (a.mode == NES_SWS_X86 && 2 * k < a.h - 2)
        to.store(a, k, filter_row<true>(row, cf, a.flt.taps));
      else
        to.store(a, k, filter_row<false>(row, cf, a.flt.taps));
    }
  }
}

static int frameprep_check(const uint8_t *rgb_a, const float *depth_a, const uint8_t *rgb_b,
                           const float *depth_b, int w, int h, int n_frames, const uint8_t *y,
                           int y_stride, const uint8_t *u, int u_stride, const uint8_t *v,
                           int v_stride, int sws_mode) {
  if (w < 2 || h < 2 || (w & 1) || (h & 1) || n_frames < 1 || !rgb_a || !y || !u || !v) {
    set_last_error("frame prep needs even w, h >= 2 and non-null buffers");
    return NES_EINVAL;
  }
  if ((rgb_b == nullptr) != (depth_b == nullptr) || (rgb_b && !depth_a)) {
    set_last_error("composite needs both depths");
    return NES_EINVAL;
  }
  if (y_stride < w || u_stride < w / 2 || v_stride < w / 2) return NES_EINVAL;
  if (sws_mode != NES_SWS_X86 && sws_mode != NES_SWS_C) return NES_EINVAL;
  if (n_frames > 65535) return NES_ERANGE;
  return NES_OK;
}

// Chroma rows per tile: tall tiles read less halo, but a small batch needs
// workgroups.  One 720p pair: 4 rows 16.2 us, 8 rows 16.5, 16 rows 18.1; 16
// of them: 48.9, 48.9, 50.8; 32: 101 us with any.
static int frameprep_rows(int w, int h, int n_frames) {
  const size_t strips = ((size_t)w + 255) / 256;
  auto blocks = [&](int rows) { return strips * (((size_t)h / 2 + rows - 1) / rows) * n_frames; };
  return blocks(16) >= 2048 ? 16 : blocks(8) >= 1024 ? 8 : 4;
}

// Inputs beyond this do not stay in the Infinity Cache (256 MB): their planes
// are stored past the caches (256 720p pairs: 763 -> 743 us).
constexpr size_t kBulkBytes = (size_t)256 << 20;

constexpr uint32_t kFpRunRows = 6;  // tile rows per run

template <int kCRows, FrameClass kClass>
static void frameprep_launch(FrameprepArgs &a, bool two, hipStream_t stream) {
  a.tiles = (uint32_t)((a.h / 2 + kCRows - 1) / kCRows);
  const uint32_t total = a.strips * a.tiles * a.frames;
  a.run = std::max(1u, std::min(a.strips * kFpRunRows, (total + kFpXcds - 1) / kFpXcds));
  const uint32_t turns = (total + a.run * kFpXcds - 1) / (a.run * kFpXcds);
  const uint32_t blocks = turns * a.run * kFpXcds;
  const dim3 grid(std::min(blocks, kFpGridRow), (blocks + kFpGridRow - 1) / kFpGridRow);
  if (two)
    frameprep_kernel<true, kCRows, kClass><<<grid, 64 * kFpWaves, 0, stream>>>(a);
  else
    frameprep_kernel<false, kCRows, kClass><<<grid, 64 * kFpWaves, 0, stream>>>(a);
}

int launch_frameprep(const uint8_t *rgb_a, const float *depth_a,
                     const uint8_t *rgb_b, const float *depth_b, int w, int h,
                     int n_frames, size_t rgb_fb, size_t depth_fb, uint8_t *y,
                     int y_stride, size_t y_fb, uint8_t *u, int u_stride,
                     size_t u_fb, uint8_t *v, int v_stride, size_t v_fb,
                     int sws_mode, hipStream_t stream) {
  NES_TRY(frameprep_check(rgb_a, depth_a, rgb_b, depth_b, w, h, n_frames, y, y_stride, u,
                          u_stride, v, v_stride, sws_mode));
  FrameprepArgs a;
  NES_TRY(get_vrows(h, &a.flt));
  a.rgb_a = rgb_a; a.depth_a = depth_a; a.rgb_b = rgb_b; a.depth_b = depth_b;
  a.y = y; a.u = u; a.v = v;
  a.rgb_fb = rgb_fb; a.depth_fb = depth_fb; a.y_fb = y_fb; a.u_fb = u_fb; a.v_fb = v_fb;
  a.w = w; a.h = h; a.y_stride = y_stride; a.u_stride = u_stride; a.v_stride = v_stride;
  a.mode = sws_mode;
  a.strips = (uint32_t)(((w + 3) / 4 + kFpQuads - 1) / kFpQuads);
  a.frames = (uint32_t)n_frames;
  const bool two = rgb_b != nullptr;
  const int rows = frameprep_rows(w, h, n_frames);
  if (w < 4)
    frameprep_launch<4, kNarrow>(a, two, stream);
  else if (rows == 4)
    frameprep_launch<4, kPlain>(a, two, stream);
  else if (rows == 8)
    frameprep_launch<8, kPlain>(a, two, stream);
  else if ((size_t)w * h * n_frames * (two ? 14 : 3) < kBulkBytes)
    frameprep_launch<16, kPlain>(a, two, stream);
  else
    frameprep_launch<16, kBulk>(a, two, stream);
  NES_HIP_TRY(hipGetLastError());
  return NES_OK;
}

// GRAY8 full range -> YUV420P limited range (the depth stream).  Luma:
// hScale8To15 (g << 7) then lumRangeFromJpeg_c; chroma planes of a gray
// source hold the constant 1 << 14 before the vertical filter.
// kDepth: the source is FP32 expected depth, quantised to the GRAY8 depth
// plane on the fly (depth_gray8, `scale` = 255 / far); that plane is also
// written to `gray_out` when it is not null.
// One 4-pixel quad per lane and row (the last one of a width that is no
// multiple of 4 overlaps its neighbour); the chroma of a row is one value,
// which depends on the row's filter taps alone (`chroma` per row_class).
struct GrayArgs {
  const uint8_t *g;
  const float *depth;
  uint8_t *y, *u, *v, *gray_out;
  int g_stride, w, h, y_stride, u_stride, v_stride;
  float scale;
  uint8_t chroma[kVClasses];
  uint8_t last_chroma;  // of the last chroma row
};

__device__ __forceinline__ uint32_t gray_luma(uint32_t g) {
  const int v15 = ((int)(g << 7) * 14071 + 33561947) >> 14;
  return (uint32_t)min(max((v15 + 64) >> 7, 0), 255);
}

template <bool kDepth>
__global__ __launch_bounds__(256) void gray_kernel(GrayArgs a) {
  const int quad = (int)(blockIdx.x * 64 + (threadIdx.x & 63u)), row = (int)(blockIdx.y * 4 + (threadIdx.x >> 6));
  if (row >= a.h || 4 * quad >= a.w) return;
  const int x0 = max(min(4 * quad, a.w - 4), 0), n = min(4, a.w);
  uint32_t g = 0;  // four GRAY8 values
  if (n == 4) {
    if (kDepth) {
      const Depth4 d = *reinterpret_cast<const Depth4 *>(a.depth + (size_t)row * a.w + x0);
#pragma unroll
      for (int i = 0; i < 4; ++i) g |= (uint32_t)depth_gray8(d[i], a.scale) << (8 * i);
    } else {
      g = load_from<Word>(a.g + (size_t)row * a.g_stride + x0);
    }
  } else {
    for (int i = 0; i < n; ++i)
      g |= (uint32_t)(kDepth ? depth_gray8(a.depth[(size_t)row * a.w + i], a.scale)
                             : a.g[(size_t)row * a.g_stride + i]) << (8 * i);
  }
  uint32_t y = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) y |= gray_luma((g >> (8 * i)) & 0xffu) << (8 * i);
  uint8_t *yr = a.y + (size_t)row * a.y_stride + x0;
  uint8_t *gr = kDepth && a.gray_out ? a.gray_out + (size_t)row * a.w + x0 : nullptr;
  const int k = row >> 1, ch = a.h >> 1;
  const int c = row_class(k, ch);
  const uint32_t uv = k == ch - 1 ? a.last_chroma
                      : c == 0 ? a.chroma[0] : c == 1 ? a.chroma[1] : c == 2 ? a.chroma[2] : a.chroma[3];
  if (n == 4) {
    store_to<false, Word>(yr, y);
    if (gr) store_to<false, Word>(gr, g);
    if (row & 1) return;
    store_to<false, Half>(a.u + (size_t)k * a.u_stride + (x0 >> 1), (uint16_t)(uv * 0x101u));
    store_to<false, Half>(a.v + (size_t)k * a.v_stride + (x0 >> 1), (uint16_t)(uv * 0x101u));
  } else {
    for (int i = 0; i < n; ++i) {
      yr[i] = (uint8_t)(y >> (8 * i));
      if (gr) gr[i] = (uint8_t)(g >> (8 * i));
    }
    if (row & 1) return;
    a.u[(size_t)k * a.u_stride] = (uint8_t)uv;
    a.v[(size_t)k * a.v_stride] = (uint8_t)uv;
  }
}

// The chroma of a gray source: its planes hold 1 << 14 before the vertical
// filter, so a row's value is a sum over its taps.
static uint8_t gray_chroma(const VRows &f, int c, bool x86) {
  int s = x86 ? (64 + 8 * (f.taps - 1)) >> 4 : 64 << 12;
  for (int j = 0; j < f.taps; ++j) s += x86 ? ((int)f.coef[c][j] << 14) >> 16 : (int)f.coef[c][j] << 14;
  return (uint8_t)std::min(std::max(s >> (x86 ? 3 : 19), 0), 255);
}

static int launch_gray(GrayArgs &a, bool depth, int sws_mode, hipStream_t stream) {
  VRows f;
  NES_TRY(get_vrows(a.h, &f));
  // every chroma row but the last takes the x86 path in that mode
  for (int c = 0; c < kVClasses; ++c) a.chroma[c] = gray_chroma(f, c, sws_mode == NES_SWS_X86);
  a.last_chroma = gray_chroma(f, row_class(a.h / 2 - 1, a.h / 2), false);
  const dim3 grid((unsigned)((a.w + 255) / 256), (unsigned)((a.h + 3) / 4));
  if (depth)
    gray_kernel<true><<<grid, 256, 0, stream>>>(a);
  else
    gray_kernel<false><<<grid, 256, 0, stream>>>(a);
  NES_HIP_TRY(hipGetLastError());
  return NES_OK;
}

int launch_depth_yuv(const float *depth, int w, int h, float scale, uint8_t *gray, uint8_t *y,
                     int y_stride, uint8_t *u, int u_stride, uint8_t *v, int v_stride,
                     int sws_mode, hipStream_t stream) {
  if (!depth || !y || !u || !v || w < 2 || h < 2 || (w & 1) || (h & 1)) return NES_EINVAL;
  if (y_stride < w || u_stride < w / 2 || v_stride < w / 2) return NES_EINVAL;
  if (sws_mode != NES_SWS_X86 && sws_mode != NES_SWS_C) return NES_EINVAL;
  GrayArgs a{};
  a.depth = depth; a.scale = scale; a.gray_out = gray;
  a.y = y; a.u = u; a.v = v;
  a.w = w; a.h = h; a.y_stride = y_stride; a.u_stride = u_stride; a.v_stride = v_stride;
  return launch_gray(a, true, sws_mode, stream);
}

namespace {
std::mutex g_host_mu;
DevBuf g_in, g_out;
}  // namespace

// nes_frameprep_device_static's documented height limit.
constexpr int kStaticMaxHeight = 8192;

}  // namespace nes

using namespace nes;

extern "C" {

int nes_frameprep(const uint8_t *rgb_a, const float *depth_a,
                  const uint8_t *rgb_b, const float *depth_b, int w, int h,
                  int rgb_stride, uint8_t *y, int y_stride, uint8_t *u,
                  int u_stride, uint8_t *v, int v_stride, int sws_mode) {
  if (!rgb_a || !y || !u || !v || w < 2 || h < 2 || (w & 1) || (h & 1)) return NES_EINVAL;
  if (rgb_stride < 3 * w || y_stride < w || u_stride < w / 2 || v_stride < w / 2) return NES_EINVAL;
  if ((rgb_b == nullptr) != (depth_b == nullptr) || (rgb_b && !depth_a)) return NES_EINVAL;
  NES_TRY(ensure_device());
  std::lock_guard<std::mutex> lk(g_host_mu);
  const size_t px = (size_t)w * h;
  const size_t rgb_bytes = 3 * px, dep_bytes = 4 * px;
  const size_t in_bytes = rgb_b ? 2 * rgb_bytes + 2 * dep_bytes + 64 : rgb_bytes + 64;
  const size_t cw = (size_t)w / 2, chh = (size_t)h / 2;
  const size_t out_bytes = px + 2 * cw * chh + 64;
  NES_TRY(g_in.reserve(in_bytes));
  NES_TRY(g_out.reserve(out_bytes));
  hipStream_t s = library_stream();
  uint8_t *d_rgb_a = g_in.as<uint8_t>();
  // depth buffers are placed 16-byte aligned after the colour planes
  size_t off_rgb_b = (rgb_bytes + 15) & ~size_t(15);
  size_t off_da = (off_rgb_b + rgb_bytes + 15) & ~size_t(15);
  size_t off_db = off_da + dep_bytes;
  uint8_t *d_rgb_b = rgb_b ? d_rgb_a + off_rgb_b : nullptr;
  float *d_da = rgb_b ? (float *)(d_rgb_a + off_da) : nullptr;
  float *d_db = rgb_b ? (float *)(d_rgb_a + off_db) : nullptr;
  NES_HIP_TRY(hipMemcpy2DAsync(d_rgb_a, 3 * w, rgb_a, rgb_stride, 3 * w, h,
                               hipMemcpyHostToDevice, s));
  if (rgb_b) {
    NES_HIP_TRY(hipMemcpy2DAsync(d_rgb_b, 3 * w, rgb_b, rgb_stride, 3 * w, h,
                                 hipMemcpyHostToDevice, s));
    NES_HIP_TRY(hipMemcpyAsync(d_da, depth_a, dep_bytes, hipMemcpyHostToDevice, s));
    NES_HIP_TRY(hipMemcpyAsync(d_db, depth_b, dep_bytes, hipMemcpyHostToDevice, s));
  }
  uint8_t *d_y = g_out.as<uint8_t>();
  uint8_t *d_u = d_y + px;
  uint8_t *d_v = d_u + cw * chh;
  NES_TRY(launch_frameprep(d_rgb_a, d_da, d_rgb_b, d_db, w, h, 1, 0, 0, d_y, w, 0,
                           d_u, (int)cw, 0, d_v, (int)cw, 0, sws_mode, s));
  NES_HIP_TRY(hipMemcpy2DAsync(y, y_stride, d_y, w, w, h, hipMemcpyDeviceToHost, s));
  NES_HIP_TRY(hipMemcpy2DAsync(u, u_stride, d_u, cw, cw, chh, hipMemcpyDeviceToHost, s));
  NES_HIP_TRY(hipMemcpy2DAsync(v, v_stride, d_v, cw, cw, chh, hipMemcpyDeviceToHost, s));
  NES_HIP_TRY(hipStreamSynchronize(s));
  return NES_OK;
}

int nes_frameprep_device(const uint8_t *rgb_a, const float *depth_a,
                         const uint8_t *rgb_b, const float *depth_b, int w,
                         int h, int n_frames, uint8_t *y, int y_stride,
                         uint8_t *u, int u_stride, uint8_t *v, int v_stride,
                         int sws_mode, float *elapsed_ms) {
  NES_TRY(ensure_device());
  hipStream_t s = library_stream();
  const size_t px = (size_t)w * h;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (elapsed_ms) {
    NES_HIP_TRY(hipEventCreate(&e0));
    NES_HIP_TRY(hipEventCreate(&e1));
    NES_HIP_TRY(hipEventRecord(e0, s));
  }
  int rc = launch_frameprep(rgb_a, depth_a, rgb_b, depth_b, w, h, n_frames, 3 * px,
                            4 * px, y, y_stride, (size_t)y_stride * h, u, u_stride,
                            (size_t)u_stride * (h / 2), v, v_stride,
                            (size_t)v_stride * (h / 2), sws_mode, s);
  if (elapsed_ms) {
    hipEventRecord(e1, s);
    hipEventSynchronize(e1);
    hipEventElapsedTime(elapsed_ms, e0, e1);
    hipEventDestroy(e0);
    hipEventDestroy(e1);
  }
  if (rc != NES_OK) return rc;
  NES_HIP_TRY(hipStreamSynchronize(s));
  return NES_OK;
}

int nes_frameprep_device_static(const uint8_t *rgb_a, const float *depth_a,
                                const uint8_t *rgb_b, const float *depth_b, int w, int h,
                                int n_frames, uint8_t *y, int y_stride, uint8_t *u,
                                int u_stride, uint8_t *v, int v_stride, int sws_mode,
                                void *stream) {
  NES_TRY(ensure_device());
  NES_TRY(frameprep_check(rgb_a, depth_a, rgb_b, depth_b, w, h, n_frames, y, y_stride, u,
                          u_stride, v, v_stride, sws_mode));
  if (h > kStaticMaxHeight) {
    set_last_error("nes_frameprep_device_static: frame height above 8192");
    return NES_ERANGE;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const size_t px = (size_t)w * h;
  NES_TRY(launch_frameprep(rgb_a, depth_a, rgb_b, depth_b, w, h, n_frames, 3 * px, 4 * px, y, y_stride,
                           (size_t)y_stride * h, u, u_stride, (size_t)u_stride * (h / 2), v, v_stride,
                           (size_t)v_stride * (h / 2), sws_mode, s));
  if (!stream) NES_HIP_TRY(hipStreamSynchronize(s));
  return NES_OK;
}

int nes_gray8_to_yuv420p(const uint8_t *gray, int w, int h, int g_stride,
                         uint8_t *y, int y_stride, uint8_t *u, int u_stride,
                         uint8_t *v, int v_stride, int sws_mode) {
  if (!gray || !y || !u || !v || w < 2 || h < 2 || (w & 1) || (h & 1)) return NES_EINVAL;
  if (g_stride < w || y_stride < w || u_stride < w / 2 || v_stride < w / 2) return NES_EINVAL;
  if (sws_mode != NES_SWS_X86 && sws_mode != NES_SWS_C) return NES_EINVAL;
  NES_TRY(ensure_device());
  std::lock_guard<std::mutex> lk(g_host_mu);
  const size_t px = (size_t)w * h, cw = (size_t)w / 2, chh = (size_t)h / 2;
  NES_TRY(g_in.reserve(px));
  NES_TRY(g_out.reserve(px + 2 * cw * chh));
  hipStream_t s = library_stream();
  uint8_t *d_g = g_in.as<uint8_t>();
  uint8_t *d_y = g_out.as<uint8_t>(), *d_u = d_y + px, *d_v = d_u + cw * chh;
  NES_HIP_TRY(hipMemcpy2DAsync(d_g, w, gray, g_stride, w, h, hipMemcpyHostToDevice, s));
  GrayArgs ga{};
  ga.g = d_g; ga.g_stride = w;
  ga.y = d_y; ga.u = d_u; ga.v = d_v;
  ga.w = w; ga.h = h; ga.y_stride = w; ga.u_stride = ga.v_stride = (int)cw;
  NES_TRY(launch_gray(ga, false, sws_mode, s));
  NES_HIP_TRY(hipMemcpy2DAsync(y, y_stride, d_y, w, w, h, hipMemcpyDeviceToHost, s));
  NES_HIP_TRY(hipMemcpy2DAsync(u, u_stride, d_u, cw, cw, chh, hipMemcpyDeviceToHost, s));
  NES_HIP_TRY(hipMemcpy2DAsync(v, v_stride, d_v, cw, cw, chh, hipMemcpyDeviceToHost, s));
  NES_HIP_TRY(hipStreamSynchronize(s));
  return NES_OK;
}

// Host-side view of the vertical chroma filter (for inspection and tests).
int nes_sws_vchroma_filter(int h, int16_t *coef, int32_t *pos, int max_taps,
                           int *taps) {
  if (h < 2 || !coef || !pos || !taps) return NES_EINVAL;
  VFilter f = build_vchroma_filter(h);
  if (f.taps > max_taps) return NES_ERANGE;
  std::memcpy(coef, f.coef.data(), f.coef.size() * sizeof(int16_t));
  std::memcpy(pos, f.pos.data(), f.pos.size() * sizeof(int32_t));
  *taps = f.taps;
  return NES_OK;
}

}  // extern "C"
