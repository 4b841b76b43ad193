// render.h -- device data structures of the render pipeline and the context.
#pragma once

#include <memory>

#include "nes_internal.h"

namespace nes {

// One camera of a render batch.  Ray slots of a view are 8x8 pixel tiles laid
// out tile-major so that a wavefront's 64 rays are a compact screen block.
struct ViewDesc {
  float c2w[12];
  float focal, inv_focal;
  uint32_t width, height, tiles_x;
  uint32_t slot_base, slot_count;  // global ray-slot range of the view
  uint32_t px_base;                // offset of the view in the output arrays
  // Bound on how far a pixel's unnormalised direction lies from its tile
  // centre's (march_emit's tile test).
  float tile_reach;
};

struct RayData {  // 32 bytes
  float o[3];
  float d[3];
  float t_start;
  uint32_t n_steps;  // candidate steps inside the box (0 = miss / no pixel)
};

struct RayAcc {  // 32 bytes, compositing state carried across passes
  float T, r, g, b, depth;
  uint32_t n_samples;
  uint32_t done;
  uint32_t pad;
};  // written for rays that have samples only

// Sample record: ray slot in the high 25 bits, step index in the low 7.
constexpr uint32_t kMaxSlots = 1u << 25;
// View descriptors the pinned upload staging holds before it grows.
constexpr uint32_t kPinnedViews = 64;

// Per ray slot, the march writes counts[slot]: samples emitted by the pass in
// the low 8 bits (at most kMaxSteps), the flags of earlier passes, and the step
// the next pass resumes at in the high 16 bits.  The composite of a pass that
// is not the last adds kRayState for rays whose RayAcc it stored and kRayDone
// for those that reached T < 1e-4.
// offsets[wavefront] is the start of the wavefront's sample range.
constexpr uint32_t kCountMask = 0xffu, kRayState = 0x100u, kRayDone = 0x200u;
static_assert(kMaxSteps <= (int)kCountMask, "a ray's samples fit its count");

// Words of RenderWork::total (device) and RenderWork::total_host (pinned),
// the same layout on both sides:
//   [0] sample cursor of the first pass, [1] sample cursor of a later pass
//   (0 in a single-pass frame), [2] samples evaluated by all passes of the
//   frame (added once per pass), then from word kTotTermBase kTotTermSlots
//   copies of the termination counters, one 128-byte line each (a wavefront
//   adds to copy wave % slots, and only when one of its rays reached
//   T < 1e-4 in the pass): [+0] rays that reached T < 1e-4, [+1] samples
//   those rays composited, [+2] samples evaluated behind that point, [+3]
//   rays that stopped before the last pass with steps left.
// Words 4.. hold 64-bit device clock stamps (100 MHz): kStampBegin and
// kStampEnd of the frame, and per pass (the last pass written for passes
// beyond two) the starts of its march, encode, MLP and composite.
// frame_begin clears every word on the device and frame_end stores them all
// into the host copy.
constexpr int kTotCursor = 0, kTotCursorLater = 1, kTotEvaluated = 2, kTotStamps = 4, kTotTermBase = 32,
              kTotTermSlots = 32, kTotTermStride = 32;
constexpr int kStampBegin = 0, kStampEnd = 1, kStampPass = 2, kStampPasses = 2, kStampStages = 4;
static_assert(kTotStamps + 2 * (kStampPass + kStampPasses * kStampStages) <= kTotTermBase, "stamps");
constexpr int kTotWords = kTotTermBase + kTotTermSlots * kTotTermStride;
constexpr size_t kTotBytes = sizeof(uint32_t) * kTotWords;

// One output array on its way to pinned host memory: src (device, 16-byte
// aligned) to dst, `bytes` long, bpp bytes per pixel of view `view`.  The array
// of one byte per pixel is the GRAY8 plane, whose source is FP32 depth times
// gray_scale.
struct HostArray {
  const uint8_t *src;
  uint8_t *dst;
  uint64_t bytes;
  uint32_t bpp, view;
  uint32_t head;  // bytes in front of dst's first multiple of 16
  float gray_scale;
};
constexpr uint32_t kHostArrays = 40;  // carried to the device as kernel arguments

inline size_t wavefronts(size_t slots) { return (slots + 63) / 64; }

// Views start on this pixel in the output arrays, so that every array of every
// view starts on 16 bytes.
constexpr size_t kViewAlign = 64;

struct RenderWork {
  DevBuf views, rays, acc, counts, offsets, samples, sample_out, sample_pos, feat, out, total;
  DevBuf ray_sh;                  // mixed path: per ray slot 16 FP16 SH values
  DevBuf t_start;                 // per ray slot that has samples: t_start
  DevBuf gray;                    // GRAY8 depth staging of nes_render_fetch
  DevBuf tile_n;                  // per wavefront of ray slots: samples of the first pass
  DevBuf host_arrays;             // device copy of host_out
  HostArray host_out[kHostArrays];  // outputs the frame stores into host memory itself
  uint32_t n_host_out = 0;
  // whether pixels without samples are stored while the encode runs
  bool store_background = false;
  uint32_t *total_host = nullptr;  // pinned
  uint32_t n_views = 0, n_slots = 0;
  uint32_t capacity = 0;          // samples the sample buffers hold
  int capacity_precision = -1;    // feature layout the buffers were sized for
  size_t out_px = 0;              // pixels of the output arrays (each view starts on kViewAlign)
  size_t pixels = 0;              // pixels of the views
  std::vector<ViewDesc> host_views;
  // Pinned staging of the view descriptors: an upload from pageable memory
  // can block the host until the stream reaches it.  ev_views marks the
  // last upload, so the staging is rewritten only after it has been read.
  ViewDesc *views_pinned = nullptr;
  uint32_t views_pinned_cap = 0;
  hipEvent_t ev_views = nullptr;
  uint64_t budget = 0;            // device bytes the buffers may hold, 0 = no limit
  // Early termination learned from the previous frame of this work area:
  // samples the first pass gives each ray (kMaxSteps = one single pass).
  uint32_t first_pass_cap = kMaxSteps;
  uint32_t frame_passes = 1;      // passes the last frame launched
  bool whole_frame = false;       // its first pass walked all steps without a capacity's limit
  // Samples of the work area's last whole frame, first and later pass (0: none
  // yet): sizes the launches of the next one, whose own count stays on the device.
  uint32_t last_total[2] = {0, 0};
};

// What one frame evaluated and composited (for early-termination stats).
struct FrameCounts {
  uint64_t evaluated = 0, composited = 0, terminated = 0, term_samples = 0, wasted = 0,
           saved_rays = 0;
  uint32_t passes = 1;
};

// Device bytes currently held by a RenderWork's buffers.
size_t work_device_bytes(const RenderWork &w);
// Reserve every buffer a render of up to max_slots ray slots, max_px pixels
// and max_views views needs (with the initial four samples per ray slot),
// so that such renders allocate nothing.
int render_work_reserve(RenderWork &w, uint64_t max_slots, uint64_t max_px, uint32_t max_views,
                        int precision);

struct SceneDev {
  float *table_f32 = nullptr;      // entries x 2
  _Float16 *table_f16 = nullptr;   // entries x 2
  float *weights_f32 = nullptr;    // 9344
  _Float16 *wfrag = nullptr;       // 20 MFMA A-fragments x 64 lanes x 8
  uint32_t *occ = nullptr;         // 65536
};

int scene_upload(SceneDev &s, const nes_scene_desc *desc);
void scene_free(SceneDev &s);
// An empty scene copy whose device memory is freed with the last reference.
std::shared_ptr<SceneDev> new_scene();
// Permute the MLP weights into the A-operand fragments of the 20
// v_mfma_f32_16x16x32_f16 instructions one 16-sample tile uses.
void build_mlp_fragments(const float *w, _Float16 *frag);

// Byte offsets of the per-pixel outputs inside RenderWork::out.
struct OutLayout {
  size_t rgb24, depth, rgbf, nsamp, total;
};
OutLayout out_layout(size_t px);

// Stages of one render:
//   render_setup            views -> ray-slot layout, ray buffers, view upload
//   render_prepare_capacity sample buffers for the expected sample count
//   render_begin            counters cleared, views uploaded
//   render_launch_pass      march_emit, encode, MLP, composite for march steps
//                           [k0, k1)
//   render_end              counters and outputs stored on the host's side.  A
//                           pass's total above work.capacity means the pass was
//                           dropped: grow with render_reserve_samples and
//                           launch it again.
int render_setup(RenderWork &w, const nes_camera *views, int n_views, hipStream_t stream);
int render_prepare_capacity(RenderWork &w, int precision);
int render_reserve_samples(RenderWork &w, int precision, size_t capacity);
// Clears the frame counters and uploads the view descriptors of render_setup;
// precedes the first pass of a frame.
int render_begin(RenderWork &w, hipStream_t stream);
// Stores the frame counters and stamps into total_host and the outputs of
// host_out into theirs; follows the last pass (or any pass whose counters the
// host reads).
int render_end(RenderWork &w, hipStream_t stream);
// Has the frame of render_setup store the requested outputs into the caller's
// memory, if all of it is pinned; n_host_out stays 0 otherwise.
void plan_host_outputs(RenderWork &w, const nes_view_out *outs);
// One pass: march steps [k0, k1) (or, with resume, from where the ray's
// previous pass stopped), at most `cap` samples per ray, then encode, MLPs
// and composite.
int render_launch_pass(const SceneDev &scene, RenderWork &w, int precision, int k0, int k1,
                       bool first, bool last, hipStream_t stream, uint32_t cap = kMaxSteps,
                       bool resume = false);
// A whole frame without a host round trip: one pass when the work area's
// previous frame composited (almost) every sample it evaluated, else two:
// the first gives each ray at most first_pass_cap samples, the second
// continues the rays still above T = 1e-4 with all their remaining samples.
// The pass totals and composite counters land in total_host (read them after
// the stream has passed the launches).  Results are bit-identical to a single
// pass.
int render_launch_frame(const SceneDev &scene, RenderWork &w, int precision, hipStream_t stream);
// After the frame's stream work is complete: the largest pass total (a value
// above w.capacity means the frame must be launched again after growth) and
// the counts; updates first_pass_cap for the next frame.
uint32_t render_frame_max_total(const RenderWork &w);
FrameCounts render_frame_finish(RenderWork &w);
// Device time between the frame's begin and end stamps in total_host.
double frame_ms(const RenderWork &w);
// Device bytes the sample buffers of `capacity` samples take (all buffers
// that grow with the sample count).
size_t sample_buffer_bytes(size_t capacity, int precision);
// Whether growing the sample buffers to `capacity` keeps the work area
// within its budget.
bool render_growth_fits(const RenderWork &w, int precision, size_t capacity);
// A frame within the current sample buffers, whatever the scene: passes that
// give each ray at most capacity / rays samples, each resuming where the
// previous one stopped (bit-identical to one pass; no overflow possible).
int render_launch_bounded(const SceneDev &scene, RenderWork &w, int precision, hipStream_t stream);

// Workgroups per XCD part of the encode for about `samples` samples: one
// sample per thread (the kernel strides over the grid where there are more).
// Measured on the stereo 1080p frame: 512 workgroups per part 2.59 ms, 32768
// (about one sample per thread) 2.20 ms.  An empty workgroup costs 0.2 ns of
// dispatch (393216 of them 83 us, 32768 7 us), so the grid follows the
// expected samples and not the capacity of the buffers.
constexpr uint32_t kMaxPartBlocks = 49152;
inline uint32_t part_blocks(size_t samples) {
  const size_t b = (samples + 255) / 256;
  return (uint32_t)(b < 16 ? 16 : b > kMaxPartBlocks ? kMaxPartBlocks : b);
}

// Single-stage launchers (training step): march_emit over prepared rays,
// FP32 encode_parts, composite (which stores the final state of rays that have
// samples in work.acc for the backward; ray slot i is output i).
int launch_march_emit(const uint32_t *occ, RenderWork &w, int k0, int k1, hipStream_t stream);
// (n: the host's sample count, for the launch size; scattered: rays in no order.)
int launch_encode_f32(const float *table, RenderWork &w, uint32_t n, bool scattered, hipStream_t stream);
int launch_mlp_f32(const float *weights, RenderWork &w, const uint32_t *n_ptr, hipStream_t stream,
                   uint64_t *stamp = nullptr);
int launch_composite(RenderWork &w, hipStream_t stream);

// Enqueue a full render of views on stream; returns after the sample count
// read-backs (one host sync per pass).  Outputs land in work.out.
// With outs, the requested outputs are in the caller's memory on return if
// *delivered is set (render_fetch gets them otherwise).
int render_enqueue(const SceneDev &scene, RenderWork &work, int precision,
                   const nes_camera *views, int n_views, int steps_per_pass,
                   hipStream_t stream, nes_render_stats *stats,
                   const nes_view_out *outs = nullptr, bool *delivered = nullptr);
int render_fetch(RenderWork &work, int view, const nes_view_out *out,
                 hipStream_t stream);
void render_work_free(RenderWork &w);

// Text overlay: one drawn glyph of one string on one RGB24 frame.
struct GlyphPlacement {  // 32 bytes
  uint64_t base;         // byte offset of the frame in the RGB24 buffer
  int32_t x0, y0;        // top-left corner of the glyph bitmap
  int32_t w, h, stride;  // frame size and RGB24 row pitch in bytes
  uint32_t glyph;
};
// Placements of the strings process_frame_thread draws on the frame of cam
// (its width and height are the frame's); timestamp NULL = local time now.
void overlay_frame_layout(const nes_font *font, const nes_camera &cam, const char *timestamp,
                          uint32_t flags, int stride, uint64_t base,
                          std::vector<GlyphPlacement> &out);
// Upload the placements through `staging` and stamp them on `rgb`; `place`
// stays alive and `staging` untouched until the stream has passed the launch.
int overlay_launch(const nes_font *font, DevBuf &staging,
                   const std::vector<GlyphPlacement> &place, uint8_t *rgb, hipStream_t stream);
std::string overlay_now_text();

}  // namespace nes

struct nes_ctx {
  // The scene renders read.  nes_ctx_update_scene uploads into another copy
  // and swaps the pointer between renders; a render or server batch holds a
  // reference to the copy it started with until its device work is complete,
  // so no frame mixes two scenes.  `spare` is the previous copy, reused by
  // the next update once nothing holds it.
  std::shared_ptr<nes::SceneDev> scene, spare;
  std::mutex scene_mu;  // guards scene / spare
  nes::RenderWork work;
  hipStream_t stream = nullptr;
  uint64_t budget = 0;
  std::mutex mu;  // serialises the context's own renders (work, stream)
};

namespace nes {
// The context's current scene (a reference that keeps it alive).
std::shared_ptr<SceneDev> ctx_scene(nes_ctx *ctx);
}  // namespace nes
