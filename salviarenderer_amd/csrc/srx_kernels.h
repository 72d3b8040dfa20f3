// Host-side launchers of the pipeline kernels: geometry, binning, clears and resolves (srx_kernels.hip), in-order
// rasterisation under queries and with SASL shaders and deferred shading (srx_raster.hip), in-order
// rasterisation otherwise (srx_inorder.hip), visibility (srx_vis.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "srx_device.h"
#include "srx_record_rules.h"

namespace srx {


// Device statistics slots (pipeline_statistics / internal_statistics, async_object.h:90-175)
enum stat_slot {
  ST_IA_VERTICES = 0, ST_IA_PRIMITIVES, ST_VS_INVOCATIONS, ST_CINVOCATIONS, ST_CPRIMITIVES,
  ST_PS_INVOCATIONS, ST_BACKEND_PIXELS, ST_COUNT
};
// Setup counters
// CT_TOTAL: records emitted (single draws); CT_WIDE: primitives on wide_list, left to the clip launch.
// The two are added to as one 64-bit word.  CT_OVERRUN: the clip launch's additions carried CT_TOTAL past 32
// bits (setup alone cannot: at most four records a primitive, whose buffers take over 600 bytes); read the
// count with record_total.
// CT_CURSOR: records given to the tiles' lists; CT_PARTS, CT_MERGES: parts of split tiles and split tiles;
// CT_CLASS: GPU tiles per record-count class (the last class: without records); CT_STEP: per vis_step.
constexpr int TILE_CLASSES = 16;
enum counter_slot { CT_TOTAL = 0, CT_WIDE, CT_CLIP_PRIMS, CT_CLIP_SLOTS, CT_CLIP_OVERFLOW, CT_CURSOR, CT_PARTS, CT_MERGES,
                    CT_OVERRUN, CT_CLASS,
                    CT_STEP = CT_CLASS + TILE_CLASSES,
                    CT_COUNT = CT_STEP + VIS_STEPS };
// Records of a single draw, 0xFFFFFFFF when the count does not fit (above every capacity).
__host__ __device__ inline uint32_t record_total(const uint32_t* counters) {
  return counters[CT_OVERRUN] ? 0xFFFFFFFFu : counters[CT_TOTAL];
}
// GPU tiles with records, of T (once the ranges' launch has run).
__host__ __device__ inline uint32_t busy_tiles(const uint32_t* counters, uint32_t T) {
  return T - counters[CT_CLASS + TILE_CLASSES - 1];
}
static_assert(CT_TOTAL % 2 == 0 && CT_WIDE == CT_TOTAL + 1, "one aligned 64-bit word");

// Where a tile's record count lies in tile_count: atomics to words of one cache line are served one after
// another (330k of them on 1,024 adjacent words take 95 us, on words spread over 32 KB 14 us), and
// neighbouring tiles are counted at the same time, so they lie at least 64 bytes apart.
constexpr uint32_t TILE_SLOT_ROWS = 512;
__host__ __device__ inline uint32_t tile_slot_shift(uint32_t T) {  // log2 of the words per row
  uint32_t w = 4;
  while ((TILE_SLOT_ROWS << w) < T) ++w;
  return w;
}
__host__ __device__ inline uint32_t tile_slot(uint32_t t, uint32_t shift) {
  return ((t % TILE_SLOT_ROWS) << shift) + t / TILE_SLOT_ROWS;
}
__host__ __device__ inline uint32_t slot_tile(uint32_t s, uint32_t shift) {
  return (s & ((1u << shift) - 1u)) * TILE_SLOT_ROWS + (s >> shift);
}
__host__ __device__ inline uint32_t tile_slots(uint32_t T) {
  return (T < TILE_SLOT_ROWS ? T : TILE_SLOT_ROWS) << tile_slot_shift(T);
}

// What the host needs to know of a single draw, written by the device into pinned host memory: seq last.
struct draw_mail {
  uint32_t seq, total, merges, clip_overflow;
};

// Per-draw device buffers (owned by the renderer, grown on demand).
struct draw_buffers {
  float4* vbuf;        // (nverts+1) * (nattr+1) clip-space vertex-shader outputs
  float4* tri_rec;     // 3*prims * 5: edges, bbox, depth plane of each clipped triangle
  float4* tri_attr;    // 3*prims * 3*(nattr+1): v0, ddx, ddy of every register
  uint32_t* vis;       // target w*h*samples: winning triangle per sample (opaque early-Z draws)
  const ps_samplers* samplers;  // device copy of the bound samplers
  uint32_t* cnt;       // batches, 3*prims: GPU-tile records per clipped triangle, then their exclusive scan
  uint8_t* clip_flag;  // prims
  int32_t* clip_slot;  // prims
  float4* clip_verts;  // clip_capacity * 5 * (nattr+1), screen space
  uint32_t* clip_hdr;  // clip_capacity
  uint32_t clip_capacity;
  uint32_t* wide_list; // prims: triangles whose records the clip launch emits (batches: counts)
  uint32_t* keys[2];   // [0] records: GPU tile id; [1] single draws: the record's rank in its tile
  uint32_t* vals[2];   // records: triangle id << 1 | tile-level accept; [0] as emitted, [1] by tile
                       // (single draws that need primitive order: sorted back into [0])
  uint32_t list_cap;      // records the tiles' lists are formed for; with more the raster passes return at once
  const uint32_t* order;  // workgroup launch order of the GPU tiles, heaviest record-count class first
  // With vis_split, tiles of more than vis_part() records are split into parts, each a workgroup of the pass whose
  // per-sample keys a second launch merges: parts (tile, part, parts, 0) at their slot of vis_partial,
  // and (tile, parts, first slot, 0) per split tile (vis_split_bounds)
  uint4* vis_parts;
  uint4* vis_merges;
  unsigned long long* vis_partial;  // the parts' keys
  bool vis_split;
  uint32_t tile_cost;  // vis_tile_cost of the draw
  uint32_t* tstart;    // GPU tiles
  uint32_t* tile_count;  // tile_slots(T) words: records per tile, at tile_slot (zero before the setup launch)
  uint32_t* tend;
  uint32_t* hist;      // batches: bucket histogram
  uint32_t* counters;  // CT_COUNT
  unsigned long long* stats;    // ST_COUNT
  unsigned long long* partial;  // per-workgroup statistics partials (>= max(setup blocks, GPU tiles))
};

// ---------------------------------------------------------------- batched jobs
// Workgroup -> job map of one batched launch: job[b] for every workgroup b; range[j] = (first
// workgroup, workgroups) of job j (no workgroups: the job has no work in this launch).
struct stage_map {
  const uint32_t* job;
  const uint2* range;
};
// One draw of a batch: its parameters and its slices of the batch's buffers.  B.keys/B.vals are the
// batch-wide record arrays; B.cnt is the job's slice of the batch-wide per-triangle counts (followed
// by the next job's slice or the trailing total slot); B.hist likewise.
struct batch_job {
  draw_params P;
  draw_buffers B;
  int32_t vis_mode;
  uint32_t tiles;          // GPU tiles
  uint32_t bucket_blocks;  // binning workgroups; the histogram is tiles x bucket_blocks
  uint32_t pad;
};
// A clear as a 16-byte pattern fill of `value` converted to format pf (texel sizes 4, 8, 16):
// `words` 16-byte stores, then `tail` bytes (whole texels).  A depth/stencil clear is the RG32F
// value (depth, stencil bits).
struct fill_item {
  uint8_t* data;
  size_t words;
  uint32_t tail;
  int32_t pf;
  float4 value;
};
struct resolve_item {
  surface_desc src, dst;
};

void launch_batch_reset(uint32_t* counters, uint32_t n, uint32_t* cnt_tail, uint32_t* hist_tail, uint32_t* status,
                        hipStream_t s);
void launch_fill_batch(const fill_item* items, stage_map m, uint32_t blocks, hipStream_t s);
void launch_resolve_batch(const resolve_item* items, stage_map m, uint32_t blocks, hipStream_t s);
void launch_vs_batch(const batch_job* jobs, stage_map m, uint32_t blocks, hipStream_t s);
void launch_setup_batch(int na, const batch_job* jobs, stage_map m, uint32_t blocks, hipStream_t s);
void launch_clip_batch(int na, const batch_job* jobs, stage_map m, uint32_t blocks, hipStream_t s);
void launch_emit_batch(const batch_job* jobs, stage_map m, uint32_t blocks, uint32_t capacity, hipStream_t s);
// binning with pt records per thread (256 * pt per workgroup): phase 0 histograms, 1 scatter
bool batch_bin_items_valid(int pt);
void launch_bucket_batch(int pt, int phase, const batch_job* jobs, stage_map m, uint32_t blocks, uint32_t capacity,
                         hipStream_t s);
void launch_range_batch(const batch_job* jobs, stage_map m, uint32_t blocks, hipStream_t s);
void launch_tile_order_batch(const batch_job* jobs, uint32_t njobs, hipStream_t s);
// threads: 64, 128 or 256 lanes per GPU tile; gt: GPU tile side 8, 16 or 32 (8 and 32 for single-sample
// draws).  False for a combination without a kernel.
bool vis_batch_supported(int samples, bool shade, int threads, int gt);
bool launch_vis_batch(int na, int samples, bool shade, int threads, int gt, const batch_job* jobs, stage_map m,
                      uint32_t blocks, hipStream_t s);
void launch_batch_check(const batch_job* jobs, uint32_t njobs, uint32_t capacity, int pt, uint32_t* status, hipStream_t s);
// out[j]: records of job j; out[njobs + j]: its clip-overflow counter
void launch_batch_counts(const batch_job* jobs, uint32_t njobs, uint32_t* out, hipStream_t s);
int vis_mode(const draw_params& P);

// The anisotropic weights: each source that samples holds its own copy.
hipError_t upload_ewa_table_raster(const float* table256, hipStream_t s);
hipError_t upload_ewa_table_inorder(const float* table256, hipStream_t s);
hipError_t upload_ewa_table_vis(const float* table256, hipStream_t s);

// stats[slot] += sum(partial[0..n))
void launch_reduce_partials(const unsigned long long* partial, uint32_t n, unsigned long long* stats, int slot, hipStream_t s);

void launch_fill_u32(uint32_t* p, uint32_t n, uint32_t v, hipStream_t s);
// The vertex launch of a single draw; it also zeroes the draw's counters and ntiles words of tiles.
void launch_vs(const draw_params& P, float4* vbuf, uint32_t* counters, uint32_t* tiles, size_t ntiles, hipStream_t s);
// Setup and clipping of a single draw, which emit its records (those beyond `capacity` are counted and
// dropped) and count them per tile.
void launch_setup(const draw_params& P, const draw_buffers& B, uint32_t capacity, hipStream_t s);
void launch_clip(const draw_params& P, const draw_buffers& B, uint32_t capacity, hipStream_t s);
// The tiles' record lists from the emitted records, in two steps.  Ranges: tstart/tend, each tile's
// record-count class and rank in it (kept in B.partial until the lists' launch).  Lists: `order` (tiles
// words), with B.vis_split the parts of split tiles (when the count is within `cap`), and vals[1], or in
// primitive order vals[0] (`sorted`), sized for `cap` records; the count is read from B.counters on the
// device.  The lists' launch writes the draw's mail (targets without GPU tiles: nothing is launched).
void launch_tile_ranges(const draw_params& P, const draw_buffers& B, hipStream_t s);
void launch_tile_lists(const draw_params& P, const draw_buffers& B, uint32_t cap, uint32_t* order, bool sorted, draw_mail* mail,
                       uint32_t seq, hipStream_t s);
// In-place exclusive scan of n u32; writes the total to *total_dev.  tmp holds >= scan_tmp_size(n).
size_t scan_tmp_size(uint32_t n);
void launch_exclusive_scan(uint32_t* data, uint32_t n, uint32_t* tmp, uint32_t* total_dev, hipStream_t s);
// Whether launch_vis will take the draw (its visibility mode exists and the tiles are 16x16).
bool vis_applicable(const draw_params& P);
// The raster passes read the record count on the device and do nothing when it exceeds B.list_cap.
void launch_raster(const draw_params& P, const draw_buffers& B, int which, hipStream_t s);
// In-order rasterisation, shading and blending with one pixel per lane: every in-order draw with 16x16
// GPU tiles, except under a statistics query and with a SASL pixel shader (launch_raster takes those).
bool inorder_applicable(const draw_params& P);
bool inorder_takes_color_clear(const draw_params& P);
void launch_inorder(const draw_params& P, const draw_buffers& B, int which, hipStream_t s);
// Order-independent visibility (and, with shade, the deferred pixel shader) of an opaque early-Z draw,
// laid out for `records` records; false when the draw needs the in-order kernel.  merges > 0: finishes
// that many split tiles (counters[CT_MERGES]) after a call with 0 has rasterised the tiles.
bool launch_vis(const draw_params& P, const draw_buffers& B, int which, bool shade, uint32_t records, uint32_t merges,
                hipStream_t s);
bool needs_shading(const draw_params& P);
// A SASL pixel shader whose colour is written: such draws run the in-order raster kernel.
bool sasl_shades(const draw_params& P);
void launch_sasl_quads(const sasl_program* prog, const ps_samplers* SM, uint32_t has_mask, const float4* in, float4* out,
                       uint32_t nquads, hipStream_t s);
void launch_shade(const draw_params& P, const draw_buffers& B, hipStream_t s);

void launch_clear(const surface_desc& s, float4 value, hipStream_t st);
// flags: 1 depth, 2 stencil
void launch_clear_ds(const surface_desc& s, uint32_t flags, float depth, uint32_t stencil, hipStream_t st);
void launch_resolve(const surface_desc& src, const surface_desc& dst, hipStream_t st);
void launch_mip(const surface_desc& src, const surface_desc& dst, int filter, hipStream_t st);

}  // namespace srx
