// Rules on a draw's record count, for host and device code: the count its lists are first formed for, and in
// the visibility pass when depth culling begins and which tiles are split.  The device applies the latter to
// the draw's own count; the host, which does not know it yet, sizes the tables for every count up to the lists'
// capacity.
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define SRX_HD __host__ __device__
#else
#define SRX_HD
#endif

namespace srx {

// Records that the lists of a draw of `prims` primitives on T tiles are formed for before its count is known:
// 5/4 of the most that recent draws had, and at least one for every triangle that clipping can leave, so that
// a large mesh among small draws seldom outgrows its lists however many of those came in between (a frame of
// one 522k-triangle mesh and ten draws of 20,000 triangles 720 -> 697 us, as nothing is queued twice).
constexpr uint32_t MAX_RECORDS = 0xFFFFFFF0u;  // a draw with more is refused
SRX_HD inline uint32_t record_estimate(uint32_t recent, uint32_t prims, uint32_t T) {
  const uint64_t grown = recent + static_cast<uint64_t>(recent) / 4, own = 3ull * prims + T, least = 1u << 16;
  const uint64_t want = grown > own ? grown : own;
  return want < least ? static_cast<uint32_t>(least) : want < MAX_RECORDS ? static_cast<uint32_t>(want) : MAX_RECORDS;
}

// Records of a tile taken before depth culling begins: few for draws whose triangles lie on VIS_LARGE or
// more GPU tiles on average, whose lists are deep (of the 323 records a tile of the 2,000-triangle
// plain scene has, 50 of the last 259 survive: 60 -> 35 us); a whole chunk for draws of smaller ones,
// which seldom cover a tile before its list ends (64 there: 161 -> 186 us for the mesh that fills the
// target).
constexpr uint32_t VIS_FIRST = 64, VIS_LARGE = 4;
SRX_HD inline bool vis_large(uint64_t records, uint32_t prims) {
  return records >= static_cast<uint64_t>(VIS_LARGE) * prims;
}

// A tile's time is its list's length and what finishing it costs, so lists much longer than an even share of
// both over the workgroups the GPU holds at a time (VIS_SLOTS of them busy) are split: the textured mesh frame
// at the oblique camera has 1,008 tiles with records, 433 in the median and 4,184 in the longest, which alone
// kept the pass running for 170 us (split: 88 + 29 us for the merge).  Where the pass outlasts its longest tile
// a split only adds work: the same mesh over most of the target takes 282 us a frame without splits and 311
// with every tile of more than an even share of the records alone split (4 samples; 1 sample 173 and 192).
// Draws of large triangles, whose lists depth culling shortens as it goes, are split later.
constexpr uint32_t VIS_PART_SMALL = 1024, VIS_PART_LARGE = 2048, VIS_SLOTS = 640;
// What finishing a tile costs, in records (depth, shading and stores): half as much splits tiles of the latter
// view, twice as much leaves long tiles of the former whole (188 -> 206 us a frame).
SRX_HD inline uint32_t vis_tile_cost(int samples, bool shade) { return shade ? 64u + 24u * static_cast<uint32_t>(samples) : 32u; }
// Part sizes go by quarters of a power of two: lists of VIS_PART_SMALL and more records are counted by step as
// the tiles' ranges are formed, so the next launch knows how many tiles a part size splits before it has
// looked at any, and the host hears of it no later than of the record count (a launch later: 4 to 6 us a frame
// of 50 to 100 us).
constexpr uint32_t VIS_STEPS = 88;
SRX_HD inline uint32_t vis_step_size(uint32_t k) { return (4u + (k & 3u)) << (8u + (k >> 2)); }
SRX_HD inline uint32_t vis_step(uint32_t records) {  // the largest step of at most `records` >= VIS_PART_SMALL
  const uint32_t lg = 31u - static_cast<uint32_t>(__builtin_clz(records));
  return 4u * (lg - 10u) + ((records >> (lg - 2u)) & 3u);
}
static_assert(VIS_PART_SMALL == 1u << 10 && VIS_PART_LARGE >= VIS_PART_SMALL, "step 0, and the two heaviest classes of tiles");
// Records per part of a draw with `records` records on `tiles` tiles: a tile with more is split, that is one
// whose step is vis_step(part + 1) or above.
SRX_HD inline uint32_t vis_part(uint32_t prims, uint32_t records, uint32_t tiles, uint32_t tile_cost) {
  const uint32_t least = vis_large(records, prims) ? VIS_PART_LARGE : VIS_PART_SMALL;
  const uint32_t share = records / VIS_SLOTS + tiles * tile_cost / VIS_SLOTS, want = least > share ? least : share;
  const uint32_t k = vis_step(want);
  return vis_step_size(vis_step_size(k) < want ? k + 1 : k) - 1;
}
// Draws of which no tile is split: a primitive gives at most three triangles, each once on a tile.
SRX_HD inline bool vis_can_split(uint32_t prims) { return 3ull * prims > VIS_PART_LARGE; }
// Upper bounds of the parts and split tiles of a draw with at most `records` records: a tile of n > part
// records has ceil(n / part) < 2 n / part parts, and part, at least VIS_PART_SMALL - 1 and records / VIS_SLOTS - 1,
// goes at most VIS_SLOTS + 2 times into them.  A part takes 256 * samples keys.
SRX_HD inline void vis_split_bounds(uint32_t prims, uint32_t records, uint32_t* parts, uint32_t* tiles) {
  const uint32_t n = records / (VIS_PART_SMALL - 1), most = n < VIS_SLOTS + 2 ? n : VIS_SLOTS + 2;
  *parts = vis_can_split(prims) ? 2 * (most + 1) : 0;
  *tiles = vis_can_split(prims) ? most + 1 : 0;
}

}  // namespace srx
