// Order-independent visibility of opaque early-Z draws, fused with their shading: one GPU tile per
// workgroup, for single draws and for batches of jobs.
#include "srx_kernel_common.h"

#include <type_traits>

namespace srx {

hipError_t upload_ewa_table_vis(const float* table256, hipStream_t s) {
  return hipMemcpyToSymbolAsync(HIP_SYMBOL(c_ewa), table256, 256 * sizeof(float), 0, hipMemcpyHostToDevice, s);
}

// ---------------------------------------------------------------- order-independent visibility
// For an opaque early-Z draw with blending off, the reference's sequential early-Z test (depth written
// at test time, framebuffer.cpp:522-614) leaves in every sample the result of a running reduction:
//   LESS/GREATER (+write): the first triangle reaching the extreme depth wins;
//   LESS_EQUAL/GREATER_EQUAL (+write): the last triangle reaching the extreme depth wins;
//   ALWAYS, depth off, EQUAL, or any function without depth write: among the triangles that pass
//   against the initial depth, the last one wins.
// Each of these is a minimum over a 64-bit key (ordered depth, primitive order), so lanes can
// rasterise different triangles of a tile at once and merge with LDS atomic-min.
enum { VIS_LESS = 0, VIS_LEQUAL = 1, VIS_GREATER = 2, VIS_GEQUAL = 3, VIS_LATEST = 4, VIS_NONE = 5 };

__device__ __forceinline__ uint32_t ord_depth(float z) {
  uint32_t u = __float_as_uint(z + 0.0f);  // -0 compares equal to +0
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ unsigned long long initial_key(int mode, float d0) {
  if (mode == VIS_LATEST || mode == VIS_NONE) return 0xFFFFFFFFull;
  if (d0 != d0) return 0ull;  // a NaN depth lets nothing pass
  uint32_t zk = ord_depth(d0);
  if (mode == VIS_GREATER || mode == VIS_GEQUAL) zk = ~zk;
  uint32_t lo = (mode == VIS_LESS || mode == VIS_GREATER) ? 0u : 0xFFFFFFFFu;
  return (static_cast<unsigned long long>(zk) << 32) | lo;
}

__device__ __forceinline__ uint32_t key_winner(int mode, unsigned long long k) {
  uint32_t lo = static_cast<uint32_t>(k);
  if (mode == VIS_LESS || mode == VIS_GREATER) return lo == 0u ? NO_WINNER : lo - 1u;
  return lo == 0xFFFFFFFFu ? NO_WINNER : 0xFFFFFFFEu - lo;
}

// Depth the reference's early-Z test wrote for winner w of sample smp of pixel (px, py).
template <int S>
__device__ __forceinline__ float winner_depth(const draw_params& P, int mode, unsigned long long key, uint32_t w,
                                              const float4* __restrict__ tri_rec, int px, int py, int smp) {
  if (mode != VIS_LATEST) {
    // depth modes carry the winning sample depth in the key; only +-0 is ambiguous there
    uint32_t zk = static_cast<uint32_t>(key >> 32);
    if (mode == VIS_GREATER || mode == VIS_GEQUAL) zk = ~zk;
    const uint32_t u = (zk & 0x80000000u) ? (zk & 0x7FFFFFFFu) : ~zk;
    if (u != 0u) return __uint_as_float(u);
  }
  // the winner's depth at this sample, as its quad computed it
  const float4* tr = tri_rec + tri_slot(P, w) * 5;
  const float4 d3 = tr[3], d4 = tr[4];
  const int qx0 = px & ~1, qy0 = py & ~1;
  const float dx = (0.5f + static_cast<float>(qx0)) - d3.y;
  const float dy = (0.5f + static_cast<float>(qy0)) - d3.z;
  float z00 = d3.w + ((d4.x * dx) + (d4.y * dy));
  float zp;
  if ((px & 1) == 0 && (py & 1) == 0) zp = z00;
  else if ((py & 1) == 0) zp = z00 + d4.x;
  else if ((px & 1) == 0) zp = z00 + d4.y;
  else zp = (z00 + d4.x) + d4.y;
  float nd = zp;
  if (S > 1) nd = ((P.sp[smp][0] - 0.5f) * d4.x + (P.sp[smp][1] - 0.5f) * d4.y) + zp;
  return nd;
}

// cmpf as a truth table over the comparison's outcome: bit 0 less, 1 equal, 2 greater, 3 unordered.
__device__ __forceinline__ uint32_t cmpf_table(int f) {
  // nibble f: never, less, equal, less_equal, greater, not_equal, greater_equal, always
  return (f >= 0 && f < 8) ? (0xF6D43210u >> (4 * f)) & 0xFu : 0xFu;
}
__device__ __forceinline__ bool cmpf_by_table(uint32_t table, float a, float b) {
  const uint32_t o = (a < b) ? 0u : (a == b) ? 1u : (a > b) ? 2u : 3u;
  return ((table >> o) & 1u) != 0u;
}

// Phase 1c of vis_body over the chunk's work list: items [0, np) are (record, 4x4 block) pairs the
// rasteriser tests sample by sample (draw_partial_tile, rasterizer.cpp:298-439), items [np, nt)
// blocks it accepts whole (draw_full_tile, :285-296).  A partial item tests, pixel by pixel, only
// the pixels a conservative bound leaves (see below), each sample with the reference's expression
// ((sx + fx) * ex) + ((sy + fy) * ey) < e_value, and every covered sample's key goes to the LDS
// atomic-min.  Depth per sample is the quad chain of
// step_2d_unproj_pos_quad (p00 = v0 + (ddx*dx + ddy*dy), +ddx to the right, +ddy below) plus the
// sample offset term of rasterize_triangle (rasterizer.cpp:678-687).
// Keys: DEPTH (the LESS, LEQUAL, GREATER, GEQUAL modes with depth writes) = the sample depth's
// order-preserving bits (complemented when the greater depth wins) over the record's order term,
// and a NaN depth passes nothing; otherwise (VIS_LATEST) the sample passes against the target's
// initial depth (always without a depth test) and the key is the order term alone.  The per-sample
// predicates are combined with bitwise operators so that each sample costs one masked atomic and
// no branch.
template <int S, int GT, bool DEPTH>
__device__ __forceinline__ void vis_items(const draw_params& P, int mode, const float4* __restrict__ recs,
                                          const uint16_t* __restrict__ work, uint32_t np, uint32_t nt,
                                          unsigned long long* __restrict__ keys, const float* __restrict__ d0s,
                                          int ox, int oy, int tw, int th, int tid, int NT) {
  constexpr int NBS = GT / 4;
  const uint32_t flip = (mode == VIS_GREATER || mode == VIS_GEQUAL) ? 0xFFFFFFFFu : 0u;
  const bool later_wins = mode == VIS_LEQUAL || mode == VIS_GEQUAL || mode == VIS_LATEST;
  const uint32_t table = P.depth_enable ? cmpf_table(P.depth_func) : 0xFu;
  const bool read_depth = P.read_depth != 0;
  // extreme sample positions inside a pixel
  float spx_lo = P.sp[0][0], spx_hi = P.sp[0][0], spy_lo = P.sp[0][1], spy_hi = P.sp[0][1];
#pragma unroll
  for (int s = 1; s < S; ++s) {
    spx_lo = fminf(spx_lo, P.sp[s][0]);
    spx_hi = fmaxf(spx_hi, P.sp[s][0]);
    spy_lo = fminf(spy_lo, P.sp[s][1]);
    spy_hi = fmaxf(spy_hi, P.sp[s][1]);
  }
  for (uint32_t wi = tid; wi < nt; wi += NT) {
    const uint32_t wk = work[wi];
    const int j = static_cast<int>(wk >> 7), b = static_cast<int>((wk >> 1) & 63u);
    const float4 r0 = recs[j * 4 + 0], r1 = recs[j * 4 + 1], r2 = recs[j * 4 + 2], r3 = recs[j * 4 + 3];
    const float e[9] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w, r2.x};
    const float z0 = r2.y, zx = r2.z, zy = r2.w, dzx = r3.x, dzy = r3.y;
    const uint32_t id = __float_as_uint(r3.z);
    const uint32_t lo = later_wins ? 0xFFFFFFFEu - id : id + 1u;
    const bool full = wi >= np;
    float aa[S];
#pragma unroll
    for (int s = 0; s < S; ++s) aa[s] = (S > 1) ? (P.sp[s][0] - 0.5f) * dzx + (P.sp[s][1] - 0.5f) * dzy : 0.0f;
    const int bc = b % NBS, br = b / NBS;
    const int Bx = ox + bc * 4, By = oy + br * 4;
    const int lbase = (br * 4 * GT + bc * 4) * S;  // the block's first sample in `keys`
    const int bw = min(4, tw - Bx), bh = min(4, th - By);  // columns and rows inside the target
    // depth at the top-left pixel of each 2x2 quad of the block
    float zq[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float dx = (0.5f + static_cast<float>(Bx + (q & 1) * 2)) - zx;
      const float dy = (0.5f + static_cast<float>(By + (q >> 1) * 2)) - zy;
      zq[q] = z0 + ((dzx * dx) + (dzy * dy));
    }
    float evp[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      evp[k] = e[k * 3 + 2] - ((static_cast<float>(Bx) * e[k * 3]) + (static_cast<float>(By) * e[k * 3 + 1]));
    // Every depth of the block is finite and above zero (almost always): each step of the quad chain is
    // monotonic in its operands, so the smallest comes from the smallest ones.  A sample's key depth word
    // is then its bits with the sign flipped (and complemented when the greater depth wins).
    // (64 batched jobs' visibility 6.96 -> 5.90 ms, the 2048x2048 shadow pass 0.47 -> 0.39 ms.)
    bool plain = false;
    if (DEPTH) {
      float lo_aa = aa[0], hi_aa = aa[0];
#pragma unroll
      for (int s = 1; s < S; ++s) {
        lo_aa = fminf(lo_aa, aa[s]);
        hi_aa = fmaxf(hi_aa, aa[s]);
      }
      const float zmin = fminf(fminf(zq[0], zq[1]), fminf(zq[2], zq[3])), zmax = fmaxf(fmaxf(zq[0], zq[1]), fmaxf(zq[2], zq[3]));
      const float any = (zq[0] + zq[1]) + (zq[2] + zq[3]);  // not finite when one of them is not
      const float nmin = ((zmin + fminf(dzx, 0.0f)) + fminf(dzy, 0.0f)) + lo_aa;
      const float nmax = ((zmax + fmaxf(dzx, 0.0f)) + fmaxf(dzy, 0.0f)) + hi_aa;
      plain = fabsf(any) < 3.0e38f && nmin > 0.0f && nmax < 3.0e38f;
    }
    const uint32_t sign = 0x80000000u ^ flip;
    if (!full) {
      // Pixels that may hold a covered sample.  Float rounding is monotonic, so an edge's value at
      // any sample of a pixel is at most its value at the pixel's extreme sample column and row
      // for that edge's signs, computed with the same operations; a pixel whose extreme value
      // fails an edge has no sample that passes it.  Only the remaining pixels are tested sample
      // by sample.
      uint32_t M = 0;
      {
        float cx[3][4], cy[3][4];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const float sx = e[k * 3] >= 0.0f ? spx_hi : spx_lo, sy = e[k * 3 + 1] >= 0.0f ? spy_hi : spy_lo;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            cx[k][c] = (sx + static_cast<float>(c)) * e[k * 3];
            cy[k][c] = (sy + static_cast<float>(c)) * e[k * 3 + 1];
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const bool maybe = !((cx[0][c] + cy[0][r]) < evp[0]) & !((cx[1][c] + cy[1][r]) < evp[1]) &
                               !((cx[2][c] + cy[2][r]) < evp[2]) & (c < bw) & (r < bh);
            if (maybe) M |= 1u << (r * 4 + c);
          }
      }
      if (S == 1 && DEPTH && plain) {
        // one sample: the bound is the sample's own test, so M is the coverage
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int p0 = (q >> 1) * 8 + (q & 1) * 2;
          const float z01 = zq[q] + dzx;
          const float zz[4] = {zq[q], z01, zq[q] + dzy, z01 + dzy};
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int px = p0 + (i >> 1) * 4 + (i & 1);
            const unsigned long long k = (static_cast<unsigned long long>(__float_as_uint(zz[i]) ^ sign) << 32) | lo;
            if ((M >> px) & 1u) atomicMin(&keys[lbase + (px >> 2) * GT + (px & 3)], k);
          }
        }
        continue;
      }
      while (M) {
        const int px = __builtin_ctz(M);
        M &= M - 1u;
        const int r = px >> 2, c = px & 3;
        const int q = ((r >> 1) << 1) | (c >> 1);
        float z = (q & 2) ? ((q & 1) ? zq[3] : zq[2]) : ((q & 1) ? zq[1] : zq[0]);
        z = (c & 1) ? z + dzx : z;
        z = (r & 1) ? z + dzy : z;
        const float fx = static_cast<float>(c), fy = static_cast<float>(r);
        const int lp = lbase + (r * GT + c) * S;
#pragma unroll
        for (int s = 0; s < S; ++s) {
          const float mx = P.sp[s][0] + fx, my = P.sp[s][1] + fy;
          const bool covered = !(((mx * e[0]) + (my * e[1])) < evp[0]) & !(((mx * e[3]) + (my * e[4])) < evp[1]) &
                               !(((mx * e[6]) + (my * e[7])) < evp[2]);
          const float nd = (S > 1) ? (aa[s] + z) : z;
          unsigned long long k;
          bool pass;
          if (DEPTH) {
            const uint32_t u = __float_as_uint(nd + 0.0f);  // -0 orders as +0
            const uint32_t ord = u ^ (static_cast<uint32_t>(static_cast<int32_t>(u) >> 31) | 0x80000000u);
            k = (static_cast<unsigned long long>(ord ^ flip) << 32) | lo;
            pass = nd == nd;
          } else {
            k = lo;
            pass = cmpf_by_table(table, nd, read_depth ? d0s[lp + s] : 0.0f);
          }
          if (covered & pass) atomicMin(&keys[lp + s], k);
        }
      }
      continue;
    }
    // a block the rasteriser accepts whole: every sample inside the target
    float zp[16];  // pixel depths (row r, column c at [r * 4 + c]) by the quad chain
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int p0 = (q >> 1) * 8 + (q & 1) * 2;
      zp[p0] = zq[q];
      zp[p0 + 1] = zq[q] + dzx;
      zp[p0 + 4] = zq[q] + dzy;
      zp[p0 + 5] = zp[p0 + 1] + dzy;
    }
    if (DEPTH && plain && bw == 4 && bh == 4) {
#pragma unroll
      for (int i = 0; i < 16; ++i)
#pragma unroll
        for (int s = 0; s < S; ++s) {
          const float nd = (S > 1) ? (aa[s] + zp[i]) : zp[i];
          atomicMin(&keys[lbase + ((i >> 2) * GT + (i & 3)) * S + s],
                    (static_cast<unsigned long long>(__float_as_uint(nd) ^ sign) << 32) | lo);
        }
      continue;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int s = 0; s < S; ++s) {
          const float nd = (S > 1) ? (aa[s] + zp[r * 4 + c]) : zp[r * 4 + c];
          const int li = lbase + (r * GT + c) * S + s;
          unsigned long long k;
          bool pass;
          if (DEPTH) {
            const uint32_t u = __float_as_uint(nd + 0.0f);
            const uint32_t ord = u ^ (static_cast<uint32_t>(static_cast<int32_t>(u) >> 31) | 0x80000000u);
            k = (static_cast<unsigned long long>(ord ^ flip) << 32) | lo;
            pass = nd == nd;
          } else {
            k = lo;
            pass = cmpf_by_table(table, nd, read_depth ? d0s[li] : 0.0f);
          }
          if (pass & (c < bw) & (r < bh)) atomicMin(&keys[li], k);
        }
  }
}

// One 16x16 GPU tile per workgroup, in three phases:
//  1. one triangle per lane: coverage with the reference's decision chain, LDS atomic-min of the
//     (ordered depth, primitive order) key of every covered sample;
//  2. one pixel per lane: winners -> depth/stencil target, and one shading item per distinct winner
//     (pixel, winner, sample mask) appended to an LDS list;
//  3. (SHADE) one item per lane: the winner's quad interpolants at the pixel's quad (the values the
//     reference's last passing draw_quad/draw_full_quad computed), the pixel shader for that pixel,
//     and the colour stored to the item's samples.  Items are spread evenly over the lanes however
//     many triangles share a pixel.
#ifndef SRX_VIS_THREADS
#define SRX_VIS_THREADS 256
#endif
// LDS shared by phase 1 (a chunk of NT records, their (record, block) work list, and up to 2 NT records
// that depth culling has let through) and phase 3 (shading items), for GT x GT GPU tiles
__host__ __device__ constexpr int vis_union_bytes(int nt, int s, bool shade, int gt = 16) {
  const int chunk = nt * 64 + nt * (gt / 4) * (gt / 4) * 2 + nt * 8;
  return chunk > (shade ? gt * gt * s * 8 : 0) ? chunk : gt * gt * s * 8;
}
// S (depth, stencil) pairs of a pixel as wide stores (surfaces are allocated at 256-byte alignment, so a
// pixel's samples start at a multiple of their size).
template <int S>
__device__ __forceinline__ void store_ds_pixel(uint8_t* p, const float (&d)[S], uint32_t stencil) {
  const float f = __uint_as_float(stencil);
  if constexpr (S == 1) {
    *reinterpret_cast<float2*>(p) = make_float2(d[0], f);
  } else {
#pragma unroll
    for (int s = 0; s < S; s += 2) *reinterpret_cast<float4*>(p + s * 8) = make_float4(d[s], f, d[s + 1], f);
  }
}
template <int S>
__device__ __forceinline__ void fill_color_pixel(const draw_params& P, int px, int py) {
  const float4 c = make_float4(P.clear_rgba[0], P.clear_rgba[1], P.clear_rgba[2], P.clear_rgba[3]);
  if (P.color.pf == PF_RGBA8 && S > 1) {
    const uint32_t u = unorm8(c.x) | (unorm8(c.y) << 8) | (unorm8(c.z) << 16) | (unorm8(c.w) << 24);
    uint8_t* p = sample_addr(P.color, px, py, 0);
    if constexpr (S == 4) *reinterpret_cast<uint4*>(p) = make_uint4(u, u, u, u);
    else *reinterpret_cast<uint2*>(p) = make_uint2(u, u);
  } else {
#pragma unroll
    for (int s = 0; s < S; ++s) store_texel(P.color.pf, sample_addr(P.color, px, py, s), c);
  }
}
// Static LDS of vis_body besides the union (keys, initial depths).
__host__ __device__ constexpr int vis_static_bytes(int s, int gt) { return gt * gt * s * 12 + 256; }
// Phases 2 and 3 of a tile whose keys are final (*nitems is zero).
template <int NA, int S, bool SHADE, int GT>
__device__ __forceinline__ void vis_finish(const draw_params& P, int mode, const unsigned long long* keys, uint2* items,
                                           uint32_t* nitems, int ox, int oy, int NT, const float4* __restrict__ tri_rec,
                                           const float4* __restrict__ tri_attr, const ps_samplers* __restrict__ SM,
                                           uint32_t* __restrict__ wout) {
  constexpr int PX = GT * GT;
  const int tw = static_cast<int>(P.target_w), th = static_cast<int>(P.target_h);
  const int tid = threadIdx.x;
  const bool has_ds = P.ds.data != nullptr;
  // phase 2: winners -> depth, shading items
  for (int p = tid; p < PX; p += NT) {
    const int px = ox + (p % GT), py = oy + (p / GT);
    if (px >= tw || py >= th) continue;
    uint32_t w[S];
    float d[S];
    uint32_t left = 0;
#pragma unroll
    for (int smp = 0; smp < S; ++smp) {
      const unsigned long long key = keys[p * S + smp];
      w[smp] = key_winner(mode, key);
      const bool won = w[smp] != NO_WINNER;
      if (won) left |= 1u << smp;
      d[smp] = P.clear_depth;
      if (won && has_ds && P.write_depth) {
        d[smp] = winner_depth<S>(P, mode, key, w[smp], tri_rec, px, py, smp);
        if (!P.clear_ds) *reinterpret_cast<float*>(sample_addr(P.ds, px, py, smp)) = d[smp];
      }
      // winners for a separate shading pass (SASL pixel shaders), laid out like the colour samples
      if (!SHADE && wout) wout[(static_cast<size_t>(py) * tw + px) * S + smp] = w[smp];
    }
    // a cleared target: every sample is written, the stencil keeps its clear value
    if (has_ds && P.clear_ds) store_ds_pixel<S>(sample_addr(P.ds, px, py, 0), d, P.clear_stencil);
    if (SHADE && P.clear_color) {
      if (left == 0) {
        fill_color_pixel<S>(P, px, py);
      } else {
#pragma unroll
        for (int smp = 0; smp < S; ++smp)
          if (!((left >> smp) & 1u))
            store_texel(P.color.pf, sample_addr(P.color, px, py, smp),
                        make_float4(P.clear_rgba[0], P.clear_rgba[1], P.clear_rgba[2], P.clear_rgba[3]));
      }
    }
    if (SHADE) {
#pragma unroll
      for (int it = 0; it < S; ++it) {
        if (!left) break;
        const int s0 = __builtin_ctz(left);
        uint32_t cur = w[0];
#pragma unroll
        for (int smp = 1; smp < S; ++smp)
          if (smp == s0) cur = w[smp];
        uint32_t m = 0;
#pragma unroll
        for (int smp = 0; smp < S; ++smp)
          if (w[smp] == cur) m |= 1u << smp;
        left &= ~m;
        items[atomicAdd(nitems, 1u)] = make_uint2(cur, static_cast<uint32_t>(p) | (m << 12));
      }
    }
  }
  if (!SHADE) return;
  __syncthreads();
  // phase 3: shading items
  const uint32_t n = *nitems;
  for (uint32_t j = tid; j < n; j += NT) {
    const uint2 item = items[j];
    const uint32_t cur = item.x, p = item.y & 4095u, m = item.y >> 12;
    if (cur >= 3u * P.prim_count) continue;  // every winner id is below 3 * prim_count
    const int px = ox + static_cast<int>(p % GT), py = oy + static_cast<int>(p / GT);
    const int pi = (px & 1) | ((py & 1) << 1);
    attr_setup<NA> at;
    load_attr<NA>(P, tri_attr, cur, at);
    const quad_lazy<NA> q(at, P, px & ~1, py & ~1);
    const float4 c = run_ps_pixel<NA>(P, SM, q, pi);
#pragma unroll
    for (int smp = 0; smp < S; ++smp)
      if (m & (1u << smp)) store_texel(P.color.pf, sample_addr(P.color, px, py, smp), c);
  }
}
// NTC > 0: NTC lanes per workgroup, static LDS.  NTC == 0: blockDim.x lanes (64, 128 or 256) with
// the phase-1/3 union in dynamic LDS of vis_union_bytes(blockDim.x, S, SHADE, GT) bytes.
// GT: GPU tile side, 8, 16 or 32 pixels: a quarter of a 16x16 stage-16 region, one region, or 2x2
// regions of the reference's 64x64 tile; the 4x4 blocks are the reference's stage-4 blocks either way.
// The tile's records are those of `ws`: a whole tile, or one part of a split tile.
struct vis_span {
  int tile;
  uint32_t t0, t1;    // records
  uint32_t parts;     // parts the tile is split into
  uint32_t slot;      // this part's keys in vis_partial
};
template <int NA, int S, bool SHADE, int NTC, int GT>
__device__ __forceinline__ void vis_body(const draw_params& P, int mode, const vis_span& ws,
                                         unsigned long long* __restrict__ partial, const uint32_t* __restrict__ vals,
                                         const float4* __restrict__ tri_rec, const float4* __restrict__ tri_attr,
                                         const ps_samplers* __restrict__ SM, uint32_t first,
                                         uint32_t* __restrict__ wout = nullptr) {
  static_assert(GT == 8 || GT == 16 || GT == 32, "GPU tile side");
  constexpr int PX = GT * GT;       // pixels per GPU tile
  constexpr int NBS = GT / 4;       // 4x4 blocks per side
  constexpr int RPS = GT > 16 ? GT / 16 : 1;  // stage-16 regions per side
  using bmask_t = typename std::conditional<(GT > 16), unsigned long long, uint32_t>::type;
  const int NT = NTC > 0 ? NTC : static_cast<int>(blockDim.x);
  constexpr int UNION_BYTES = NTC > 0 ? vis_union_bytes(NTC, S, SHADE, GT) : 16;
  __shared__ unsigned long long keys[PX * S];
  __shared__ float d0s[PX * S];
  __shared__ __align__(16) unsigned char lds_static[UNION_BYTES];
  extern __shared__ __align__(16) unsigned char lds_dynamic[];
  unsigned char* const lds_union = NTC > 0 ? lds_static : lds_dynamic;
  __shared__ uint32_t wsum[4];
  __shared__ uint32_t hiz[NBS * NBS];
  __shared__ uint32_t nitems, nlist, far_now, far_start;
  float4* recs = reinterpret_cast<float4*>(lds_union);                           // [NT][4]
  uint16_t* work = reinterpret_cast<uint16_t*>(lds_union + NT * 64);             // [NT * NBS^2]
  uint32_t* list = reinterpret_cast<uint32_t*>(lds_union + NT * 64 + NT * NBS * NBS * 2);  // [2 * NT]
  uint2* items = reinterpret_cast<uint2*>(lds_union);                            // [PX * S]
  const int gtile = ws.tile;
  const uint32_t t0 = ws.t0, t1 = ws.t1;
  const int gx = gtile % P.gtiles_x, gy = gtile / P.gtiles_x;
  const int ox = gx * GT, oy = gy * GT;
  const int t64x = ox & ~(TILE - 1), t64y = oy & ~(TILE - 1);
  const int tw = static_cast<int>(P.target_w), th = static_cast<int>(P.target_h);
  const int tid = threadIdx.x;
  const bool has_ds = P.ds.data != nullptr;
  // A tile without records takes the pending clears (88% of the textured mesh frame's tiles at the
  // oblique camera, whose empty passes through the phases below were 40% of its instructions).
  if (t0 == t1) {
    for (int p = tid; p < PX; p += NT) {
      const int px = ox + (p % GT), py = oy + (p / GT);
      if (px >= tw || py >= th) continue;
      if (has_ds && P.clear_ds) {
        float d[S];
#pragma unroll
        for (int smp = 0; smp < S; ++smp) d[smp] = P.clear_depth;
        store_ds_pixel<S>(sample_addr(P.ds, px, py, 0), d, P.clear_stencil);
      }
      if (SHADE && P.clear_color) fill_color_pixel<S>(P, px, py);
      if (!SHADE && wout) {
#pragma unroll
        for (int smp = 0; smp < S; ++smp) wout[(static_cast<size_t>(py) * tw + px) * S + smp] = NO_WINNER;
      }
    }
    return;
  }
  if (tid == 0) {
    nitems = 0;
    far_start = 0;
  }
  {
    uint32_t far = 0;
    for (int i = tid; i < PX * S; i += NT) {
      int px = ox + ((i / S) % GT), py = oy + ((i / S) / GT), smp = i % S;
      float d0 = 0.0f;
      bool blocked = false;
      if (has_ds && px < tw && py < th) {
        const float2 ds = P.clear_ds ? make_float2(P.clear_depth, __uint_as_float(P.clear_stencil))
                                     : *reinterpret_cast<const float2*>(sample_addr(P.ds, px, py, smp));
        d0 = ds.x;
        if (P.vis_stencil) {
          // framebuffer.cpp:445-479 (both faces share the function here); a failing sample takes
          // no colour and no depth
          const uint32_t os = __float_as_uint(ds.y) & P.read_mask;
          blocked = !cmpu(P.st_func[1], P.stencil_ref, os);
        }
      }
      d0s[i] = d0;
      // a blocked sample's key is below every candidate's and decodes as no winner
      keys[i] = blocked ? ((mode == VIS_LEQUAL || mode == VIS_GEQUAL) ? 0xFFFFFFFFull : 0ull) : initial_key(mode, d0);
      if (px < tw && py < th) far = max(far, static_cast<uint32_t>(keys[i] >> 32));
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) far = max(far, static_cast<uint32_t>(__shfl_xor(static_cast<int>(far), off, 64)));
    __syncthreads();  // far_start is zero
    if ((tid & 63) == 0) atomicMax(&far_start, far);
  }
  const int jx0 = (ox - t64x) >> 4, jy0 = (oy - t64y) >> 4;  // first stage-16 region of the tile
  // an 8x8 tile covers blocks [qx, qx+2) x [qy, qy+2) of its region; larger tiles whole regions
  const int qx = GT < 16 ? ((ox - t64x) & 15) >> 2 : 0, qy = GT < 16 ? ((oy - t64y) & 15) >> 2 : 0;
  constexpr int CW = GT < 16 ? GT / 4 : 4;  // block columns (rows) of a region inside the tile
  const float tvx = static_cast<float>(t64x), tvy = static_cast<float>(t64y);
  // Depth culling after the first records (vis_first): hiz[b] is the largest key depth word of 4x4 block b's
  // samples inside the target after the previous chunks, far_now the largest of the tile.  Keys only
  // decrease, so a record whose smallest possible depth word over the tile (or a block) exceeds it
  // cannot win any sample there.  Once the tile's farthest depth has come nearer than at the start,
  // every lane tests one record against it and the survivors are listed, so that chunks stay full of
  // records that can still win: of the lists of ~150 layers that the plain scenes give a tile, 15-35%
  // survive.
  const bool depth_keys = mode == VIS_LESS || mode == VIS_LEQUAL || mode == VIS_GREATER || mode == VIS_GEQUAL;
  const bool far_is_min = mode == VIS_GREATER || mode == VIS_GEQUAL;
  // smallest possible key depth word of a record's samples in the size x size square at (x, y): the depth
  // plane's extreme, widened by far more than the rounding of the per-sample evaluation; planes with
  // inf or nan terms are never culled
  auto nearest_key = [&](float4 d3, float4 d4, int x, int y, float size) -> uint32_t {
    const float z0 = d3.w, zx = d3.y, zy = d3.z, dzx = d4.x, dzy = d4.y;
    const float ax = static_cast<float>(x) - zx, ay = static_cast<float>(y) - zy;
    const float tx0 = dzx * ax, tx1 = dzx * (ax + size), ty0 = dzy * ay, ty1 = dzy * (ay + size);
    const float margin = (fabsf(z0) + fmaxf(fabsf(tx0), fabsf(tx1)) + fmaxf(fabsf(ty0), fabsf(ty1))) * 1.52587890625e-05f;
    const float zext = far_is_min ? (z0 + fmaxf(tx0, tx1) + fmaxf(ty0, ty1)) + margin
                                  : (z0 + fminf(tx0, tx1) + fminf(ty0, ty1)) - margin;
    if (!(fabsf(zext) < 3.0e38f)) return 0u;
    return far_is_min ? ~ord_depth(zext) : ord_depth(zext);
  };
  uint32_t next = t0, held = 0;  // records not yet looked at; survivors waiting in `list` (both uniform)
  while (next < t1 || held) {
    __syncthreads();  // the previous chunk's work list is consumed (and the keys are initialised)
    const bool hiz_on = depth_keys && next > t0;
    bool cull = false;
    if (hiz_on) {
      if (tid == 0) far_now = 0;
      // 16 consecutive lanes take one block's 16 pixels
      uint32_t far = 0;
      for (int u = tid; u < PX; u += NT) {
        const int b = u >> 4, q = u & 15;
        const int pr = (b / NBS) * 4 + (q >> 2), pc = (b % NBS) * 4 + (q & 3);
        const int pl = pr * GT + pc;
        uint32_t m = 0;
#pragma unroll
        for (int smp = 0; smp < S; ++smp) m = max(m, static_cast<uint32_t>(keys[pl * S + smp] >> 32));
        if (ox + pc >= tw || oy + pr >= th) m = 0;
        m = max(m, static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), 1, 64)));
        m = max(m, static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), 2, 64)));
        m = max(m, static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), 4, 64)));
        m = max(m, static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), 8, 64)));
        if (q == 0) hiz[b] = m;
        far = max(far, m);
      }
      __syncthreads();
      far = max(far, static_cast<uint32_t>(__shfl_xor(static_cast<int>(far), 16, 64)));
      far = max(far, static_cast<uint32_t>(__shfl_xor(static_cast<int>(far), 32, 64)));
      if ((tid & 63) == 0) atomicMax(&far_now, far);
      __syncthreads();
      cull = far_now < far_start;
    }
    uint32_t rec = 0xFFFFFFFFu;  // this lane's record of the chunk
    if (cull) {
      const uint32_t far = far_now;
      if (tid == 0) nlist = held;
      __syncthreads();
      while (next < t1 && held < static_cast<uint32_t>(NT)) {
        const uint32_t ri = next + tid;
        uint32_t v = 0;
        bool keep = false;
        if (ri < t1) {
          v = vals[ri];
          const float4* tr = tri_rec + tri_slot(P, v >> 1) * 5;
          keep = nearest_key(tr[3], tr[4], ox, oy, static_cast<float>(GT)) <= far;
        }
        const uint64_t km = __ballot(keep);
        uint32_t at = 0;
        if ((tid & 63) == 0 && km) at = atomicAdd(&nlist, static_cast<uint32_t>(__popcll(km)));
        at = static_cast<uint32_t>(__shfl(static_cast<int>(at), 0, 64));
        if (keep) list[at + __popcll(km & ((1ull << (tid & 63)) - 1ull))] = v;
        next = min(next + static_cast<uint32_t>(NT), t1);
        __syncthreads();
        held = nlist;
        __syncthreads();  // read before the next step adds to it
      }
      if (static_cast<uint32_t>(tid) < held) rec = list[tid];
      if (!held) break;  // nothing left that can win
    } else {
      const uint32_t take = min(min(t1 - next, static_cast<uint32_t>(NT)), depth_keys && next == t0 ? first : static_cast<uint32_t>(NT));
      if (static_cast<uint32_t>(tid) < take) rec = vals[next + tid];
      next += take;
    }
    // phase 1a: one record per lane -> the 4x4 blocks of this GPU tile it reaches (full or partial)
    bmask_t bm = 0, fm = 0;
    if (rec != 0xFFFFFFFFu) {
      const uint32_t id = rec >> 1;
      const float4* tr = tri_rec + tri_slot(P, id) * 5;
      float e[9], bb[4];
      read_tri_rec(tr, e, bb);
      const float4 d3 = tr[3], d4 = tr[4];
      const float bx0 = bb[0] - tvx, bx1 = bb[1] - tvx, by0 = bb[2] - tvy, by1 = bb[3] - tvy;
      // per-stage constants (rasterize_triangle, rasterizer.cpp:662-675, 704-710)
      float s1x[3], s1y[3], ra1[3], ev1[3], s2x[3], s2y[3], ra2[3], ev2[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        float ex = e[k * 3], ey = e[k * 3 + 1], ez = e[k * 3 + 2];
        bool mx = ex > 0, my = ey > 0;
        float sx = TILE * ex, sy = TILE * ey;
        float ra = -fabsf(sx) - fabsf(sy);
        float part = static_cast<float>(mx * TILE) * ex + static_cast<float>(my * TILE) * ey;
        sx *= 0.25f; sy *= 0.25f; ra *= 0.25f; part *= 0.25f;
        s1x[k] = sx; s1y[k] = sy; ra1[k] = ra;
        ev1[k] = (ez - part) - ((tvx * ex) + (tvy * ey));
        sx *= 0.25f; sy *= 0.25f; ra *= 0.25f; part *= 0.25f;
        s2x[k] = sx; s2y[k] = sy; ra2[k] = ra;
        ev2[k] = ez - part;
      }
      const bool rec_full = (rec & 1) != 0;  // the record covers its whole 64x64 tile
#pragma unroll
      for (int rr = 0; rr < RPS * RPS; ++rr) {
        const int jx = jx0 + rr % RPS, jy = jy0 + rr / RPS;
        bool region_full = rec_full;
        bool keep = true;
        if (!region_full) {
          // stage 16 (subdivide_tile on the 64x64 tile)
          bool rej = false, nacc = false;
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            float r = (s1x[k] * static_cast<float>(jx)) + (s1y[k] * static_cast<float>(jy));
            float a = r + ra1[k];
            rej |= r < ev1[k];
            nacc |= a < ev1[k];
          }
          rej |= bx0 >= static_cast<float>(jx * 16 + 16);
          rej |= bx1 < static_cast<float>(jx * 16);
          rej |= by0 >= static_cast<float>(jy * 16 + 16);
          rej |= by1 < static_cast<float>(jy * 16);
          keep = !rej;
          region_full = !nacc;
        }
        if (!keep) continue;
        const int rox = t64x + jx * 16, roy = t64y + jy * 16;  // the region's origin
        float ev2q[3];
#pragma unroll
        for (int k = 0; k < 3; ++k)
          ev2q[k] = ev2[k] - ((static_cast<float>(rox) * e[k * 3]) + (static_cast<float>(roy) * e[k * 3 + 1]));
        // candidate 4x4 blocks of the region inside this tile: all of them for an accepted region,
        // else those the stage-4 bounding-box test keeps (bx0 < mxr + 4 and bx1 >= mxr, the same
        // comparisons on the same floats)
        uint32_t cols = 0, rows = 0;
#pragma unroll
        for (int cc = 0; cc < CW; ++cc) {
          const int cx = qx + cc, cy = qy + cc;
          const int mxr = jx * 16 + cx * 4, myr = jy * 16 + cy * 4;
          if (region_full || !(bx0 >= static_cast<float>(mxr + 4) || bx1 < static_cast<float>(mxr))) cols |= 0x1111u << cx;
          if (region_full || !(by0 >= static_cast<float>(myr + 4) || by1 < static_cast<float>(myr))) rows |= 0xFu << (cy * 4);
          if (rox + cx * 4 >= tw) cols &= ~(0x1111u << cx);  // blocks outside the target
          if (roy + cy * 4 >= th) rows &= ~(0xFu << (cy * 4));
        }
        uint32_t blocks = cols & rows;
        while (blocks) {
          const int b16 = __builtin_ctz(blocks);
          blocks &= blocks - 1;
          const int ix4 = b16 & 3, iy4 = b16 >> 2;
          bool block_full = region_full;
          if (!block_full) {
            // stage 4 (subdivide_tile on the 16x16 region); the bounding-box half was applied above
            bool rej = false, nacc = false;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
              float r = (s2x[k] * static_cast<float>(ix4)) + (s2y[k] * static_cast<float>(iy4));
              float a = r + ra2[k];
              rej |= r < ev2q[k];
              nacc |= a < ev2q[k];
            }
            if (rej) continue;
            block_full = !nacc;
          }
          // the block's index in this tile
          const int b = ((rr / RPS) * 4 + iy4 - qy) * NBS + (rr % RPS) * 4 + ix4 - qx;
          if (hiz_on && nearest_key(d3, d4, rox + ix4 * 4, roy + iy4 * 4, 4.0f) > hiz[b]) continue;
          bm |= static_cast<bmask_t>(1) << b;
          if (block_full) fm |= static_cast<bmask_t>(1) << b;
        }
      }
      float4* rs = recs + tid * 4;
      rs[0] = make_float4(e[0], e[1], e[2], e[3]);
      rs[1] = make_float4(e[4], e[5], e[6], e[7]);
      rs[2] = make_float4(e[8], d3.w, d3.y, d3.z);          // z0, zx, zy
      rs[3] = make_float4(d4.x, d4.y, __uint_as_float(id), 0.0f);  // dzx, dzy, id
    }
    // phase 1b: work list of (record, block) pairs spread evenly over the lanes: blocks tested
    // sample by sample first, then blocks accepted whole, so each wave runs one kind
    const bmask_t pm = bm & ~fm;
    const uint32_t np = GT > 16 ? static_cast<uint32_t>(__popcll(static_cast<unsigned long long>(pm))) : __popc(static_cast<uint32_t>(pm));
    const uint32_t nf = GT > 16 ? static_cast<uint32_t>(__popcll(static_cast<unsigned long long>(fm))) : __popc(static_cast<uint32_t>(fm));
    const uint32_t cnt = np | (nf << 16);  // both sums stay below 2^16 (NT * NBS^2 <= 16384)
    const uint32_t incl = wave_incl_scan(cnt);
    if ((tid & 63) == 63) wsum[tid >> 6] = incl;
    __syncthreads();
    if (held) {  // survivors beyond this chunk move to the front
      const uint32_t rest = held > static_cast<uint32_t>(NT) ? held - NT : 0u;
      if (static_cast<uint32_t>(tid) < rest) list[tid] = list[NT + tid];
      held = rest;
    }
    uint32_t off = incl - cnt, total = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (w >= NT / 64) break;
      if (w < (tid >> 6)) off += wsum[w];
      total += wsum[w];
    }
    const uint32_t total_p = total & 0xFFFFu, total_all = total_p + (total >> 16);
    uint32_t off_p = off & 0xFFFFu, off_f = total_p + (off >> 16);
    bmask_t pr = pm, fr = fm;
    while (pr) {
      const uint32_t b = static_cast<uint32_t>(__builtin_ctzll(static_cast<unsigned long long>(pr)));
      pr &= pr - 1;
      work[off_p++] = static_cast<uint16_t>((tid << 7) | (b << 1));
    }
    while (fr) {
      const uint32_t b = static_cast<uint32_t>(__builtin_ctzll(static_cast<unsigned long long>(fr)));
      fr &= fr - 1;
      work[off_f++] = static_cast<uint16_t>((tid << 7) | (b << 1) | 1u);
    }
    __syncthreads();
    // phase 1c: one (record, block) item per lane: coverage, depth and the key atomic-min
    if (depth_keys)
      vis_items<S, GT, true>(P, mode, recs, work, total_p, total_all, keys, d0s, ox, oy, tw, th, tid, NT);
    else if (mode == VIS_LATEST)
      vis_items<S, GT, false>(P, mode, recs, work, total_p, total_all, keys, d0s, ox, oy, tw, th, tid, NT);
  }
  __syncthreads();
  if (ws.parts > 1) {  // one part of a split tile: leave its keys for the merge
    unsigned long long* dst = partial + static_cast<size_t>(ws.slot) * (PX * S);
    for (int i = tid; i < PX * S; i += NT) dst[i] = keys[i];
    return;
  }
  vis_finish<NA, S, SHADE, GT>(P, mode, keys, items, &nitems, ox, oy, NT, tri_rec, tri_attr, SM, wout);
}
// Single draws.  The first `max_parts` workgroups take the parts of split tiles, the others the tiles in
// scheduling order; vis_merge_kernel then finishes the split tiles.
struct vis_lists {
  const uint32_t *order, *vals, *tstart, *tend, *counters;
  const uint4 *parts, *merges;
  unsigned long long* partial;
  uint32_t cap, max_parts, tile_cost;
};
template <int NA, int S, bool SHADE>
__global__ void __launch_bounds__(SRX_VIS_THREADS, 4) vis_kernel(draw_params P, int mode, vis_lists V,
                                                   const float4* __restrict__ tri_rec, const float4* __restrict__ tri_attr,
                                                   const ps_samplers* __restrict__ SM, uint32_t* __restrict__ wout) {
  const uint32_t records = record_total(V.counters);
  if (records > V.cap) return;  // records were dropped: the draw is emitted again
  const uint32_t T = static_cast<uint32_t>(P.gtiles_x * P.gtiles_y);
  const uint32_t part = V.max_parts ? vis_part(P.prim_count, records, busy_tiles(V.counters, T), V.tile_cost) : 0u;
  vis_span ws;
  ws.parts = 1;
  ws.slot = 0;
  const uint32_t b = blockIdx.x;
  if (b < V.max_parts) {
    if (b >= V.counters[CT_PARTS]) return;
    const uint4 e = V.parts[b];
    ws.tile = static_cast<int>(e.x);
    ws.parts = e.z;
    ws.slot = b;
    ws.t0 = V.tstart[e.x] + e.y * part;
    ws.t1 = min(V.tend[e.x], ws.t0 + part);
  } else {
    const uint32_t t = V.order[b - V.max_parts];
    ws.tile = static_cast<int>(t);
    ws.t0 = V.tstart[t];
    ws.t1 = V.tend[t];
    if (V.max_parts && ws.t1 - ws.t0 > part) return;  // its parts take it
  }
  vis_body<NA, S, SHADE, SRX_VIS_THREADS, 16>(P, mode, ws, V.partial, V.vals, tri_rec, tri_attr, SM,
                                              vis_large(records, P.prim_count) ? VIS_FIRST : SRX_VIS_THREADS, wout);
}

// One split tile per workgroup: its keys are the minimum of the parts' keys (each started from the
// target's depth), so the parts' order is immaterial.  512 lanes, as the tiles are few and full: 400 split
// tiles of the textured mesh frame took 84 us with 256, 46 us with 512.
constexpr int VIS_MERGE_THREADS = 512;
template <int NA, int S, bool SHADE>
__global__ void __launch_bounds__(VIS_MERGE_THREADS, 2) vis_merge_kernel(draw_params P, int mode, vis_lists V,
                                                   const float4* __restrict__ tri_rec, const float4* __restrict__ tri_attr,
                                                   const ps_samplers* __restrict__ SM, uint32_t* __restrict__ wout) {
  constexpr int PX = 256;
  __shared__ unsigned long long keys[PX * S];
  __shared__ uint2 items[SHADE ? PX * S : 1];
  __shared__ uint32_t nitems;
  if (blockIdx.x >= V.counters[CT_MERGES]) return;  // the host's count, by steps, is the same
  const uint4 m = V.merges[blockIdx.x];
  const unsigned long long* src = V.partial + static_cast<size_t>(m.z) * (PX * S);
  for (int i = threadIdx.x; i < PX * S; i += VIS_MERGE_THREADS) {
    unsigned long long k = src[i];
    for (uint32_t q = 1; q < m.y; ++q) {
      const unsigned long long kq = src[static_cast<size_t>(q) * (PX * S) + i];
      k = kq < k ? kq : k;
    }
    keys[i] = k;
  }
  if (threadIdx.x == 0) nitems = 0;
  __syncthreads();
  const int ox = static_cast<int>(m.x) % P.gtiles_x * 16, oy = static_cast<int>(m.x) / P.gtiles_x * 16;
  vis_finish<NA, S, SHADE, 16>(P, mode, keys, items, &nitems, ox, oy, VIS_MERGE_THREADS, tri_rec, tri_attr, SM, wout);
}

template <int NA, int S, bool SHADE, int GT>
__global__ void __launch_bounds__(256, 4) vis_batch_kernel(const batch_job* __restrict__ jobs, stage_map m) {
  uint32_t lb, nb;
  const batch_job& J = jobs[stage_job(m, lb, nb)];
  const uint32_t t = J.B.order[lb];
  const vis_span ws{static_cast<int>(t), J.B.tstart[t], J.B.tend[t], 1u, 0u};
  const uint32_t records = J.B.cnt[3 * J.P.prim_count] - J.B.cnt[0];
  vis_body<NA, S, SHADE, 0, GT>(J.P, J.vis_mode, ws, nullptr, J.B.vals[1], J.B.tri_rec, J.B.tri_attr, J.B.samplers,
                                vis_large(records, J.P.prim_count) ? min(VIS_FIRST, blockDim.x) : blockDim.x);
}

// ============================================================== host launchers
// Visibility mode of an opaque early-Z draw for vis_kernel, or -1 when only the in-order kernel
// reproduces the reference (NOT_EQUAL with depth writes).
int vis_mode(const draw_params& P) {
  if (P.vis_stencil && !(P.depth_enable && P.write_depth && (P.depth_func == 1 || P.depth_func == 3 ||
                                                            P.depth_func == 4 || P.depth_func == 6)))
    return -1;  // a stencil mask is expressed through the depth keys only
  if (!P.depth_enable) return VIS_LATEST;
  if (P.depth_func == 0) return VIS_NONE;
  if (!P.write_depth) return VIS_LATEST;
  switch (P.depth_func) {
  case 1: return VIS_LESS;
  case 3: return VIS_LEQUAL;
  case 4: return VIS_GREATER;
  case 6: return VIS_GEQUAL;
  case 2:
  case 7: return VIS_LATEST;  // EQUAL keeps the depth it compares against; ALWAYS ignores it
  default: return -1;
  }
}

bool launch_vis(const draw_params& P, const draw_buffers& B, int which, bool shade, uint32_t records, uint32_t merges,
                hipStream_t s) {
  int mode = vis_mode(P);
  // a SASL pixel shader runs in its own pass (launch_shade) over the winners this pass writes
  uint32_t* const wout = sasl_shades(P) ? B.vis : nullptr;
  if (wout) shade = false;
  uint32_t T = static_cast<uint32_t>(P.gtiles_x * P.gtiles_y);
  if (mode < 0 || P.gt != 16) return false;
  if (!T) return true;
  uint32_t np, nm;
  vis_split_bounds(P.prim_count, records, &np, &nm);
  const vis_lists V{B.order, B.vals[which], B.tstart, B.tend, B.counters, B.vis_parts, B.vis_merges, B.vis_partial,
                    B.list_cap, B.vis_split ? np : 0u, B.tile_cost};
#define SRX_VIS_LAUNCH(NA, S, SH)                                                                                       \
  if (merges)                                                                                                           \
    hipLaunchKernelGGL((vis_merge_kernel<NA, S, SH>), dim3(merges), dim3(VIS_MERGE_THREADS), 0, s, P, mode, V, B.tri_rec, \
                       B.tri_attr, B.samplers, wout);                                                                   \
  else                                                                                                                  \
    hipLaunchKernelGGL((vis_kernel<NA, S, SH>), dim3(np + T), dim3(SRX_VIS_THREADS), 0, s, P, mode, V, B.tri_rec,       \
                       B.tri_attr, B.samplers, wout)
#define SRX_VIS_SHADE(NA)                   \
  switch (P.samples) {                      \
  case 1: SRX_VIS_LAUNCH(NA, 1, true); break; \
  case 2: SRX_VIS_LAUNCH(NA, 2, true); break; \
  default: SRX_VIS_LAUNCH(NA, 4, true); break; \
  }
  if (shade) {
    SRX_NA_DISPATCH(P.nattr, SRX_VIS_SHADE)
  } else {
    switch (P.samples) {
    case 1: SRX_VIS_LAUNCH(1, 1, false); break;
    case 2: SRX_VIS_LAUNCH(1, 2, false); break;
    default: SRX_VIS_LAUNCH(1, 4, false); break;
    }
  }
#undef SRX_VIS_SHADE
#undef SRX_VIS_LAUNCH
  return true;
}

bool vis_applicable(const draw_params& P) { return vis_mode(P) >= 0 && P.gt == 16; }

// GPU tiles of 8 and 32 pixels are built for single-sample draws; every variant must fit 64 KB of LDS.
bool vis_batch_supported(int samples, bool shade, int threads, int gt) {
  if (!(threads == 64 || threads == 128 || threads == 256)) return false;
  if (gt != 16 && !(gt == 8 || gt == 32)) return false;
  if (gt != 16 && samples != 1) return false;
  return vis_static_bytes(samples, gt) + vis_union_bytes(threads, samples, shade, gt) <= 65536;
}
bool launch_vis_batch(int na, int samples, bool shade, int threads, int gt, const batch_job* jobs, stage_map m,
                      uint32_t blocks, hipStream_t s) {
  if (!vis_batch_supported(samples, shade, threads, gt)) return false;
  if (!blocks) return true;
  const size_t lds = static_cast<size_t>(vis_union_bytes(threads, samples, shade, gt));
#define SRX_VIS_B(NA, S, SH, GT) \
  hipLaunchKernelGGL((vis_batch_kernel<NA, S, SH, GT>), dim3(blocks), dim3(threads), lds, s, jobs, m)
#define SRX_VIS_BS(NA)                       \
  switch (samples) {                         \
  case 1: SRX_VIS_B(NA, 1, true, 16); break; \
  case 2: SRX_VIS_B(NA, 2, true, 16); break; \
  default: SRX_VIS_B(NA, 4, true, 16); break; \
  }
#define SRX_VIS_B8(NA) SRX_VIS_B(NA, 1, true, 8)
#define SRX_VIS_B32(NA) SRX_VIS_B(NA, 1, true, 32)
  if (gt == 8) {
    if (shade) {
      SRX_NA_DISPATCH_BATCH(na, SRX_VIS_B8)
    } else {
      SRX_VIS_B(1, 1, false, 8);
    }
  } else if (gt == 32) {
    if (shade) {
      SRX_NA_DISPATCH_BATCH(na, SRX_VIS_B32)
    } else {
      SRX_VIS_B(1, 1, false, 32);
    }
  } else if (shade) {
    SRX_NA_DISPATCH_BATCH(na, SRX_VIS_BS)
  } else {
    switch (samples) {
    case 1: SRX_VIS_B(1, 1, false, 16); break;
    case 2: SRX_VIS_B(1, 2, false, 16); break;
    default: SRX_VIS_B(1, 4, false, 16); break;
    }
  }
#undef SRX_VIS_B32
#undef SRX_VIS_B8
#undef SRX_VIS_BS
#undef SRX_VIS_B
  return true;
}
}  // namespace srx
