// Draws whose samples depend on primitive order (blending, stencil that changes): one 16x16 GPU tile per
// workgroup, one pixel per lane.
#include "srx_kernel_common.h"

namespace srx {

hipError_t upload_ewa_table_inorder(const float* table256, hipStream_t s) {
  return hipMemcpyToSymbolAsync(HIP_SYMBOL(c_ewa), table256, 256 * sizeof(float), 0, hipMemcpyHostToDevice, s);
}

// RGBA8 / BGRA8 texels held as one word per sample (the values load_texel / store_texel give)
__device__ __forceinline__ float4 unpack_texel(int pf, uint32_t u) {
  const float inv = 1.0f / 255;
  const float b0 = (u & 0xFF) * inv, b1 = ((u >> 8) & 0xFF) * inv, b2 = ((u >> 16) & 0xFF) * inv, b3 = (u >> 24) * inv;
  return pf == PF_RGBA8 ? make_float4(b0, b1, b2, b3) : make_float4(b2, b1, b0, b3);
}
__device__ __forceinline__ uint32_t pack_texel(int pf, float4 c) {
  const uint32_t x = unorm8(c.x), y = unorm8(c.y), z = unorm8(c.z), w = unorm8(c.w);
  return (pf == PF_RGBA8 ? x | (z << 16) : z | (x << 16)) | (y << 8) | (w << 24);
}

// S consecutive 4-byte or 8-byte samples of a pixel as one wide access (a pixel's samples start at a
// multiple of their size: surfaces are allocated at 256-byte alignment)
template <int S>
__device__ __forceinline__ void load_words(const uint8_t* p, uint32_t (&w)[S]) {
  if constexpr (S == 4) {
    const uint4 q = *reinterpret_cast<const uint4*>(p);
    w[0] = q.x; w[1] = q.y; w[2] = q.z; w[3] = q.w;
  } else if constexpr (S == 2) {
    const uint2 q = *reinterpret_cast<const uint2*>(p);
    w[0] = q.x; w[1] = q.y;
  } else {
    w[0] = *reinterpret_cast<const uint32_t*>(p);
  }
}
template <int S>
__device__ __forceinline__ void store_words(uint8_t* p, const uint32_t (&w)[S]) {
  if constexpr (S == 4) *reinterpret_cast<uint4*>(p) = make_uint4(w[0], w[1], w[2], w[3]);
  else if constexpr (S == 2) *reinterpret_cast<uint2*>(p) = make_uint2(w[0], w[1]);
  else *reinterpret_cast<uint32_t*>(p) = w[0];
}

// One 16x16 GPU tile per workgroup; its records (in primitive order) in chunks of 64:
//  1. four lanes per record, one per row of 4x4 blocks: the reference's stage-16 and stage-4 decisions;
//     partially covered blocks go to an LDS list, blocks accepted whole set the record's bit in the
//     block's mask;
//  2. one listed (record, block) per lane: the covered samples of its 16 pixels (4 bits each) and the
//     record's bit in the mask of every pixel that has one;
//  3. one pixel per lane: the lane walks its own records in primitive order with its samples' depth,
//     stencil and (8-bit colour formats) colour in registers, tests each against them, and shades and
//     blends those that pass.  Lanes of a wave are at different records at the same time.
// Measured (32k blended, trilinearly textured triangles over most of 1280x720, 4 samples): this kernel
// 0.14 ms, the whole frame 0.14-0.24 ms (among others, alone); a wave walking the records together, with only the lanes of
// the current record's quads shading and every blend a round trip to the target, 4.2 ms (frame 4.0-4.2).
// It is bound by the pixel shader's latency at the 2 waves per SIMD its registers leave (229 for two
// attributes and 4 samples; capping them for 3 or 4 waves cost the textured frame 8 and 33% and gained
// the nine-tap shadow frame 1 and 2%) and by the deepest pixel of each wave.
constexpr int IO_CHUNK = 64;
template <int NA, int S>
__global__ void __launch_bounds__(256) inorder_kernel(draw_params P, const ps_samplers* __restrict__ SM,
                                                      const uint32_t* __restrict__ order, const uint32_t* __restrict__ vals,
                                                      const uint32_t* __restrict__ tstart, const uint32_t* __restrict__ tend,
                                                      const float4* __restrict__ tri_rec, const float4* __restrict__ tri_attr,
                                                      const uint32_t* __restrict__ counters, uint32_t cap) {
  if (record_total(counters) > cap) return;  // records were dropped: the draw is emitted again
  __shared__ float4 recs[IO_CHUNK * 4];            // edges, depth plane, id << 1 | front
  __shared__ unsigned long long cov[IO_CHUNK][16];  // covered samples of a record's block, 4 bits a pixel
  __shared__ unsigned long long pmask[256];         // records with a covered sample in the pixel (partial blocks)
  __shared__ unsigned long long fmask[16];          // records that cover the block whole
  __shared__ uint16_t work[IO_CHUNK * 16];
  __shared__ uint32_t nwork;
  const int gtile = static_cast<int>(order[blockIdx.x]);
  const uint32_t t0 = tstart[gtile], t1 = tend[gtile];
  if (t0 == t1 && !P.clear_ds && !P.clear_color) return;
  const int tid = threadIdx.x;
  const int ox = (gtile % P.gtiles_x) * 16, oy = (gtile / P.gtiles_x) * 16;
  const int t64x = ox & ~(TILE - 1), t64y = oy & ~(TILE - 1);
  const int tw = static_cast<int>(P.target_w), th = static_cast<int>(P.target_h);
  const int blk = tid >> 4, lp = tid & 15;  // this lane's 4x4 block and its pixel in it
  const int px = ox + (blk & 3) * 4 + (lp & 3), py = oy + (blk >> 2) * 4 + (lp >> 2);
  const bool pin = px < tw && py < th;
  const bool has_ds = P.ds.data != nullptr;
  const bool colored = P.color.data != nullptr && P.blend_id != BLEND_DISABLED;
  const bool packed = P.color.pf == PF_RGBA8 || P.color.pf == PF_BGRA8;
  // the pixel's samples: (depth, stencil) pairs and colour words
  float depth[S];
  uint32_t stencil[S], color[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    depth[s] = 0.0f;
    stencil[s] = 0;
    color[s] = 0;
  }
  if (pin) {
    if (P.clear_ds) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        depth[s] = P.clear_depth;
        stencil[s] = P.clear_stencil;
      }
    } else if (has_ds) {
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const float2 d = *reinterpret_cast<const float2*>(sample_addr(P.ds, px, py, s));
        depth[s] = d.x;
        stencil[s] = __float_as_uint(d.y);
      }
    }
    if (P.clear_color) {
      const uint32_t c = pack_texel(P.color.pf, make_float4(P.clear_rgba[0], P.clear_rgba[1], P.clear_rgba[2], P.clear_rgba[3]));
#pragma unroll
      for (int s = 0; s < S; ++s) color[s] = c;
    } else if (colored && packed) {
      load_words<S>(sample_addr(P.color, px, py, 0), color);
    }
  }
  // Stencil changes only where the stencil test passes, so a tile none of whose samples passes it now
  // can never pass it during this draw: nothing in the tile changes.
  bool live = t0 != t1;
  if (live && P.stencil_enable) {
    int can = 0;
    if (pin)
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const uint32_t os = stencil[s] & P.read_mask;
        can |= cmpu(P.st_func[0], P.stencil_ref, os) || cmpu(P.st_func[1], P.stencil_ref, os);
      }
    live = __syncthreads_or(can) != 0;
    if (!live && !P.clear_ds && !P.clear_color) return;
  }
  bool drawn = false;  // the pixel's colour words changed
  const int jx = (ox - t64x) >> 4, jy = (oy - t64y) >> 4;  // the tile's stage-16 region of its 64x64 tile
  const float tvx = static_cast<float>(t64x), tvy = static_cast<float>(t64y);
  const uint32_t full_px = (1u << S) - 1u;
  constexpr unsigned long long ALL = S == 4 ? ~0ull : S == 2 ? 0x3333333333333333ull : 0x1111111111111111ull;
  if (live)
    for (uint32_t c0 = t0; c0 < t1; c0 += IO_CHUNK) {
      __syncthreads();  // the previous chunk's masks are walked
      pmask[tid] = 0;
      if (tid < 16) fmask[tid] = 0;
      if (tid == 0) nwork = 0;
      __syncthreads();
      // 1. record r, block row by: the blocks of the row it reaches
      const int r = tid >> 2, by = tid & 3;
      const uint32_t ri = c0 + static_cast<uint32_t>(r);
      if (ri < t1) {
        const uint32_t rec = vals[ri];
        const uint32_t id = rec >> 1;
        const float4* tr = tri_rec + tri_slot(P, id) * 5;
        float e[9], bb[4];
        read_tri_rec(tr, e, bb);
        if (by == 0) {
          const float4 d3 = tr[3], d4 = tr[4];
          recs[r * 4 + 0] = make_float4(e[0], e[1], e[2], e[3]);
          recs[r * 4 + 1] = make_float4(e[4], e[5], e[6], e[7]);
          recs[r * 4 + 2] = make_float4(e[8], d3.w, d3.y, d3.z);  // z0, zx, zy
          recs[r * 4 + 3] = make_float4(d4.x, d4.y, __uint_as_float(id), d4.z);
        }
        const float bx0 = bb[0] - tvx, bx1 = bb[1] - tvx, by0 = bb[2] - tvy, by1 = bb[3] - tvy;
        // per-stage constants (rasterize_triangle, rasterizer.cpp:662-675, 704-710)
        float s2x[3], s2y[3], ra2[3], ev2q[3];
        bool rej = false, nacc = false;
        const float lf = static_cast<float>(ox), tf = static_cast<float>(oy);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const float ex = e[k * 3], ey = e[k * 3 + 1], ez = e[k * 3 + 2];
          float sx = TILE * ex, sy = TILE * ey;
          float ra = -fabsf(sx) - fabsf(sy);
          float part = static_cast<float>((ex > 0) * TILE) * ex + static_cast<float>((ey > 0) * TILE) * ey;
          sx *= 0.25f; sy *= 0.25f; ra *= 0.25f; part *= 0.25f;
          // stage 16 (subdivide_tile on the 64x64 tile)
          const float ev = (ez - part) - ((tvx * ex) + (tvy * ey));
          const float rr = (sx * static_cast<float>(jx)) + (sy * static_cast<float>(jy));
          rej |= rr < ev;
          nacc |= rr + ra < ev;
          sx *= 0.25f; sy *= 0.25f; ra *= 0.25f; part *= 0.25f;
          s2x[k] = sx; s2y[k] = sy; ra2[k] = ra;
          ev2q[k] = (ez - part) - ((lf * ex) + (tf * ey));
        }
        rej |= bx0 >= static_cast<float>(jx * 16 + 16);
        rej |= bx1 < static_cast<float>(jx * 16);
        rej |= by0 >= static_cast<float>(jy * 16 + 16);
        rej |= by1 < static_cast<float>(jy * 16);
        const bool tile_full = (rec & 1) != 0;  // the record covers its whole 64x64 tile
        const bool region_full = tile_full || !nacc;
        if ((tile_full || !rej) && oy + by * 4 < th) {
          const int myr = jy * 16 + by * 4;
          const bool row_in = !(by0 >= static_cast<float>(myr + 4) || by1 < static_cast<float>(myr));
#pragma unroll
          for (int bx = 0; bx < 4; ++bx) {
            bool block_full = region_full, keep = true;
            if (!region_full) {
              // stage 4 (subdivide_tile on the 16x16 region)
              const int mxr = jx * 16 + bx * 4;
              keep = row_in && !(bx0 >= static_cast<float>(mxr + 4) || bx1 < static_cast<float>(mxr));
              bool na = false;
#pragma unroll
              for (int k = 0; k < 3; ++k) {
                const float rr = (s2x[k] * static_cast<float>(bx)) + (s2y[k] * static_cast<float>(by));
                keep &= !(rr < ev2q[k]);
                na |= rr + ra2[k] < ev2q[k];
              }
              block_full = !na;
            }
            if (!keep || ox + bx * 4 >= tw) continue;
            const int b = by * 4 + bx;
            if (block_full) {
              cov[r][b] = ALL;
              atomicOr(&fmask[b], 1ull << r);
            } else {
              work[atomicAdd(&nwork, 1u)] = static_cast<uint16_t>((r << 4) | b);
            }
          }
        }
      }
      __syncthreads();
      // 2. draw_partial_tile's samples of one block (rasterizer.cpp:298-439)
      const uint32_t nw = nwork;
      for (uint32_t wi = tid; wi < nw; wi += 256) {
        const uint32_t wk = work[wi];
        const int rw = static_cast<int>(wk >> 4), b = static_cast<int>(wk & 15u);
        const float4 r0 = recs[rw * 4 + 0], r1 = recs[rw * 4 + 1];
        const float e[9] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w, recs[rw * 4 + 2].x};
        const float Bx = static_cast<float>(ox + (b & 3) * 4), By = static_cast<float>(oy + (b >> 2) * 4);
        float evp[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) evp[k] = e[k * 3 + 2] - ((Bx * e[k * 3]) + (By * e[k * 3 + 1]));
        unsigned long long m = 0;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          const float fx = static_cast<float>(q & 3), fy = static_cast<float>(q >> 2);
          uint32_t pm = 0;
#pragma unroll
          for (int s = 0; s < S; ++s) {
            const float mx = P.sp[s][0] + fx, my = P.sp[s][1] + fy;
            bool out = false;
#pragma unroll
            for (int k = 0; k < 3; ++k) out |= ((mx * e[k * 3]) + (my * e[k * 3 + 1])) < evp[k];
            if (!out) pm |= 1u << s;
          }
          m |= static_cast<unsigned long long>(pm) << (4 * q);
          if (pm) atomicOr(&pmask[b * 16 + q], 1ull << rw);
        }
        cov[rw][b] = m;
      }
      __syncthreads();
      // 3. this pixel's records in primitive order
      unsigned long long m = pin ? pmask[tid] | fmask[blk] : 0ull;
      while (true) {
        uint32_t passed = 0, id = 0;
        float nd[S];
        bool front = false;
        while (m) {
          const int rw = __builtin_ctzll(m);
          m &= m - 1;
          const uint32_t c = static_cast<uint32_t>(cov[rw][blk] >> (4 * lp)) & full_px;
          const float4 r2 = recs[rw * 4 + 2], r3 = recs[rw * 4 + 3];
          id = __float_as_uint(r3.z);
          front = r3.w != 0.0f;
          // depth of the quad chain (step_2d_unproj_pos_quad, z lane)
          const float dx = (0.5f + static_cast<float>(px & ~1)) - r2.z;
          const float dy = (0.5f + static_cast<float>(py & ~1)) - r2.w;
          float z = r2.y + ((r3.x * dx) + (r3.y * dy));
          z = (px & 1) ? z + r3.x : z;
          z = (py & 1) ? z + r3.y : z;
          // the depth and stencil tests of a sample depend only on that sample (framebuffer.cpp:445-479,
          // 522-614), not on the colour, and the shaders never discard: they run before the shader
          const int face = front ? 0 : 1;
#pragma unroll
          for (int s = 0; s < S; ++s) {
            nd[s] = (S > 1) ? z + ((P.sp[s][0] - 0.5f) * r3.x + (P.sp[s][1] - 0.5f) * r3.y) : z;
            const bool dp = !(has_ds && P.depth_enable) || cmpf(P.depth_func, nd[s], P.read_depth ? depth[s] : 0.0f);
            const bool sp = !P.stencil_enable || cmpu(P.st_func[face], P.stencil_ref, stencil[s] & P.read_mask);
            if (((c >> s) & 1u) && dp && sp) passed |= 1u << s;
          }
          if (passed) break;
        }
        if (!passed) break;
#pragma unroll
        for (int s = 0; s < S; ++s)
          if ((passed >> s) & 1u) {
            if (P.write_depth) depth[s] = nd[s];
            if (P.stencil_enable)
              stencil[s] = stencil_op(P.st_pass_op[front ? 0 : 1], P.stencil_ref, stencil[s] & P.read_mask) & P.write_mask;
          }
        if (!colored) continue;
        attr_setup<NA> at;
        load_attr<NA>(P, tri_attr, id, at);
        const quad_lazy<NA> q(at, P, px & ~1, py & ~1);
        const float4 src = run_ps_pixel<NA>(P, SM, q, (px & 1) | ((py & 1) << 1));
        if (packed) {
          drawn = true;
          const uint32_t flat = P.blend_id == BLEND_OFF ? pack_texel(P.color.pf, src) : 0u;
#pragma unroll
          for (int s = 0; s < S; ++s)
            if ((passed >> s) & 1u)
              color[s] = P.blend_id == BLEND_OFF ? flat
                                                 : pack_texel(P.color.pf, lerp4(unpack_texel(P.color.pf, color[s]), src, src.w));
        } else {
          for (int s = 0; s < S; ++s)
            if ((passed >> s) & 1u) blend_store(P, px, py, s, src);
        }
      }
    }
  if (!pin) return;
  if (P.clear_ds || (live && has_ds && (P.write_depth || P.stencil_enable))) {
#pragma unroll
    for (int s = 0; s < S; ++s)
      *reinterpret_cast<float2*>(sample_addr(P.ds, px, py, s)) = make_float2(depth[s], __uint_as_float(stencil[s]));
  }
  if (P.clear_color || drawn) store_words<S>(sample_addr(P.color, px, py, 0), color);
}

bool inorder_applicable(const draw_params& P) {
  const bool deferred = P.early_z && (P.blend_id == BLEND_OFF || P.blend_id == BLEND_DISABLED);
  return P.gt == 16 && !P.count_stats && !deferred && !sasl_shades(P);
}

// A pending colour clear can start the tiles' colour words (8-bit formats whose colour the draw writes).
bool inorder_takes_color_clear(const draw_params& P) {
  return P.color.data != nullptr && P.blend_id != BLEND_DISABLED && (P.color.pf == PF_RGBA8 || P.color.pf == PF_BGRA8);
}

void launch_inorder(const draw_params& P, const draw_buffers& B, int which, hipStream_t s) {
  const uint32_t T = static_cast<uint32_t>(P.gtiles_x * P.gtiles_y);
  if (!T) return;
#define SRX_INORDER_S(NA, S)                                                                                            \
  hipLaunchKernelGGL((inorder_kernel<NA, S>), dim3(T), dim3(256), 0, s, P, B.samplers, B.order, B.vals[which], B.tstart, \
                     B.tend, B.tri_rec, B.tri_attr, B.counters, B.list_cap)
#define SRX_INORDER(NA)                  \
  switch (P.samples) {                   \
  case 1: SRX_INORDER_S(NA, 1); break;   \
  case 2: SRX_INORDER_S(NA, 2); break;   \
  default: SRX_INORDER_S(NA, 4); break;  \
  }
  SRX_NA_DISPATCH(P.nattr, SRX_INORDER)
#undef SRX_INORDER
#undef SRX_INORDER_S
}

}  // namespace srx
