// In-order rasterisation of the draws that inorder_kernel (srx_inorder.hip) does not take: statistics
// queries, SASL pixel shaders, 32-pixel tiles, NOT_EQUAL depth; and the deferred pixel shader passes over
// the winners of an opaque draw.
#include "srx_kernel_common.h"
#include "srx_sasl_exec.h"

namespace srx {

hipError_t upload_ewa_table_raster(const float* table256, hipStream_t s) {
  return hipMemcpyToSymbolAsync(HIP_SYMBOL(c_ewa), table256, 256 * sizeof(float), 0, hipMemcpyHostToDevice, s);
}

// ============================================================== raster
struct prim_lds {
  float e[9];
  float bb[4];     // relative to the 64x64 tile origin
  float ev1[3];    // stage-16 rejection value, already offset by the 64x64 tile origin
  float s1x[3], s1y[3], ra1[3];
  float ev2[3], s2x[3], s2y[3], ra2[3];
  float zx, zy, z0, dzx, dzy;
  float aa[4];
  uint32_t idf;    // triangle id << 1 | tile-level accept
  uint32_t r16;    // bit k: 16x16 region k of the GPU tile rejected; bit 16+k: accepted
  uint32_t front;
};

// Pixel shader and backend for one triangle on a 2x2 quad: `pm` holds the samples to store, bits
// 4i..4i+S-1 for pixel i.  Interpolants are formed per pixel where read (quad_lazy), so only one
// pixel's registers are live at a time; the colour of each pixel is the quad shader's.
template <int NA, int S, bool SASL = false>
__device__ __forceinline__ void shade_store(const draw_params& P, const ps_samplers* __restrict__ SM,
                                         const float4* __restrict__ tri_attr, uint32_t id, int px0, int py0, uint32_t pm) {
  attr_setup<NA> at;
  load_attr<NA>(P, tri_attr, id, at);
  const quad_lazy<NA> q(at, P, px0, py0);
  if constexpr (SASL) {
    // pixel_shader_unit::update + execute (shader_unit.cpp:106-176) on the whole quad: input i is
    // attribute inputs[i].attr of each pixel, the program runs the four pixels together
    const sasl_program* __restrict__ prog = P.sasl;
    sasl_regs R;
    const uint32_t nregs = prog->nregs;
    for (uint32_t r = 0; r < nregs; ++r)
      for (int px = 0; px < 4; ++px) R.r[r][px] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const uint32_t nin = prog->ninputs;
    for (int px = 0; px < 4; ++px) {
      const float iw = q.inv_w(px);
      for (uint32_t k = 0; k < nin; ++k) {
        const sasl_input inp = prog->inputs[k];
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
        for (int a = 0; a < NA; ++a)
          if (a == inp.attr) v = q.reg(a + 1, px, iw);
        R.r[inp.reg][px] = make_float4(v.x, inp.ncomp > 1 ? v.y : 0.0f, inp.ncomp > 2 ? v.z : 0.0f, inp.ncomp > 3 ? v.w : 0.0f);
      }
    }
    sasl_exec(prog, R, [&](int slot, int, float u, float v, float dxu, float dxv, float dyu, float dyv) -> float4 {
      if (!P.has_sampler[slot]) return make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      const sampler_desc_dev& sp = SM->s[slot];
      return sample_grad(sp, u, v, dxu, dxv, dyu, dyv);
    });
    for (int i = 0; i < 4; ++i) {
      const uint32_t m = (pm >> (4 * i)) & 15u;
      if (!m) continue;
      const float4 c = sasl_color0(prog, R, i);
      for (int s = 0; s < S; ++s)
        if (m & (1u << s)) blend_store(P, px0 + (i & 1), py0 + (i >> 1), s, c);
    }
    return;
  }
#pragma unroll 1
  for (int i = 0; i < 4; ++i) {
    const uint32_t m = (pm >> (4 * i)) & 15u;
    if (!m) continue;
    const float4 c = run_ps_pixel<NA>(P, SM, q, i);
    for (int s = 0; s < S; ++s)
      if (m & (1u << s)) blend_store(P, px0 + (i & 1), py0 + (i >> 1), s, c);
  }
}

// One workgroup per GPU tile, one thread per 2x2 quad.  VIS: opaque early-Z draws -- record for every
// sample the last triangle that passed (the colour it ends with) into `vis`; the pixel shader runs
// later in shade_kernel.  Otherwise every quad runs the pixel shader and the backend in primitive order.
template <int NA, int S, bool VIS, bool SASL = false>
__global__ void __launch_bounds__(256) raster_kernel(draw_params P, const ps_samplers* __restrict__ SM,
                                                      const uint32_t* __restrict__ order, const uint32_t* __restrict__ vals,
                                                      const uint32_t* __restrict__ tstart, const uint32_t* __restrict__ tend,
                                                      const float4* __restrict__ tri_rec, const float4* __restrict__ tri_attr,
                                                      uint32_t* __restrict__ vis, unsigned long long* __restrict__ partial,
                                                      const uint32_t* __restrict__ counters, uint32_t cap) {
  if (record_total(counters) > cap) {  // records were dropped: the draw is emitted again
    if (P.count_stats) block_partial(partial, 0ull);
    return;
  }
  extern __shared__ prim_lds lds[];
  const int G = P.gt, QW = G / 2;
  const int gtile = static_cast<int>(order[blockIdx.x]);
  const int gx = gtile % P.gtiles_x, gy = gtile / P.gtiles_x;
  const int tid = threadIdx.x, nthreads = blockDim.x;
  const int qx = tid % QW, qy = tid / QW;
  const int px0 = gx * G + qx * 2, py0 = gy * G + qy * 2;  // quad origin
  const int t64x = (gx * G) & ~(TILE - 1), t64y = (gy * G) & ~(TILE - 1);
  const int tw = static_cast<int>(P.target_w), th = static_cast<int>(P.target_h);
  // pixel i of the quad: (px0 + (i & 1), py0 + (i >> 1))
  bool pin[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) pin[i] = (px0 + (i & 1)) < tw && (py0 + (i >> 1)) < th;

  // depth/stencil of the quad's samples, held in registers for the whole tile
  // VIS draws have stencil off, so only depth is kept (and written back)
  float depth[4][S];
  uint32_t stencil[4][VIS ? 1 : S];
  uint32_t winner[4][VIS ? S : 1];
  const bool has_ds = P.ds.data != nullptr;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int s = 0; s < S; ++s) {
      depth[i][s] = 0.0f;
      if constexpr (!VIS) stencil[i][s] = 0;
      if constexpr (VIS) winner[i][s] = NO_WINNER;
      if (has_ds && pin[i]) {
        if constexpr (VIS) {
          depth[i][s] = *reinterpret_cast<const float*>(sample_addr(P.ds, px0 + (i & 1), py0 + (i >> 1), s));
        } else {
          float2 d = *reinterpret_cast<const float2*>(sample_addr(P.ds, px0 + (i & 1), py0 + (i >> 1), s));
          depth[i][s] = d.x;
          stencil[i][s] = __float_as_uint(d.y);
        }
      }
    }
  if constexpr (!VIS) {
    // Stencil changes only where the stencil test passes, so a tile none of whose samples passes it
    // now can never pass it during this draw: nothing in the tile changes (exact early-out, taken
    // only when no statistics are counted).
    if (P.stencil_enable && !P.count_stats) {
      int can = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int s = 0; s < S; ++s)
          if (pin[i]) {
            const uint32_t os = stencil[i][s] & P.read_mask;
            can |= cmpu(P.st_func[0], P.stencil_ref, os) || cmpu(P.st_func[1], P.stencil_ref, os);
          }
      if (!__syncthreads_or(can)) return;
    }
  }
  const bool any_in = pin[0];
  unsigned long long ps_inv = 0, be_pix = 0;
  const uint32_t full_px = (S == 1) ? 1u : (S == 2 ? 3u : 15u);

  const uint32_t t0 = tstart[gtile], t1 = tend[gtile];
  // 16x16, 4x4 regions of this quad inside its 64x64 tile
  const int rx64 = px0 - t64x, ry64 = py0 - t64y;
  const int ix16 = rx64 >> 4, iy16 = ry64 >> 4;
  const int r16k = ((py0 - gy * G) >> 4) * (G / 16) + ((px0 - gx * G) >> 4);
  const int R16x = t64x + ix16 * 16, R16y = t64y + iy16 * 16;
  const int ix4 = (px0 - R16x) >> 2, iy4 = (py0 - R16y) >> 2;
  const int Bx = R16x + ix4 * 4, By = R16y + iy4 * 4;

  for (uint32_t base = t0; base < t1; base += nthreads) {
    uint32_t nb = min(static_cast<uint32_t>(nthreads), t1 - base);
    if (tid < static_cast<int>(nb)) {
      prim_lds& L = lds[tid];
      uint32_t rec = vals[base + tid];
      uint32_t id = rec >> 1;
      const float4* tr = tri_rec + tri_slot(P, id) * 5;
      float e[9], bb[4];
      read_tri_rec(tr, e, bb);
      float4 d3 = tr[3], d4 = tr[4];
      for (int k = 0; k < 9; ++k) L.e[k] = e[k];
      const float tvx = static_cast<float>(t64x), tvy = static_cast<float>(t64y);
      L.bb[0] = bb[0] - tvx;
      L.bb[1] = bb[1] - tvx;
      L.bb[2] = bb[2] - tvy;
      L.bb[3] = bb[3] - tvy;
      // per-stage constants (rasterize_triangle, rasterizer.cpp:662-675, 704-710)
      for (int k = 0; k < 3; ++k) {
        float ex = e[k * 3], ey = e[k * 3 + 1], ez = e[k * 3 + 2];
        bool mx = ex > 0, my = ey > 0;
        float sx = TILE * ex, sy = TILE * ey;
        float ra = -fabsf(sx) - fabsf(sy);
        float part = static_cast<float>(mx * TILE) * ex + static_cast<float>(my * TILE) * ey;
        sx *= 0.25f; sy *= 0.25f; ra *= 0.25f; part *= 0.25f;
        float ev = ez - part;
        L.s1x[k] = sx; L.s1y[k] = sy; L.ra1[k] = ra;
        L.ev1[k] = ev - ((tvx * ex) + (tvy * ey));
        sx *= 0.25f; sy *= 0.25f; ra *= 0.25f; part *= 0.25f;
        L.s2x[k] = sx; L.s2y[k] = sy; L.ra2[k] = ra;
        L.ev2[k] = ez - part;
      }
      L.zx = d3.y;
      L.zy = d3.z;
      L.z0 = d3.w;
      L.dzx = d4.x;
      L.dzy = d4.y;
      L.front = d4.z != 0.0f;
      for (int s = 0; s < 4; ++s) L.aa[s] = (S > 1 && s < S) ? (P.sp[s][0] - 0.5f) * d4.x + (P.sp[s][1] - 0.5f) * d4.y : 0.0f;
      L.idf = rec;
      // stage-16 decision for each 16x16 region of the GPU tile (subdivide_tile, SSE order)
      uint32_t bits = 0;
      int nreg = G / 16;
      for (int ry = 0; ry < nreg; ++ry)
        for (int rx = 0; rx < nreg; ++rx) {
          int jx = ((gx * G - t64x) >> 4) + rx, jy = ((gy * G - t64y) >> 4) + ry;
          bool rej = false, nacc = false;
          for (int k = 0; k < 3; ++k) {
            float r = (L.s1x[k] * static_cast<float>(jx)) + (L.s1y[k] * static_cast<float>(jy));
            float a = r + L.ra1[k];
            rej |= r < L.ev1[k];
            nacc |= a < L.ev1[k];
          }
          int mxr = jx * 16, myr = jy * 16;
          rej |= L.bb[0] >= static_cast<float>(mxr + 16);
          rej |= L.bb[1] < static_cast<float>(mxr);
          rej |= L.bb[2] >= static_cast<float>(myr + 16);
          rej |= L.bb[3] < static_cast<float>(myr);
          int k = ry * nreg + rx;
          if (rej) bits |= 1u << k;
          else if (!nacc) bits |= 1u << (16 + k);
        }
      L.r16 = bits;
    }
    __syncthreads();
    if (any_in) {
      for (uint32_t j = 0; j < nb; ++j) {
        const prim_lds& L = lds[j];
        uint32_t cov[4];
        if (L.idf & 1) {
          cov[0] = cov[1] = cov[2] = cov[3] = full_px;
        } else {
          uint32_t bits = L.r16;
          if (bits & (1u << r16k)) continue;
          if (bits & (1u << (16 + r16k))) {
            cov[0] = cov[1] = cov[2] = cov[3] = full_px;
          } else {
            // stage 4: child (ix4, iy4) of the 16x16 region at (R16x, R16y)
            bool rej = false, nacc = false;
            const float lf = static_cast<float>(R16x), tf = static_cast<float>(R16y);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
              float ev = L.ev2[k] - ((lf * L.e[k * 3]) + (tf * L.e[k * 3 + 1]));
              float r = (L.s2x[k] * static_cast<float>(ix4)) + (L.s2y[k] * static_cast<float>(iy4));
              float a = r + L.ra2[k];
              rej |= r < ev;
              nacc |= a < ev;
            }
            int mxr = ix16 * 16 + ix4 * 4, myr = iy16 * 16 + iy4 * 4;
            rej |= L.bb[0] >= static_cast<float>(mxr + 4);
            rej |= L.bb[1] < static_cast<float>(mxr);
            rej |= L.bb[2] >= static_cast<float>(myr + 4);
            rej |= L.bb[3] < static_cast<float>(myr);
            if (rej) continue;
            if (!nacc) {
              cov[0] = cov[1] = cov[2] = cov[3] = full_px;
            } else {
              // pixel level: draw_partial_tile on the 4x4 block at (Bx, By)
              float evp[3];
              const float bl = static_cast<float>(Bx), bt = static_cast<float>(By);
#pragma unroll
              for (int k = 0; k < 3; ++k) evp[k] = L.e[k * 3 + 2] - ((bl * L.e[k * 3]) + (bt * L.e[k * 3 + 1]));
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                uint32_t m = 0;
                const float fx = static_cast<float>(px0 + (i & 1) - Bx), fy = static_cast<float>(py0 + (i >> 1) - By);
#pragma unroll
                for (int s = 0; s < S; ++s) {
                  float mx = P.sp[s][0] + fx, my = P.sp[s][1] + fy;
                  bool r = false;
#pragma unroll
                  for (int k = 0; k < 3; ++k) r |= ((mx * L.e[k * 3]) + (my * L.e[k * 3 + 1])) < evp[k];
                  if (!r) m |= 1u << s;
                }
                cov[i] = m;
              }
            }
          }
        }
        // pixels outside the render target are never drawn
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (!pin[i]) cov[i] = 0;
        if ((cov[0] | cov[1] | cov[2] | cov[3]) == 0) continue;
        // depth of the quad's pixels (step_2d_unproj_pos_quad, z lane)
        const float dx = (0.5f + static_cast<float>(px0)) - L.zx;
        const float dy = (0.5f + static_cast<float>(py0)) - L.zy;
        float z[4];
        z[0] = L.z0 + ((L.dzx * dx) + (L.dzy * dy));
        z[1] = z[0] + L.dzx;
        z[2] = z[0] + L.dzy;
        z[3] = z[1] + L.dzy;
        const uint32_t id = L.idf >> 1;
        if (P.early_z) {
          // early_z_test (framebuffer.cpp:522-614): depth written at test time
          uint32_t tested[4] = {0, 0, 0, 0};
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int s = 0; s < S; ++s) {
              if (!(cov[i] & (1u << s))) continue;
              float nd = (S > 1) ? (L.aa[s] + z[i]) : z[i];
              float od = P.read_depth ? depth[i][s] : 0.0f;
              bool pass = P.depth_enable ? cmpf(P.depth_func, nd, od) : true;
              if (pass) {
                if (P.write_depth) depth[i][s] = nd;
                tested[i] |= 1u << s;
              }
            }
          if ((tested[0] | tested[1] | tested[2] | tested[3]) == 0) continue;
          ps_inv += 4;
          be_pix += 4;
          if constexpr (VIS) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
              for (int s = 0; s < S; ++s)
                if (tested[i] & (1u << s)) winner[i][s] = id;
          } else {
            shade_store<NA, S, SASL>(P, SM, tri_attr, id, px0, py0,
                                     tested[0] | (tested[1] << 4) | (tested[2] << 8) | (tested[3] << 12));
          }
        } else if constexpr (!VIS) {
          // late depth/stencil (render_sample, framebuffer.cpp:445-479); writes only when both pass.
          // The tests of a sample depend only on that sample's depth/stencil, not on the colour, so
          // they run first and the pixel shader (side-effect free) runs only when some sample passes.
          ps_inv += 4;
          be_pix += 4;
          const int face = L.front ? 0 : 1;
          uint32_t passed[4] = {0, 0, 0, 0};
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int s = 0; s < S; ++s) {
              if (!(cov[i] & (1u << s))) continue;
              float nd = (S > 1) ? (z[i] + L.aa[s]) : z[i];
              float od = P.read_depth ? depth[i][s] : 0.0f;
              uint32_t os = P.stencil_enable ? (stencil[i][s] & P.read_mask) : 0u;
              bool dp = has_ds ? (P.depth_enable ? cmpf(P.depth_func, nd, od) : true) : true;
              bool sp = P.stencil_enable ? cmpu(P.st_func[face], P.stencil_ref, os) : true;
              if (dp && sp) passed[i] |= 1u << s;
            }
          if ((passed[0] | passed[1] | passed[2] | passed[3]) == 0) continue;
          shade_store<NA, S, SASL>(P, SM, tri_attr, id, px0, py0,
                                   passed[0] | (passed[1] << 4) | (passed[2] << 8) | (passed[3] << 12));
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int s = 0; s < S; ++s) {
              if (!(passed[i] & (1u << s))) continue;
              float nd = (S > 1) ? (z[i] + L.aa[s]) : z[i];
              uint32_t os = P.stencil_enable ? (stencil[i][s] & P.read_mask) : 0u;
              uint32_t ns = P.stencil_enable ? stencil_op(P.st_pass_op[face], P.stencil_ref, os) : 0u;
              if (P.write_depth) depth[i][s] = nd;
              if (P.stencil_enable) stencil[i][s] = ns & P.write_mask;
            }
        }
      }
    }
    __syncthreads();
  }

  if constexpr (VIS) {
    // winners for the shading pass, laid out like the colour target's samples
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (pin[i]) {
        size_t base = (static_cast<size_t>(py0 + (i >> 1)) * tw + (px0 + (i & 1))) * S;
#pragma unroll
        for (int s = 0; s < S; ++s) vis[base + s] = winner[i][s];
      }
    if (has_ds && P.write_depth) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (pin[i])
#pragma unroll
          for (int s = 0; s < S; ++s)
            *reinterpret_cast<float*>(sample_addr(P.ds, px0 + (i & 1), py0 + (i >> 1), s)) = depth[i][s];
    }
  } else if (has_ds && (P.write_depth || P.stencil_enable)) {
    // write back depth/stencil
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (pin[i])
#pragma unroll
        for (int s = 0; s < S; ++s)
          *reinterpret_cast<float2*>(sample_addr(P.ds, px0 + (i & 1), py0 + (i >> 1), s)) =
              make_float2(depth[i][s], __uint_as_float(stencil[i][s]));
  }
  // ps_invocations and backend_input_pixels advance together (+4 per shaded quad: the sample shaders
  // never discard), so one partial carries both
  (void)be_pix;
  if (P.count_stats) block_partial(partial, ps_inv);  // uniform over the launch
}

// Deferred pixel shading of an opaque early-Z draw: one thread per pixel (16x16 pixels per
// workgroup).  For each distinct winning triangle of the pixel's samples, the thread evaluates that
// triangle's quad interpolants (the values the reference's last passing draw_quad/draw_full_quad
// computed for this quad), runs the pixel shader for its own pixel and writes the winning samples.
template <int NA, int S>
__global__ void __launch_bounds__(256) shade_kernel(draw_params P, const ps_samplers* __restrict__ SM,
                                                     const float4* __restrict__ tri_attr, const uint32_t* __restrict__ vis) {
  const int x = blockIdx.x * 16 + (threadIdx.x & 15), y = blockIdx.y * 16 + (threadIdx.x >> 4);
  const int tw = static_cast<int>(P.target_w), th = static_cast<int>(P.target_h);
  if (x >= tw || y >= th) return;
  const int px0 = x & ~1, py0 = y & ~1;
  const int pi = (x & 1) | ((y & 1) << 1);  // position in the quad
  const size_t base = (static_cast<size_t>(y) * tw + x) * S;
  uint32_t w[S];
#pragma unroll
  for (int s = 0; s < S; ++s) w[s] = vis[base + s];
#pragma unroll
  for (int it = 0; it < S; ++it) {
    uint32_t cur = NO_WINNER;
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (cur == NO_WINNER) cur = w[s];
    if (cur >= 3u * P.prim_count) break;  // NO_WINNER (every id is below 3 * prim_count)
    attr_setup<NA> at;
    load_attr<NA>(P, tri_attr, cur, at);
    const quad_lazy<NA> q(at, P, px0, py0);
    const float4 c = run_ps_pixel<NA>(P, SM, q, pi);
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (w[s] == cur) {
        store_texel(P.color.pf, sample_addr(P.color, x, y, s), c);
        w[s] = NO_WINNER;
      }
  }
}

// Deferred SASL shading of an opaque early-Z draw: one thread per 2x2 quad of a 16x16 GPU tile
// (the tiles the visibility pass wrote).  For each distinct winning triangle among the quad's samples
// the program runs once on the whole quad (pixel_shader_unit::execute, shader_unit.cpp:147-176) and
// the samples that triangle won take their pixel's colour: a SASL pixel's colour depends only on the
// triangle and the quad, so this equals shading every early-Z pass in order.
template <int NA, int S>
__global__ void __launch_bounds__(64) sasl_shade_kernel(draw_params P, const ps_samplers* __restrict__ SM,
                                                        const float4* __restrict__ tri_attr, const uint32_t* __restrict__ vis) {
  const int px0 = blockIdx.x * 16 + (threadIdx.x & 7) * 2, py0 = blockIdx.y * 16 + (threadIdx.x >> 3) * 2;
  const int tw = static_cast<int>(P.target_w), th = static_cast<int>(P.target_h);
  if (px0 >= tw || py0 >= th) return;
  uint32_t w[4][S];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int x = px0 + (i & 1), y = py0 + (i >> 1);
    const bool in = x < tw && y < th;
#pragma unroll
    for (int s = 0; s < S; ++s) w[i][s] = in ? vis[(static_cast<size_t>(y) * tw + x) * S + s] : NO_WINNER;
  }
  const sasl_program* __restrict__ prog = P.sasl;
  for (int it = 0; it < 4 * S; ++it) {
    uint32_t cur = NO_WINNER;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int s = 0; s < S; ++s)
        if (cur == NO_WINNER) cur = w[i][s];
    if (cur >= 3u * P.prim_count) break;  // NO_WINNER (every id is below 3 * prim_count)
    attr_setup<NA> at;
    load_attr<NA>(P, tri_attr, cur, at);
    const quad_lazy<NA> q(at, P, px0, py0);
    sasl_regs R;
    const uint32_t nregs = prog->nregs, nin = prog->ninputs;
    for (uint32_t r = 0; r < nregs; ++r)
      for (int px = 0; px < 4; ++px) R.r[r][px] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int px = 0; px < 4; ++px) {
      const float iw = q.inv_w(px);
      for (uint32_t k = 0; k < nin; ++k) {
        const sasl_input inp = prog->inputs[k];
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
        for (int a = 0; a < NA; ++a)
          if (a == inp.attr) v = q.reg(a + 1, px, iw);
        R.r[inp.reg][px] = make_float4(v.x, inp.ncomp > 1 ? v.y : 0.0f, inp.ncomp > 2 ? v.z : 0.0f, inp.ncomp > 3 ? v.w : 0.0f);
      }
    }
    sasl_exec(prog, R, [&](int slot, int, float u, float v, float dxu, float dxv, float dyu, float dyv) -> float4 {
      if (!P.has_sampler[slot]) return make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      const sampler_desc_dev& sp = SM->s[slot];
      return sample_grad(sp, u, v, dxu, dxv, dyu, dyv);
    });
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      bool any = false;
#pragma unroll
      for (int s = 0; s < S; ++s) any |= w[i][s] == cur;
      if (!any) continue;
      const float4 c = sasl_color0(prog, R, i);
      const int x = px0 + (i & 1), y = py0 + (i >> 1);
#pragma unroll
      for (int s = 0; s < S; ++s)
        if (w[i][s] == cur) {
          store_texel(P.color.pf, sample_addr(P.color, x, y, s), c);
          w[i][s] = NO_WINNER;
        }
    }
  }
}

// ============================================================== host launchers
void launch_raster(const draw_params& P, const draw_buffers& B, int which, hipStream_t s) {
  uint32_t T = static_cast<uint32_t>(P.gtiles_x * P.gtiles_y);
  if (!T) return;
  int threads = (P.gt / 2) * (P.gt / 2);
  size_t lds = sizeof(prim_lds) * threads;
  bool vis = P.early_z && (P.blend_id == BLEND_OFF || P.blend_id == BLEND_DISABLED);
  const bool sasl = !vis && sasl_shades(P);  // in-order shading by the SASL program
#define SRX_RASTER_S(NA, S)                                                                                          \
  do {                                                                                                               \
    if (vis)                                                                                                         \
      hipLaunchKernelGGL((raster_kernel<NA, S, true>), dim3(T), dim3(threads), lds, s, P, B.samplers, B.order, B.vals[which], \
                         B.tstart, B.tend, B.tri_rec, B.tri_attr, B.vis, B.partial, B.counters, B.list_cap);                                 \
    else if (sasl)                                                                                                   \
      hipLaunchKernelGGL((raster_kernel<NA, S, false, true>), dim3(T), dim3(threads), lds, s, P, B.samplers, B.order, \
                         B.vals[which], B.tstart, B.tend, B.tri_rec, B.tri_attr, B.vis, B.partial, B.counters, B.list_cap);                  \
    else                                                                                                             \
      hipLaunchKernelGGL((raster_kernel<NA, S, false>), dim3(T), dim3(threads), lds, s, P, B.samplers, B.order,      \
                         B.vals[which], B.tstart, B.tend, B.tri_rec, B.tri_attr, B.vis, B.partial, B.counters, B.list_cap);                  \
  } while (0)
#define SRX_RASTER(NA)                     \
  switch (P.samples) {                     \
  case 1: SRX_RASTER_S(NA, 1); break;      \
  case 2: SRX_RASTER_S(NA, 2); break;      \
  default: SRX_RASTER_S(NA, 4); break;     \
  }
  SRX_NA_DISPATCH(P.nattr, SRX_RASTER)
#undef SRX_RASTER
#undef SRX_RASTER_S
  if (P.count_stats) {
    launch_reduce_partials(B.partial, T, B.stats, ST_PS_INVOCATIONS, s);
    launch_reduce_partials(B.partial, T, B.stats, ST_BACKEND_PIXELS, s);
  }
}

// One thread per quad: pixel_shader_unit::update/execute on caller-supplied inputs (the quad
// evaluation behind srx_ps_execute_quads).  in: [quad][pixel][input] float4, out: [quad][pixel][output].
__global__ void __launch_bounds__(64) sasl_quads_kernel(const sasl_program* __restrict__ prog,
                                                        const ps_samplers* __restrict__ SM, uint32_t has_mask,
                                                        const float4* __restrict__ in, float4* __restrict__ out,
                                                        uint32_t nquads) {
  const uint32_t qi = blockIdx.x * blockDim.x + threadIdx.x;
  if (qi >= nquads) return;
  const uint32_t nin = prog->ninputs, nout = prog->noutputs, nregs = prog->nregs;
  sasl_regs R;
  for (uint32_t r = 0; r < nregs; ++r)
    for (int px = 0; px < 4; ++px) R.r[r][px] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  for (int px = 0; px < 4; ++px)
    for (uint32_t k = 0; k < nin; ++k) {
      const sasl_input inp = prog->inputs[k];
      const float4 v = in[(static_cast<size_t>(qi) * 4 + px) * nin + k];
      R.r[inp.reg][px] = make_float4(v.x, inp.ncomp > 1 ? v.y : 0.0f, inp.ncomp > 2 ? v.z : 0.0f, inp.ncomp > 3 ? v.w : 0.0f);
    }
  sasl_exec(prog, R, [&](int slot, int, float u, float v, float dxu, float dxv, float dyu, float dyv) -> float4 {
    if (!((has_mask >> slot) & 1u)) return make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const sampler_desc_dev& sp = SM->s[slot];
    return sample_grad(sp, u, v, dxu, dxv, dyu, dyv);
  });
  for (int px = 0; px < 4; ++px)
    for (uint32_t o = 0; o < nout; ++o) {
      const float4 v = R.r[prog->outputs[o].reg][px];
      const int nc = prog->outputs[o].ncomp;
      out[(static_cast<size_t>(qi) * 4 + px) * nout + o] =
          make_float4(v.x, nc > 1 ? v.y : 0.0f, nc > 2 ? v.z : 0.0f, nc > 3 ? v.w : 0.0f);
    }
}

void launch_sasl_quads(const sasl_program* prog, const ps_samplers* SM, uint32_t has_mask, const float4* in, float4* out,
                       uint32_t nquads, hipStream_t s) {
  if (!nquads) return;
  hipLaunchKernelGGL(sasl_quads_kernel, dim3((nquads + 63) / 64), dim3(64), 0, s, prog, SM, has_mask, in, out, nquads);
}

bool sasl_shades(const draw_params& P) {
  return P.ps_id == PS_SASL && P.color.data != nullptr && P.blend_id != BLEND_DISABLED;
}

bool needs_shading(const draw_params& P) {
  return (P.early_z || P.vis_stencil) && P.blend_id == BLEND_OFF && P.color.data != nullptr;
}

// Covers exactly the 16x16 GPU tiles vis_kernel wrote: pixels of the target beyond the viewport's
// 64x64 tile grid hold no winners of this draw.
void launch_shade(const draw_params& P, const draw_buffers& B, hipStream_t s) {
  if (P.gtiles_x <= 0 || P.gtiles_y <= 0) return;
  dim3 grid(P.gtiles_x, P.gtiles_y);
  if (P.ps_id == PS_SASL) {
#define SRX_SASL_SHADE_S(NA, S) \
  hipLaunchKernelGGL((sasl_shade_kernel<NA, S>), grid, dim3(64), 0, s, P, B.samplers, B.tri_attr, B.vis)
#define SRX_SASL_SHADE(NA)                    \
  switch (P.samples) {                        \
  case 1: SRX_SASL_SHADE_S(NA, 1); break;     \
  case 2: SRX_SASL_SHADE_S(NA, 2); break;     \
  default: SRX_SASL_SHADE_S(NA, 4); break;    \
  }
    SRX_NA_DISPATCH(P.nattr, SRX_SASL_SHADE)
#undef SRX_SASL_SHADE
#undef SRX_SASL_SHADE_S
    return;
  }
#define SRX_SHADE_S(NA, S) \
  hipLaunchKernelGGL((shade_kernel<NA, S>), grid, dim3(256), 0, s, P, B.samplers, B.tri_attr, B.vis)
#define SRX_SHADE(NA)                    \
  switch (P.samples) {                   \
  case 1: SRX_SHADE_S(NA, 1); break;     \
  case 2: SRX_SHADE_S(NA, 2); break;     \
  default: SRX_SHADE_S(NA, 4); break;    \
  }
  SRX_NA_DISPATCH(P.nattr, SRX_SHADE)
#undef SRX_SHADE
#undef SRX_SHADE_S
}

}  // namespace srx
