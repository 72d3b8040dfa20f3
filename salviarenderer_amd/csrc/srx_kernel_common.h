// Device code shared by the kernel sources: shader and state numbering, wave and workgroup
// reductions, the depth/stencil comparisons, the pixel shaders and the blended store of a sample.
#pragma once

#include "srx_kernels.h"
#include "srx_sampler.h"
#include "srx_shade_common.h"

namespace srx {

enum { VS_PASSTHROUGH_COLOR = 1, VS_WVP_NORMAL_UV = 2, VS_WVP_COLOR = 3, VS_WVP_COLOR_LIGHT = 4, VS_COLORIZED = 5,
       VS_MESH = 6, VS_SSM_DRAW = 7, VS_CUP = 8, VS_BOX = 9 };
enum { PS_GOURAUD = 1, PS_LAMBERT_TEX = 2, PS_TEX_CPP = 3, PS_CONSTANT = 4, PS_SHADOW_PCF = 5, PS_COLORIZED = 6,
       PS_MESH = 7, PS_SSM = 8, PS_CUP = 9, PS_BOX = 10 };
enum { BLEND_OFF = 0, BLEND_ON = 1, BLEND_DISABLED = 2 };
enum { TOPO_TRIANGLE_LIST = 2, TOPO_TRIANGLE_STRIP = 4 };
enum { FMT_RGBA32F = 2, FMT_RGBA32I = 4, FMT_RGB32F = 6, FMT_RG32F = 16, FMT_R32F = 41 };
enum { CULL_NONE = 0, CULL_FRONT = 1, CULL_BACK = 2 };
enum { SOP_KEEP = 1, SOP_ZERO, SOP_REPLACE, SOP_INCR_SAT, SOP_DECR_SAT, SOP_INVERT, SOP_INCR_WRAP, SOP_DECR_WRAP };

// Register selects of whole vertices, one float at a time: a conditional over vertex lvalues
// would select addresses and push the vertices into scratch memory.
__device__ __forceinline__ float4 sel4(bool c, float4 a, float4 b) {
  return make_float4(c ? a.x : b.x, c ? a.y : b.y, c ? a.z : b.z, c ? a.w : b.w);
}
// Edges and bounding box of a set-up triangle (words 0..3 of its record).
__device__ __forceinline__ void read_tri_rec(const float4* rec, float* e, float* bb) {
  float4 a = rec[0], b = rec[1], c = rec[2], d = rec[3];
  e[0] = a.x; e[1] = a.y; e[2] = a.z; e[3] = a.w; e[4] = b.x; e[5] = b.y; e[6] = b.z; e[7] = b.w; e[8] = c.x;
  bb[0] = c.y; bb[1] = c.z; bb[2] = c.w; bb[3] = d.x;
}

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
  int lane = __lane_id();
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    uint32_t t = __shfl_up(v, off, 64);
    if (lane >= off) v += t;
  }
  return v;
}

// Sums v over the workgroup and stores the total in partial[blockIdx.x] (no global atomics: many
// same-address device-scope atomics from every XCD serialise badly).  All threads must call it.
__device__ __forceinline__ void block_partial(unsigned long long* __restrict__ partial, unsigned long long v) {
  __shared__ unsigned long long wsum[16];
  unsigned long long s = v;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  const int wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) wsum[wave] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t = 0;
    for (int w = 0; w < nw; ++w) t += wsum[w];
    partial[blockIdx.x] = t;
  }
}

// The job of this workgroup in a batched launch, its index among the job's workgroups and their count.
__device__ __forceinline__ uint32_t stage_job(const stage_map& m, uint32_t& local, uint32_t& blocks) {
  const uint32_t j = m.job[blockIdx.x];
  const uint2 r = m.range[j];
  local = blockIdx.x - r.x;
  blocks = r.y;
  return j;
}

// ============================================================== pixel shaders
__device__ __forceinline__ void normalize3(float x, float y, float z, float& ox, float& oy, float& oz) {
  float t = 0.0f;
  t += x * x;
  t += y * y;
  t += z * z;
  float len = sqrtf(t);
  if (equal_eps(len, 0.0f)) len = 1.0f;
  float inv = 1.0f / len;
  ox = x * inv;
  oy = y * inv;
  oz = z * inv;
}

// 3x3 percentage-closer shadow lookup of one pixel (attr0 colour, attr1 light clip position): the
// tap layout of StandardShadowMap.cpp:86-106, each tap a tex2dlod at lod 0, lit when the light-space
// depth minus the bias does not exceed it.
__device__ __forceinline__ float4 shadow_pcf(const draw_params& P, const ps_samplers* __restrict__ SM, float4 a, float4 l) {
  const float lx = l.x / l.w, ly = l.y / l.w, lz = l.z / l.w;
  const float cu = (lx + 1.0f) * 0.5f, cv = 1.0f - (ly + 1.0f) * 0.5f;
  const float o = P.ps_consts[2];
  int count = 0;
  if (P.has_sampler[0]) {
    for (int ty = -1; ty <= 1; ++ty)
      for (int tx = -1; tx <= 1; ++tx) {
        const float u = cu + static_cast<float>(tx) * o, v = cv + static_cast<float>(ty) * o;
        const float4 t = sample_lod0(SM->s[0], u, v);
        if (lz - P.ps_consts[1] <= t.x) ++count;
      }
  }
  const float lit = static_cast<float>(count) / 9.0f;
  const float k = P.ps_consts[0] + (1.0f - P.ps_consts[0]) * lit;
  return make_float4(a.x * k, a.y * k, a.z * k, a.w);
}

// Whether the shaders that any draw may use (PS_LAMBERT_TEX, PS_TEX_CPP, PS_BOX) sample by the inline paths.  With
// three attributes and more their registers are spilled around every shader of the kernel, the ones in use
// included: there only PS_CUP and PS_SSM, made for such draws, inline theirs (130k triangles at 1920x1080,
// 4 samples: PS_CUP 274 -> 250 us a frame, PS_COLORIZED 240 -> 229, PS_MESH 230 -> 217).
template <int NA>
constexpr bool INLINE_TAPS = NA < 3;

// cpp_pixel_shader::tex2d(s, reg) (cpp_pixel_shader.cpp:13-31): one LOD per quad from the register's
// p1 - p0 and p2 - p0 (calc_lod_2d, sampler.cpp:834-852), then sample_2d_lod at pixel pi
template <int NA, bool FAST = INLINE_TAPS<NA>>
__device__ __forceinline__ float4 tex2d_cpp(const sampler_desc_dev& sp, const quad_lazy<NA>& q, int reg, int pi) {
  const float4 u0 = q.reg(reg, 0, q.inv_w(0), 2), u1 = q.reg(reg, 1, q.inv_w(1), 2), u2 = q.reg(reg, 2, q.inv_w(2), 2);
  const float dxu = u1.x - u0.x, dxv = u1.y - u0.y;
  const float dyu = u2.x - u0.x, dyv = u2.y - u0.y;
  const float lod = (sp.mip_filter == FILTER_ANISO && sp.max_aniso > 1) ? calc_aniso(sp, dxu, dxv, dyu, dyv, 0.0f).lod
                                                                        : calc_lod(sp, dxu, dxv, dyu, dyv, 0.0f);
  const float4 uv = q.reg(reg, pi, q.inv_w(pi), 2);
  if (FAST && sp.fast_linear) return sample_linear_fast(sp, uv.x, uv.y, lod);
  return sample_impl(sp, uv.x, uv.y, lod, nullptr);
}
// eflib vector helpers on .xyz (vector_generic.h:110-118, math.cpp:39-41,85-87)
__device__ __forceinline__ float dot3(float4 a, float4 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ float length3(float4 a) {
  float t = 0.0f;
  t += a.x * a.x;
  t += a.y * a.y;
  t += a.z * a.z;
  return sqrtf(t);
}
__device__ __forceinline__ float4 normalize3v(float4 v) {
  float x, y, z;
  normalize3(v.x, v.y, v.z, x, y, z);
  return make_float4(x, y, z, 0.0f);
}
__device__ __forceinline__ float4 reflect3(float4 i, float4 n) {
  const float k = 2.0f * dot3(i, n);
  return make_float4(i.x - n.x * k, i.y - n.y * k, i.z - n.z * k, 0.0f);
}

// ColorizedTriangle.cpp:55-92: three lights, attr0 normal, attr1..3 light vectors
template <int NA>
__device__ __forceinline__ float4 ps_colorized(const quad_lazy<NA>& q, int pi) {
  const float iw = q.inv_w(pi);
  const float4 n = q.reg(1, pi, iw, 3);
  float4 ld[3];
  float inv[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    ld[i] = q.reg(2 + i, pi, iw, 3);
    inv[i] = 1.0f / length3(ld[i]);
  }
  const float4 nn = normalize3v(n);
  float refl[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) refl[i] = dot3(nn, make_float4(ld[i].x * inv[i], ld[i].y * inv[i], ld[i].z * inv[i], 0.0f));
  const float c[3][3] = {{0.7f, 0.1f, 0.3f}, {0.1f, 0.3f, 0.7f}, {0.3f, 0.7f, 0.1f}};
  float o[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    float a = ((c[0][k] * refl[0]) * inv[0]) * inv[0];
    float b = ((c[1][k] * refl[1]) * inv[1]) * inv[1];
    float d = ((c[2][k] * refl[2]) * inv[2]) * inv[2];
    o[k] = std_clamp((a + b) + d, 0.0f, 1.0f);
  }
  return make_float4(o[0], o[1], o[2], 1.0f);
}

// ComplexMesh.cpp:227-246
template <int NA>
__device__ __forceinline__ float4 ps_mesh(const quad_lazy<NA>& q, int pi) {
  const float iw = q.inv_w(pi);
  const float4 l = normalize3v(q.reg(1, pi, iw, 3)), e = normalize3v(q.reg(2, pi, iw, 3)), n = normalize3v(q.reg(3, pi, iw, 3));
  const float n_dot_l = dot3(n, l);
  const float4 h = normalize3v(make_float4(l.x + e.x, l.y + e.y, l.z + e.z, 0.0f));
  const float spec = 3.5f * powf(std_max(dot3(h, n), 0.0f), 5.0f);  // (roughness + 2) / 2 with roughness 5
  const float clr = n_dot_l * (0.8f + spec * 0.4f);
  return make_float4(clr, clr, clr, 1.0f);
}

// StandardShadowMap.cpp:62-142 (exponential shadow map, esm_constant 25000, 3x3 Gaussian weights)
template <int NA>
__device__ __forceinline__ float4 ps_ssm(const draw_params& P, const ps_samplers* __restrict__ SM, const quad_lazy<NA>& q,
                                         int pi) {
  const float iw = q.inv_w(pi);
  float occlusion = 0.0f;
  if (P.has_sampler[0]) {
    const float4 l4 = q.reg(5, pi, iw);
    const float lx = l4.x / l4.w, ly = l4.y / l4.w, lz = l4.z / l4.w;
    const float cx = (lx + 1.0f) * 0.5f, cy = 1.0f - (ly + 1.0f) * 0.5f;
    const float o = 1 / 512.0f;
    const float ox[9] = {-o, 0.0f, +o, -o, 0.0f, +o, -o, 0.0f, +o};
    const float oy[9] = {-o, -o, -o, 0.0f, 0.0f, 0.0f, +o, +o, +o};
    const float gw[9] = {0.027681f, 0.111014f, 0.027681f, 0.111014f, 0.445213f, 0.111014f, 0.027681f, 0.111014f, 0.027681f};
    float sd[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) sd[i] = sample_lod0(SM->s[0], cx + ox[i], cy + oy[i]).x;
    const float esm = 25000.0f;
    float occ = 0.0f;
#pragma unroll
    for (int i = 1; i < 9; ++i) occ += gw[i] * expf(esm * (sd[i] - sd[0]));
    occ += gw[0];
    occ = logf(occ);
    occ += esm * sd[0];
    occlusion = std_clamp(expf(occ - esm * lz), 0.0f, 1.0f);
  }
  float4 tex = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
  if (P.has_sampler[1]) tex = tex2d_cpp<NA, true>(SM->s[1], q, 1, pi);
  const float4 n = normalize3v(q.reg(2, pi, iw, 3)), ld = normalize3v(q.reg(3, pi, iw, 3)), ed = normalize3v(q.reg(4, pi, iw, 3));
  const float idiff = std_clamp(dot3(ld, n), 0.0f, 1.0f);
  const float4 r = reflect3(ld, n);
  const float ispec = std_clamp(dot3(make_float4(-r.x, -r.y, -r.z, 0.0f), ed), 0.0f, 1.0f);
  // pow(float, int) promotes to double (C++11 <cmath>), then the vec4 product rounds it to float
  const float p = static_cast<float>(pow(static_cast<double>(ispec), static_cast<double>(__float_as_int(P.ps_consts[12]))));
  const float* amb = P.ps_consts;
  const float* dif = P.ps_consts + 4;
  const float* spc = P.ps_consts + 8;
  float4 out;
  out.x = tex.x * (amb[0] + (dif[0] * idiff + spc[0] * p) * occlusion);
  out.y = tex.y * (amb[1] + (dif[1] * idiff + spc[1] * p) * occlusion);
  out.z = tex.z * (amb[2] + (dif[2] * idiff + spc[2] * p) * occlusion);
  out.w = 1.0f;
  return out;
}

// StencilMirror.cpp:66-110
template <int NA>
__device__ __forceinline__ float4 ps_cup(const draw_params& P, const ps_samplers* __restrict__ SM, const quad_lazy<NA>& q,
                                         int pi) {
  const float iw = q.inv_w(pi);
  float4 tex = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
  if (P.has_sampler[0]) tex = tex2d_cpp<NA, true>(SM->s[0], q, 1, pi);
  const float4 n = normalize3v(q.reg(2, pi, iw, 3)), ld = normalize3v(q.reg(3, pi, iw, 3)), ed = normalize3v(q.reg(4, pi, iw, 3));
  const float idiff = std_clamp(dot3(ld, n), 0.0f, 1.0f);
  const float ispec = std_clamp(dot3(reflect3(ld, n), ed), 0.0f, 1.0f);
  const float* amb = P.ps_consts;
  const float* dif = P.ps_consts + 4;
  const float* spc = P.ps_consts + 8;
  float4 out;
  out.x = tex.x * ((amb[0] + dif[0] * idiff) + spc[0] * ispec);
  out.y = tex.y * ((amb[1] + dif[1] * idiff) + spc[1] * ispec);
  out.z = tex.z * ((amb[2] + dif[2] * idiff) + spc[2] * ispec);
  out.w = 1.0f;
  return out;
}

// Pixel shader (cpp_pixel_shader::execute, cpp_pixel_shader.cpp:62-74) colour of quad pixel pi
// only; the other three pixels supply derivatives.  The sample shaders never discard.
template <int NA>
__device__ __forceinline__ float4 run_ps_pixel(const draw_params& P, const ps_samplers* __restrict__ SM,
                                               const quad_lazy<NA>& q, int pi) {
  switch (P.ps_id) {
  case PS_GOURAUD:
    return q.reg(1, pi, q.inv_w(pi));
  case PS_CONSTANT:
    return make_float4(P.ps_consts[0], P.ps_consts[1], P.ps_consts[2], P.ps_consts[3]);
  case PS_LAMBERT_TEX:
    if constexpr (NA >= 2) {
      // SASL tex2D: ddx per row (p1-p0, p3-p2), ddy per column (p2-p0, p3-p1)
      // (sasl/src/codegen/cgs_simd.cpp:275-312), then sample_2d_grad (sampler_api.cpp:13-18);
      // uv at pi and its row and column neighbours
      const int pr = pi ^ 1, pc = pi ^ 2;
      const float iw = q.inv_w(pi), iwr = q.inv_w(pr), iwc = q.inv_w(pc);
      const float4 uv = q.reg(2, pi, iw, 2), uvr = q.reg(2, pr, iwr, 2), uvc = q.reg(2, pc, iwc, 2);
      const bool col1 = (pi & 1) != 0, row1 = (pi & 2) != 0;
      // row: (left, right) = col1 ? (neighbour, pi) : (pi, neighbour); column likewise
      const float4 r0 = sel4(col1, uvr, uv), r1 = sel4(col1, uv, uvr);
      const float4 c0 = sel4(row1, uvc, uv), c1 = sel4(row1, uv, uvc);
      const float dxu = r1.x - r0.x, dxv = r1.y - r0.y;
      const float dyu = c1.x - c0.x, dyv = c1.y - c0.y;
      const float4 nrm = q.reg(1, pi, iw, 3);
      float4 t = make_float4(0, 0, 0, 0);
      if (P.has_sampler[0]) t = sample_grad<INLINE_TAPS<NA>>(SM->s[0], uv.x, uv.y, dxu, dxv, dyu, dyv);
      float nx, ny, nz;
      normalize3(nrm.x, nrm.y, nrm.z, nx, ny, nz);
      float d = nx * P.ps_consts[0] + ny * P.ps_consts[1] + nz * P.ps_consts[2];
      float k = std_clamp(d, 0.0f, 1.0f);
      return make_float4(t.x * k, t.y * k, t.z * k, 1.0f);
    }
    return make_float4(0, 0, 0, 0);
  case PS_TEX_CPP: {
    // AnisotropicFilter / TextureAndBlending ps_plane: tex2d(s0, attr0) with alpha 1
    if (!P.has_sampler[0]) return make_float4(0, 0, 0, 1.0f);
    float4 t = tex2d_cpp(SM->s[0], q, 1, pi);
    t.w = 1.0f;
    return t;
  }
  case PS_COLORIZED:
    if constexpr (NA >= 4) return ps_colorized(q, pi);
    return make_float4(0, 0, 0, 0);
  case PS_MESH:
    if constexpr (NA >= 3) return ps_mesh(q, pi);
    return make_float4(0, 0, 0, 0);
  case PS_SSM:
    if constexpr (NA >= 5) return ps_ssm(P, SM, q, pi);
    return make_float4(0, 0, 0, 0);
  case PS_CUP:
    if constexpr (NA >= 4) return ps_cup(P, SM, q, pi);
    return make_float4(0, 0, 0, 0);
  case PS_BOX: {  // TextureAndBlending.cpp:96-114
    if constexpr (NA >= 2) {
      if (!P.has_sampler[0]) return make_float4(1.0f, 1.0f, 1.0f, 0.5f);
      float4 t = tex2d_cpp(SM->s[0], q, 2, pi);
      t.w = 0.5f;
      return t;
    }
    return make_float4(0, 0, 0, 0);
  }
  case PS_SHADOW_PCF:
    if constexpr (NA >= 2) {
      const float iw = q.inv_w(pi);
      return shadow_pcf(P, SM, q.reg(1, pi, iw), q.reg(2, pi, iw));
    }
    return make_float4(0, 0, 0, 0);
  default:
    return make_float4(0, 0, 0, 0);
  }
}

__device__ __forceinline__ bool cmpf(int f, float a, float b) {
  switch (f) {
  case 0: return false;
  case 1: return a < b;
  case 2: return a == b;
  case 3: return a <= b;
  case 4: return a > b;
  case 5: return a != b;
  case 6: return a >= b;
  default: return true;
  }
}
__device__ __forceinline__ bool cmpu(int f, uint32_t a, uint32_t b) {
  switch (f) {
  case 0: return false;
  case 1: return a < b;
  case 2: return a == b;
  case 3: return a <= b;
  case 4: return a > b;
  case 5: return a != b;
  case 6: return a >= b;
  default: return true;
  }
}
// framebuffer.cpp:136-166
__device__ __forceinline__ uint32_t stencil_op(int op, uint32_t ref, uint32_t cur) {
  switch (op) {
  case SOP_ZERO: return 0;
  case SOP_REPLACE: return ref;
  case SOP_INCR_SAT: return min(0xFFu, cur + 1);
  case SOP_DECR_SAT: return cur - 1;  // std::max<uint32_t>(0, cur - 1) never clamps
  case SOP_INVERT: return ~cur;
  case SOP_INCR_WRAP: return (cur + 1) & 0xFF;
  case SOP_DECR_WRAP: return (cur - 1 + 256) & 0xFF;
  default: return cur;
  }
}


__device__ __forceinline__ void blend_store(const draw_params& P, int x, int y, int smp, float4 src) {
  if (!P.color.data) return;
  uint8_t* a = sample_addr(P.color, x, y, smp);
  if (P.blend_id == BLEND_OFF) {
    store_texel(P.color.pf, a, src);
  } else if (P.blend_id == BLEND_ON) {
    store_texel(P.color.pf, a, lerp4(load_texel(P.color.pf, a), src, src.w));
  }
}


// Kernels are instantiated per attribute count: the vertex and setup buffers are strided by it.
#define SRX_NA_DISPATCH(NAV, CALL) \
  switch (NAV) {                   \
  case 1: CALL(1); break;          \
  case 2: CALL(2); break;          \
  case 3: CALL(3); break;          \
  case 4: CALL(4); break;          \
  default: CALL(5); break;         \
  }
// Batched draws are refused above two attributes when they are recorded (batch_max_attrs).
#define SRX_NA_DISPATCH_BATCH(NAV, CALL) \
  switch (NAV) {                         \
  case 1: CALL(1); break;                \
  default: CALL(2); break;               \
  }

}  // namespace srx
