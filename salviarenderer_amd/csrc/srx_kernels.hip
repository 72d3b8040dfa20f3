// HIP kernels of the Salvia rasterization pipeline for MI355X (gfx950).
//
// Draw pipeline (one HIP stream per renderer):
//   vs_kernel       vertex fetch + vertex shader, one thread per vertex    (stream_assembler.cpp,
//                   default_vertex_cache.cpp: the shader runs once per vertex instead of per cache miss)
//   setup_kernel    index fetch, near/far trivial accept, cull, winding, viewport transform and
//                   triangle setup, one thread per primitive                (clipper.cpp, rasterizer.cpp:864-945)
//   clip_kernel     Sutherland-Hodgman near/far clipping for the few primitives that need it; the
//                   draw's record total from setup's per-block totals
//   emit_kernel     per-triangle GPU-tile records written in clipped-primitive order (offsets from
//                   the per-block totals and a workgroup scan)
//   sort            by GPU tile: a counting sort (order-independent draws) or a stable 8-bit LSD
//                   radix sort -> per-tile lists in primitive order (the reference's per-tile
//                   std::sort, rasterizer.cpp:947-994)
//   raster_kernel   (srx_raster.hip) one workgroup per GPU tile, one thread per 2x2 quad; walks its tile's list in
//                   order and evaluates the reference's 64->16->4->sample decision chain per quad
//                   (rasterizer.cpp:298-773), early/late depth-stencil, pixel shader and blending
//                   (framebuffer.cpp).  Opaque early-Z draws defer the pixel shader to one pass over
//                   the final per-sample winners.
//   vis_kernel      (srx_vis.hip) the same decisions for opaque early-Z draws, whose result does not
//                   depend on primitive order, fused with their shading
#include "srx_kernel_common.h"

namespace srx {

template <int NA>
struct vtx {
  float4 r[NA + 1];
};

// ============================================================== vertex stage
// eflib::transform(out, v, m): out[i] = dot_prod4(v, column i) (eflib/src/math.cpp:142-154)
__device__ __forceinline__ float4 transform_rowvec(float4 v, const float* m) {
  float o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = v.x * m[0 * 4 + i] + v.y * m[1 * 4 + i] + v.z * m[2 * 4 + i] + v.w * m[3 * 4 + i];
  return make_float4(o[0], o[1], o[2], o[3]);
}

// eflib::transform33(out, v, m): out[i] = dot_prod3(v.xyz, column i.xyz), out.w = 0 (math.cpp:184-197)
__device__ __forceinline__ float4 transform33_rowvec(float4 v, const float* m) {
  float o[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) o[i] = v.x * m[0 * 4 + i] + v.y * m[1 * 4 + i] + v.z * m[2 * 4 + i];
  return make_float4(o[0], o[1], o[2], 0.0f);
}
// a float4 constant minus a register, component by component
__device__ __forceinline__ float4 sub4(const float* c, float4 v) {
  return make_float4(c[0] - v.x, c[1] - v.y, c[2] - v.z, c[3] - v.w);
}

__device__ __forceinline__ float4 fetch_elem(const input_elem_dev& e, uint32_t v) {
  uint32_t need;
  switch (e.fmt) {
  case FMT_R32F: need = 4; break;
  case FMT_RG32F: need = 8; break;
  case FMT_RGB32F: need = 12; break;
  default: need = 16; break;
  }
  uint64_t off = static_cast<uint64_t>(e.stride) * v;
  if (off + need > e.avail) return make_float4(0, 0, 0, 0);  // the reference reads out of bounds
  const float* f = reinterpret_cast<const float*>(e.base + off);
  // get_vec4 (stream_assembler.cpp:26-44)
  switch (e.fmt) {
  case FMT_R32F: return make_float4(f[0], 0.0f, 0.0f, e.default_w);
  case FMT_RG32F: return make_float4(f[0], f[1], 0.0f, e.default_w);
  case FMT_RGB32F: return make_float4(f[0], f[1], f[2], e.default_w);
  default: return make_float4(f[0], f[1], f[2], f[3]);
  }
}

// a[i] for i < n, else 0, loaded without a branch (the index is clamped): guarded loads in an
// unrolled loop would each sit in a branch of its own and wait for its data before the next issues.
// n must be at least 1.
__device__ __forceinline__ uint32_t load_or_zero(const uint32_t* __restrict__ a, uint32_t i, uint32_t n) {
  const uint32_t x = a[min(i, n - 1u)];
  return i < n ? x : 0u;
}

// Coalesced stores of a wave's per-lane blocks of W float4 (lane i's block at dst + i*W): the lanes
// in `mask` put their blocks in the wave's LDS staging area, then the wave stores the span with
// consecutive lanes on consecutive float4, skipping the blocks of lanes not in `mask` (their memory
// is left as it was).  Blocks wider than the staging area are staged a group of lanes at a time.
constexpr int WAVE_STAGE = 320;  // float4 of LDS staging per wave
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
template <int W>
__device__ __forceinline__ void wave_store_blocks(float4* __restrict__ dst, const float4 (&blk)[W], uint64_t mask,
                                                  float4* __restrict__ stage) {
  constexpr int LG = WAVE_STAGE / W < 64 ? WAVE_STAGE / W : 64;  // lanes per pass
  const int lane = __lane_id();
  for (int g = 0; g < 64; g += LG) {
    const uint64_t pm = (mask >> g) & (LG >= 64 ? ~0ull : ((1ull << LG) - 1ull));
    if (!pm) continue;  // wave-uniform
    if (lane >= g && lane < g + LG && ((mask >> lane) & 1ull)) {
#pragma unroll
      for (int k = 0; k < W; ++k) stage[(lane - g) * W + k] = blk[k];
    }
    wave_lds_sync();
    const int n = min(LG, 64 - g) * W;
    for (int j = lane; j < n; j += 64)
      if ((pm >> (j / W)) & 1ull) dst[static_cast<size_t>(g) * W + j] = stage[j];
    wave_lds_sync();  // the stores have read the staging area before the next group writes it
  }
}
// The same with a run-time block width w <= MAX_REGS (lane i's block: blk[0..w)).
__device__ __forceinline__ void wave_store_blocks_n(float4* __restrict__ dst, const float4 (&blk)[MAX_REGS], int w,
                                                    uint64_t mask, float4* __restrict__ stage) {
  const int lg = min(WAVE_STAGE / w, 64);
  const int lane = __lane_id();
  for (int g = 0; g < 64; g += lg) {
    const uint64_t pm = (mask >> g) & (lg >= 64 ? ~0ull : ((1ull << lg) - 1ull));
    if (!pm) continue;  // wave-uniform
    if (lane >= g && lane < g + lg && ((mask >> lane) & 1ull)) {
#pragma unroll
      for (int k = 0; k < MAX_REGS; ++k)
        if (k < w) stage[(lane - g) * w + k] = blk[k];
    }
    wave_lds_sync();
    const int n = min(lg, 64 - g) * w;
    for (int j = lane; j < n; j += 64)
      if ((pm >> (j / w)) & 1ull) dst[static_cast<size_t>(g) * w + j] = stage[j];
    wave_lds_sync();
  }
}

// Kernel bodies take their workgroup index `bx` (and grid size where they stride) as arguments:
// the single-draw kernels pass blockIdx.x, the batched kernels a job's local workgroup index.
__device__ __forceinline__ void vs_body(const draw_params& P, float4* __restrict__ vbuf, uint32_t bx) {
  uint32_t v = bx * blockDim.x + threadIdx.x;
  const bool live = v <= P.nverts;  // slot nverts holds the output for an all-out-of-bounds fetch
  float4 in[MAX_INPUTS];
#pragma unroll
  for (int i = 0; i < MAX_INPUTS; ++i) in[i] = make_float4(0, 0, 0, 0);
  if (v < P.nverts)
    for (int i = 0; i < P.nin; ++i) {
      const float4 x = fetch_elem(P.in[i], v);
#pragma unroll
      for (int r = 0; r < MAX_INPUTS; ++r)  // register-resident: no dynamically indexed array
        if (P.in[i].reg == r) in[r] = x;
    }
  float4 out[MAX_REGS];
#pragma unroll
  for (int r = 0; r < MAX_REGS; ++r) out[r] = make_float4(0, 0, 0, 0);
  const float* k = P.vs_consts;
  switch (P.vs_id) {
  case VS_PASSTHROUGH_COLOR:
    out[0] = in[0];
    out[1] = in[1];
    break;
  case VS_WVP_COLOR:
    out[0] = transform_rowvec(in[0], k);
    out[1] = in[1];
    break;
  case VS_WVP_COLOR_LIGHT:  // light-space position for the shadow lookup (StandardShadowMap.cpp)
    out[0] = transform_rowvec(in[0], k);
    out[1] = in[1];
    out[2] = transform_rowvec(in[0], k + 16);
    break;
  case VS_COLORIZED:  // ColorizedTriangle.cpp:44-52
    out[0] = transform_rowvec(in[0], k);
    out[1] = in[1];
    out[2] = sub4(k + 16, in[0]);
    out[3] = sub4(k + 20, in[0]);
    out[4] = sub4(k + 24, in[0]);
    break;
  case VS_MESH: {  // ComplexMesh.cpp:202-211
    const float4 es = transform_rowvec(in[0], k);
    out[0] = transform_rowvec(es, k + 16);
    out[1] = make_float4(k[32] - es.x, k[33] - es.y, k[34] - es.z, 1.0f);
    out[2] = make_float4(k[36] - es.x, k[37] - es.y, k[38] - es.z, 1.0f);
    out[3] = transform33_rowvec(in[1], k);
    break;
  }
  case VS_SSM_DRAW:  // resources/ssm/Draw.savs: consts cameraPos, cameraWvp, lightPos, lightWvp
    out[0] = transform_rowvec(in[0], k + 4);
    out[1] = in[2];
    out[2] = in[1];
    out[3] = sub4(k + 20, in[0]);
    out[4] = sub4(k, in[0]);
    out[5] = transform_rowvec(in[0], k + 24);
    break;
  case VS_CUP:  // StencilMirror.cpp:47-55: consts wvp, eyePos, lightPos
    out[0] = transform_rowvec(in[0], k);
    out[1] = in[2];
    out[2] = in[1];
    out[3] = sub4(k + 20, in[0]);
    out[4] = sub4(k + 16, in[0]);
    break;
  case VS_BOX:  // TextureAndBlending.cpp:76-81
    out[0] = transform_rowvec(in[0], k);
    out[1] = in[0];
    out[2] = in[1];
    break;
  default:  // VS_WVP_NORMAL_UV
    out[0] = transform_rowvec(in[0], k);
    out[1] = in[1];
    out[2] = in[2];
    break;
  }
  // the wave's 64 consecutive vertices' outputs are stored coalesced (blockDim.x is 256)
  __shared__ float4 stage[4 * WAVE_STAGE];
  const uint64_t mask = __ballot(live);
  if (mask) {
    const int w = P.nattr + 1;
    const size_t v0 = static_cast<size_t>(bx) * blockDim.x + (threadIdx.x & ~63u);
    wave_store_blocks_n(vbuf + v0 * w, out, w, mask, stage + (threadIdx.x >> 6) * WAVE_STAGE);
  }
}
// A single draw's first launch: it also zeroes the draw's counters and ntiles per-tile record counts
// and cursors, which the launches after it add to.
__global__ void __launch_bounds__(256) vs_kernel(draw_params P, float4* __restrict__ vbuf, uint32_t* __restrict__ counters,
                                                 uint32_t* __restrict__ tiles, uint32_t ntiles) {
  const uint32_t nz = max(ntiles, static_cast<uint32_t>(CT_COUNT));
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nz; i += gridDim.x * blockDim.x) {
    if (i < static_cast<uint32_t>(CT_COUNT)) counters[i] = 0u;
    if (i < ntiles) tiles[i] = 0u;
  }
  vs_body(P, vbuf, blockIdx.x);
}

// ============================================================== primitive assembly helpers
__device__ __forceinline__ uint32_t fetch_index(const draw_params& P, uint32_t prim, int k) {
  uint32_t id;
  if (P.topo == TOPO_TRIANGLE_LIST) {
    id = prim * 3 + k;
  } else {  // strip: odd primitives swap ids 0 and 2 (index_fetcher.cpp:69-77)
    id = prim + k;
    if (prim & 1) id = (k == 0) ? prim + 2 : (k == 2 ? prim : prim + 1);
  }
  if (!P.indexed) return id + static_cast<uint32_t>(P.basevert);
  uint64_t off = static_cast<uint64_t>(P.istart_bytes) + static_cast<uint64_t>(id) * P.istride;
  uint32_t v = 0;
  if (off + P.istride <= P.ib_size)
    v = (P.istride == 2) ? *reinterpret_cast<const uint16_t*>(P.ib + off) : *reinterpret_cast<const uint32_t*>(P.ib + off);
  return v + static_cast<uint32_t>(P.basevert);
}

template <int NA>
__device__ __forceinline__ void load_vertex(const draw_params& P, const float4* vbuf, uint32_t index, vtx<NA>& out) {
  uint32_t slot = index < P.nverts ? index : P.nverts;
  const float4* src = vbuf + static_cast<size_t>(slot) * (NA + 1);
#pragma unroll
  for (int r = 0; r <= NA; ++r) out.r[r] = src[r];
}

__device__ __forceinline__ float dot4(float4 p, float4 v) { return p.x * v.x + p.y * v.y + p.z * v.z + p.w * v.w; }

// raster_state cull functions (raster_state.cpp:10-32)
__device__ __forceinline__ bool cull_fn(const draw_params& P, float area) {
  switch (P.cull_mode) {
  case CULL_FRONT: return P.front_ccw ? (area <= 0) : (area >= 0);
  case CULL_BACK: return P.front_ccw ? (area >= 0) : (area <= 0);
  default: return false;
  }
}

// viewport_transform + project_n (shader.cpp:499-511, 117-135)
template <int NA>
__device__ __forceinline__ void viewport_project(vtx<NA>& v, const draw_params& P) {
  float4 p = v.r[0];
  float invw = equal_eps(p.w, 0.0f) ? 1.0f : 1.0f / p.w;
  float px = p.x * invw, py = p.y * invw, pz = p.z * invw;
  float ox = (P.vp[0] + P.vp[2]) * 0.5f, oy = (P.vp[1] + P.vp[3]) * 0.5f;
  v.r[0].x = (P.vp[2] * 0.5f) * px + ox;
  v.r[0].y = (P.vp[3] * 0.5f) * -py + oy;
  v.r[0].z = (P.vp[5] - P.vp[4]) * pz + P.vp[4];
  v.r[0].w = invw;
#pragma unroll
  for (int a = 0; a < NA; ++a)
    if (!(P.attr_mod[a] & AM_NOPERSPECTIVE)) {
      v.r[a + 1].x *= invw;
      v.r[a + 1].y *= invw;
      v.r[a + 1].z *= invw;
      v.r[a + 1].w *= invw;
    }
}

template <int NA>
struct tri_setup {
  vtx<NA> v0, ddx, ddy;
  float e[3][3];
  float bb[4];
  bool front, valid;
};

// compute_triangle_info (rasterizer.cpp:864-945) + compute_derivative_n (shader.cpp:414-450)
template <int NA>
__device__ __forceinline__ vtx<NA> vsel(bool c, const vtx<NA>& a, const vtx<NA>& b) {
  vtx<NA> o;
#pragma unroll
  for (int r = 0; r <= NA; ++r) o.r[r] = sel4(c, a.r[r], b.r[r]);
  return o;
}
template <int NA>
__device__ __forceinline__ vtx<NA> pick3(int i, const vtx<NA>& a, const vtx<NA>& b, const vtx<NA>& c) {
  vtx<NA> o;
#pragma unroll
  for (int r = 0; r <= NA; ++r) o.r[r] = sel4(i == 0, a.r[r], sel4(i == 1, b.r[r], c.r[r]));
  return o;
}

template <int NA>
__device__ __forceinline__ void triangle_info(const vtx<NA>& a, const vtx<NA>& b, const vtx<NA>& c, tri_setup<NA>& t) {
  const vtx<NA>* V[3] = {&a, &b, &c};  // constant indices only (after unrolling)
  double dist[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) dist[i] = static_cast<double>(fabsf(V[i]->r[0].x) + fabsf(V[i]->r[0].y));
  int r0;
  if (dist[0] < dist[1]) r0 = dist[0] < dist[2] ? 0 : 2;
  else r0 = dist[1] < dist[2] ? 1 : 2;
  int r1 = (r0 + 1) % 3, r2 = (r1 + 1) % 3;
  // cyclic reorder by selects, so the vertices stay in registers
  const vtx<NA> R0 = pick3<NA>(r0, a, b, c);
  const vtx<NA> R1 = pick3<NA>(r1, a, b, c);
  const vtx<NA> R2 = pick3<NA>(r2, a, b, c);
  float e01[NA + 1][4], e02[NA + 1][4];
#pragma unroll
  for (int r = 0; r <= NA; ++r) {
    e01[r][0] = R1.r[r].x - R0.r[r].x; e01[r][1] = R1.r[r].y - R0.r[r].y;
    e01[r][2] = R1.r[r].z - R0.r[r].z; e01[r][3] = R1.r[r].w - R0.r[r].w;
    e02[r][0] = R2.r[r].x - R0.r[r].x; e02[r][1] = R2.r[r].y - R0.r[r].y;
    e02[r][2] = R2.r[r].z - R0.r[r].z; e02[r][3] = R2.r[r].w - R0.r[r].w;
  }
  float area = e02[0][0] * e01[0][1] - e02[0][1] * e01[0][0];
  t.valid = !equal_eps(area, 0.0f);
  if (!t.valid) return;
  t.front = area > 0.0f;
  float inv_area = 1.0f / area;
  t.bb[0] = std_min(std_min(a.r[0].x, b.r[0].x), c.r[0].x);
  t.bb[1] = std_max(std_max(a.r[0].x, b.r[0].x), c.r[0].x);
  t.bb[2] = std_min(std_min(a.r[0].y, b.r[0].y), c.r[0].y);
  t.bb[3] = std_max(std_max(a.r[0].y, b.r[0].y), c.r[0].y);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const float4& s = V[i]->r[0];
    const float4& e = V[(i + 1) % 3]->r[0];
    t.e[i][0] = s.y - e.y;
    t.e[i][1] = e.x - s.x;
    t.e[i][2] = e.x * s.y - e.y * s.x;
  }
  float e01x = e01[0][0], e01y = e01[0][1], e02x = e02[0][0], e02y = e02[0][1];
#pragma unroll
  for (int r = 0; r <= NA; ++r) {
    float dx[4], dy[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float xd = e02[r][k] * e01y - e01[r][k] * e02y;
      float yd = e01[r][k] * e02x - e02[r][k] * e01x;
      dx[k] = xd * inv_area;
      dy[k] = yd * inv_area;
    }
    t.ddx.r[r] = make_float4(dx[0], dx[1], dx[2], dx[3]);
    t.ddy.r[r] = make_float4(dy[0], dy[1], dy[2], dy[3]);
  }
  t.v0 = R0;
}

// compute_front (clipper.cpp:92-101)
__device__ __forceinline__ bool compute_front(float4 p0, float4 p1, float4 p2) {
  float i0 = 1.0f / p0.w, i1 = 1.0f / p1.w, i2 = 1.0f / p2.w;
  float x0 = p0.x * i0, y0 = p0.y * i0, x1 = p1.x * i1, y1 = p1.y * i1, x2 = p2.x * i2, y2 = p2.y * i2;
  float ax = x2 - x0, ay = y2 - y0, bx = x1 - x0, by = y1 - y0;
  return (ax * by - ay * bx) > 0.0f;
}

// Screen-space vertices of clipped triangle `id` (= 3 * primitive + fan index).
template <int NA>
__device__ __forceinline__ void load_clipped_triangle(const draw_params& P, const float4* vbuf, const uint8_t* clip_flag,
                                                      const int32_t* clip_slot, const float4* clip_verts,
                                                      const uint32_t* clip_hdr, uint32_t id, vtx<NA>* out) {
  uint32_t prim = id / 3, k = id - prim * 3;
  if (!clip_flag[prim]) {
    vtx<NA> v[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) load_vertex<NA>(P, vbuf, fetch_index(P, prim, i), v[i]);
    bool front = compute_front(v[0].r[0], v[1].r[0], v[2].r[0]);
    // winding normalisation (clipper.cpp:59-65) by selects
    out[0] = v[0];
    out[1] = vsel<NA>(front, v[1], v[2]);
    out[2] = vsel<NA>(front, v[2], v[1]);
#pragma unroll
    for (int i = 0; i < 3; ++i) viewport_project<NA>(out[i], P);
    return;
  }
  int32_t slot = clip_slot[prim];
  uint32_t hdr = clip_hdr[slot];
  bool front = (hdr >> 8) & 1;
  const float4* base = clip_verts + static_cast<size_t>(slot) * 5 * (NA + 1);
  int ia = 0, ib = static_cast<int>(k) + 1, ic = static_cast<int>(k) + 2;
  if (!front) {
    int tmp = ib;
    ib = ic;
    ic = tmp;
  }
  int idx[3] = {ia, ib, ic};
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int r = 0; r <= NA; ++r) out[i].r[r] = base[idx[i] * (NA + 1) + r];
}

// ============================================================== binning geometry
// Visits, in order, the GPU tiles that may hold pixels of a triangle, with the reference's
// 64x64 tile-level decision (threaded_dispatch_primitive, rasterizer.cpp:775-862).
// Binning of a triangle to GPU tiles.  The reference bins by 64x64 tile (rasterizer.cpp:947-994,
// the tile's corner test rejects or fully accepts it); a GPU tile of a partially covered 64x64 tile
// gets a record when its rows and columns meet the triangle's bounding box and one of its 16x16
// stage-16 regions passes the rasteriser's first subdivision test (subdivide_tile on the 64x64
// tile, rasterizer.cpp:662-675, the same float expressions as the visibility and raster kernels):
// a region that test rejects produces no fragment, so its record could change nothing.
// Larger triangles skip the region test: their partially covered 64x64 tiles are few next to the
// inner ones, and the test would lengthen the per-triangle counting loop.
constexpr int REGION_TEST_TILES = 16;
struct tri_bin {
  int sx, sy, ex, ey;  // 64x64 tiles [sx, ex) x [sy, ey)
  bool small;          // one 64x64 tile: the corner test is skipped (rasterizer.cpp:957)
  bool regions;        // at most REGION_TEST_TILES 64x64 tiles: GPU tiles are region-tested
  bool mx[3], my[3];
  float r2a[3], s1x[3], s1y[3];
};
__device__ __forceinline__ void bin_setup(const draw_params& P, const float* e, const float* bb, tri_bin& t) {
  const int tx = P.tiles_x, ty = P.tiles_y;
  t.sx = min(fast_floori(std_max(0.0f, bb[0]) / TILE), tx);
  t.sy = min(fast_floori(std_max(0.0f, bb[2]) / TILE), ty);
  t.ex = min(fast_ceili(std_max(0.0f, bb[1]) / TILE) + 1, tx);
  t.ey = min(fast_ceili(std_max(0.0f, bb[3]) / TILE) + 1, ty);
  t.small = (t.sx + 1 == t.ex) && (t.sy + 1 == t.ey);
  t.regions = (t.ex - t.sx) * (t.ey - t.sy) <= REGION_TEST_TILES;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float ex = e[k * 3 + 0], ey = e[k * 3 + 1];
    t.mx[k] = ex > 0;
    t.my[k] = ey > 0;
    float stx = TILE * ex, sty = TILE * ey;
    t.r2a[k] = -fabsf(stx) - fabsf(sty);
    stx *= 0.25f;
    sty *= 0.25f;
    t.s1x[k] = stx;
    t.s1y[k] = sty;
  }
}
// The GPU tiles of 64x64 tile (x, y) that get a record, bit j * sub + i for GPU tile (i, j) of it
// (row-major, the order records are written in); full: the tile is fully accepted.
__device__ __forceinline__ uint64_t tile_gmask(const draw_params& P, const float* e, const float* bb, const tri_bin& t,
                                               int x, int y, bool& full) {
  full = false;
  if (!t.small) {
    bool rej = false, acc = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      float ev = e[k * 3 + 2] - ((static_cast<float>(x + t.mx[k]) * TILE) * e[k * 3 + 0] +
                                 (static_cast<float>(y + t.my[k]) * TILE) * e[k * 3 + 1]);
      rej |= (0 < ev);
      acc &= (t.r2a[k] >= ev);
    }
    if (rej) return 0;
    full = acc;
  }
  const int sub = TILE / P.gt;
  const float xmin = bb[0] - static_cast<float>(x * TILE), xmax = bb[1] - static_cast<float>(x * TILE);
  const float ymin = bb[2] - static_cast<float>(y * TILE), ymax = bb[3] - static_cast<float>(y * TILE);
  uint32_t rows = 0, cols = 0;
  for (int j = 0; j < sub; ++j) {
    if (y * sub + j >= P.gtiles_y) break;
    if (full || !(ymin >= static_cast<float>(j * P.gt + P.gt) || ymax < static_cast<float>(j * P.gt))) rows |= 1u << j;
  }
  for (int i = 0; i < sub; ++i) {
    if (x * sub + i >= P.gtiles_x) break;
    if (full || !(xmin >= static_cast<float>(i * P.gt + P.gt) || xmax < static_cast<float>(i * P.gt))) cols |= 1u << i;
  }
  if (!rows || !cols) return 0;
  uint64_t all = 0;  // every GPU tile in the bounding-box rows and columns
  for (uint32_t rm = rows; rm; rm &= rm - 1) all |= static_cast<uint64_t>(cols) << (__builtin_ctz(rm) * sub);
  if (full || !t.regions) return all;
  // stage-16 regions the first subdivision rejects (bit ry * 4 + rx)
  uint32_t rrej = 0;
  {
    const float tvx = static_cast<float>(x * TILE), tvy = static_cast<float>(y * TILE);
    float ev1[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const float ex = e[k * 3], ey = e[k * 3 + 1], ez = e[k * 3 + 2];
      float part = static_cast<float>(t.mx[k] * TILE) * ex + static_cast<float>(t.my[k] * TILE) * ey;
      part *= 0.25f;
      ev1[k] = (ez - part) - ((tvx * ex) + (tvy * ey));
    }
    // regions inside the bounding-box rows and columns only
    const int r0 = (__builtin_ctz(rows) * P.gt) >> 4, r1 = ((31 - __builtin_clz(rows)) * P.gt + P.gt - 1) >> 4;
    const int c0 = (__builtin_ctz(cols) * P.gt) >> 4, c1 = ((31 - __builtin_clz(cols)) * P.gt + P.gt - 1) >> 4;
    for (int ry = r0; ry <= r1; ++ry)
      for (int rx = c0; rx <= c1; ++rx) {
        bool rej = false;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const float r = (t.s1x[k] * static_cast<float>(rx)) + (t.s1y[k] * static_cast<float>(ry));
          rej |= r < ev1[k];
        }
        if (rej) rrej |= 1u << (ry * 4 + rx);
      }
  }
  if (!rrej) return all;
  if (P.gt == 16) return all & ~static_cast<uint64_t>(rrej);  // GPU tile (i, j) is region (i, j)
  uint64_t m = 0;
  for (uint32_t rm = rows; rm; rm &= rm - 1) {
    const int j = __builtin_ctz(rm);
    const int ry0 = (j * P.gt) >> 4, ry1 = (j * P.gt + P.gt - 1) >> 4;
    for (uint32_t cm = cols; cm; cm &= cm - 1) {
      const int i = __builtin_ctz(cm);
      const int rx0 = (i * P.gt) >> 4, rx1 = (i * P.gt + P.gt - 1) >> 4;
      bool any = false;  // a region of the GPU tile the first subdivision keeps
      for (int ry = ry0; ry <= ry1; ++ry)
        for (int rx = rx0; rx <= rx1; ++rx) any |= !((rrej >> (ry * 4 + rx)) & 1u);
      if (any) m |= 1ull << (j * sub + i);
    }
  }
  return m;
}

template <class F>
__device__ __forceinline__ void for_each_gtile(const draw_params& P, const float* e, const float* bb, F&& f) {
  tri_bin t;
  bin_setup(P, e, bb, t);
  const int sub = TILE / P.gt;
  for (int y = t.sy; y < t.ey; ++y)
    for (int x = t.sx; x < t.ex; ++x) {
      bool full;
      for (uint64_t m = tile_gmask(P, e, bb, t, x, y, full); m; m &= m - 1) {
        const int b = __builtin_ctzll(m);
        f(static_cast<uint32_t>((y * sub + b / sub) * P.gtiles_x + x * sub + b % sub), full);
      }
    }
}

// 64x64 tiles in a triangle's bounding box (as bin_setup clamps it)
__device__ __forceinline__ int bin_span(const draw_params& P, const float* bb) {
  const int sx = min(fast_floori(std_max(0.0f, bb[0]) / TILE), P.tiles_x);
  const int sy = min(fast_floori(std_max(0.0f, bb[2]) / TILE), P.tiles_y);
  const int ex = min(fast_ceili(std_max(0.0f, bb[1]) / TILE) + 1, P.tiles_x);
  const int ey = min(fast_ceili(std_max(0.0f, bb[3]) / TILE) + 1, P.tiles_y);
  return (ex > sx && ey > sy) ? (ex - sx) * (ey - sy) : 0;
}
// Triangles over more than this many 64x64 tiles are counted by a whole wave (clip launch), not by
// setup's one lane.
constexpr int COUNT_WIDE = 32;

// count_gtiles by a whole wave (every lane calls it with the same triangle): lanes take the 64x64
// tiles, the wave sums their GPU tiles.
__device__ __forceinline__ uint32_t count_gtiles_wave(const draw_params& P, const float* e, const float* bb) {
  tri_bin t;
  bin_setup(P, e, bb, t);
  const int w = t.ex - t.sx;
  const int R = (t.ex > t.sx && t.ey > t.sy) ? w * (t.ey - t.sy) : 0;
  uint32_t n = 0;
  for (int tt = __lane_id(); tt < R; tt += 64) {
    bool full;
    n += static_cast<uint32_t>(__popcll(tile_gmask(P, e, bb, t, t.sx + tt % w, t.sy + tt / w, full)));
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) n += static_cast<uint32_t>(__shfl_xor(static_cast<int>(n), off, 64));
  return n;
}

// The number of GPU tiles for_each_gtile visits.
__device__ __forceinline__ uint32_t count_gtiles(const draw_params& P, const float* e, const float* bb) {
  tri_bin t;
  bin_setup(P, e, bb, t);
  uint32_t n = 0;
  for (int y = t.sy; y < t.ey; ++y)
    for (int x = t.sx; x < t.ex; ++x) {
      bool full;
      n += static_cast<uint32_t>(__popcll(tile_gmask(P, e, bb, t, x, y, full)));
    }
  return n;
}

// count_gtiles that also keeps the first four GPU tiles for_each_gtile visits, packed as
// tile << 1 | full (setup's pairs, which spare the emission the walk of triangles with at most four
// records).
constexpr uint32_t NO_PAIRS = 0xFFFFFFFFu;  // no tile is that large
__device__ __forceinline__ uint32_t count_gtiles_pairs(const draw_params& P, const float* e, const float* bb, uint4& k) {
  tri_bin t;
  bin_setup(P, e, bb, t);
  const int sub = TILE / P.gt;
  uint32_t n = 0;
  k = make_uint4(NO_PAIRS, NO_PAIRS, NO_PAIRS, NO_PAIRS);
  for (int y = t.sy; y < t.ey; ++y)
    for (int x = t.sx; x < t.ex; ++x) {
      bool full;
      uint64_t m = tile_gmask(P, e, bb, t, x, y, full);
      const uint32_t c = static_cast<uint32_t>(__popcll(m));
      for (uint32_t i = n; m && i < 4; m &= m - 1, ++i) {
        const int b = __builtin_ctzll(m);
        const uint32_t g = static_cast<uint32_t>((y * sub + b / sub) * P.gtiles_x + x * sub + b % sub);
        const uint32_t v = (g << 1) | (full ? 1u : 0u);
        if (i == 0) k.x = v;
        else if (i == 1) k.y = v;
        else if (i == 2) k.z = v;
        else k.w = v;
      }
      n += c;
    }
  return n;
}

template <int NA>
__device__ __forceinline__ void tri_rec_words(const tri_setup<NA>& t, float4 (&rec)[5]) {
  rec[0] = make_float4(t.e[0][0], t.e[0][1], t.e[0][2], t.e[1][0]);
  rec[1] = make_float4(t.e[1][1], t.e[1][2], t.e[2][0], t.e[2][1]);
  rec[2] = make_float4(t.e[2][2], t.bb[0], t.bb[1], t.bb[2]);
  rec[3] = make_float4(t.bb[3], t.v0.r[0].x, t.v0.r[0].y, t.v0.r[0].z);
  rec[4] = make_float4(t.ddx.r[0].z, t.ddy.r[0].z, t.front ? 1.0f : 0.0f, 0.0f);
}
template <int NA>
__device__ __forceinline__ void tri_attr_words(const tri_setup<NA>& t, float4 (&a)[3 * (NA + 1)]) {
#pragma unroll
  for (int r = 0; r <= NA; ++r) {
    a[r] = t.v0.r[r];
    a[NA + 1 + r] = t.ddx.r[r];
    a[2 * (NA + 1) + r] = t.ddy.r[r];
  }
}

template <int NA>
__device__ __forceinline__ void write_tri_rec(float4* rec, const tri_setup<NA>& t) {
  float4 w[5];
  tri_rec_words<NA>(t, w);
#pragma unroll
  for (int k = 0; k < 5; ++k) rec[k] = w[k];
}

template <int NA>
__device__ __forceinline__ void write_tri_attr(float4* a, const tri_setup<NA>& t) {
  float4 w[3 * (NA + 1)];
  tri_attr_words<NA>(t, w);
#pragma unroll
  for (int k = 0; k < 3 * (NA + 1); ++k) a[k] = w[k];
}

// Sum of v over the workgroup, returned to thread 0.  All threads must call it.
__device__ __forceinline__ uint32_t block_sum_u32(uint32_t v) {
  __shared__ uint32_t wsum[16];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), off, 64));
  const int wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  if ((threadIdx.x & 63) == 0) wsum[wave] = v;
  __syncthreads();
  uint32_t t = 0;
  if (threadIdx.x == 0)
    for (int w = 0; w < nw; ++w) t += wsum[w];
  return t;
}

// stats[slot] += sum(partial[0..n))
__global__ void __launch_bounds__(256) reduce_partials_kernel(const unsigned long long* __restrict__ partial, uint32_t n,
                                                               unsigned long long* __restrict__ stats, int slot) {
  __shared__ unsigned long long wsum[4];
  unsigned long long t = 0;
  for (uint32_t i = threadIdx.x; i < n; i += 256) t += partial[i];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = t;
  __syncthreads();
  if (threadIdx.x == 0) stats[slot] += wsum[0] + wsum[1] + wsum[2] + wsum[3];
}

// ============================================================== setup (fast path)
template <int NA>
__device__ __forceinline__ void setup_body(const draw_params& P, const float4* __restrict__ vbuf, float4* __restrict__ tri_rec,
                                           float4* __restrict__ tri_attr, uint32_t* __restrict__ cnt,
                                           uint8_t* __restrict__ clip_flag, uint32_t* __restrict__ counters,
                                           uint32_t* __restrict__ wide_list, unsigned long long* __restrict__ partial,
                                           uint32_t* __restrict__ bsum, uint4* __restrict__ pairs, uint32_t bx) {
  uint32_t p = bx * blockDim.x + threadIdx.x;
  unsigned long long cprims = 0;
  float4 rec[5], attr[3 * (NA + 1)];  // this lane's setup words, stored by the whole wave below
  bool have = false;
  uint32_t c0 = 0;  // records of fan triangle 0 counted here
  uint4 kp = make_uint4(NO_PAIRS, NO_PAIRS, NO_PAIRS, NO_PAIRS);  // its first four (tile, full) pairs
  if (p < P.prim_count) {
    cnt[3 * p + 1] = 0;
    cnt[3 * p + 2] = 0;
    vtx<NA> v[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) load_vertex<NA>(P, vbuf, fetch_index(P, p, i), v[i]);
    // near (0,0,1,0) and far (0,0,-1,1) planes (clipper.cpp:21-27,104-120)
    const float4 pn = make_float4(0.0f, 0.0f, 1.0f, 0.0f), pf = make_float4(0.0f, 0.0f, -1.0f, 1.0f);
    bool in = true;
#pragma unroll
    for (int i = 0; i < 3; ++i) in &= !(dot4(pn, v[i].r[0]) < 0);
    if (in)
#pragma unroll
      for (int i = 0; i < 3; ++i) in &= !(dot4(pf, v[i].r[0]) < 0);
    clip_flag[p] = in ? 0 : 1;
    if (!in) {
      atomicAdd(&counters[CT_CLIP_PRIMS], 1u);
    } else {
      bool front = compute_front(v[0].r[0], v[1].r[0], v[2].r[0]);
      if (!cull_fn(P, front ? 1.0f : -1.0f)) {
        cprims = 1;
        // winding normalisation (clipper.cpp:59-65) by selects
        vtx<NA> o[3] = {v[0], vsel<NA>(front, v[1], v[2]), vsel<NA>(front, v[2], v[1])};
#pragma unroll
        for (int i = 0; i < 3; ++i) viewport_project<NA>(o[i], P);
        tri_setup<NA> t;
        triangle_info<NA>(o[0], o[1], o[2], t);
        if (t.valid) {
          have = true;
          tri_rec_words<NA>(t, rec);
          tri_attr_words<NA>(t, attr);
          float e[9], bb[4];
          for (int i = 0; i < 3; ++i)
            for (int j = 0; j < 3; ++j) e[i * 3 + j] = t.e[i][j];
          for (int i = 0; i < 4; ++i) bb[i] = t.bb[i];
          if (bin_span(P, bb) > COUNT_WIDE)
            wide_list[atomicAdd(&counters[CT_WIDE], 1u)] = p;  // counted in the clip launch
          else if (pairs)
            c0 = count_gtiles_pairs(P, e, bb, kp);
          else
            c0 = count_gtiles(P, e, bb);
        }
      }
    }
    cnt[3 * p] = c0;
    if (pairs) {
      if (c0 > 4u) kp.x = NO_PAIRS;
      pairs[p] = kp;
    }
  }
  // The fan-0 slots of the wave's 64 consecutive primitives are consecutive: store the set-up
  // triangles' words coalesced (blockDim.x is 256).
  {
    __shared__ float4 stage[4 * WAVE_STAGE];
    const uint64_t mask = __ballot(have);
    if (mask) {
      const size_t p0 = static_cast<size_t>(bx) * blockDim.x + (threadIdx.x & ~63u);
      float4* ws = stage + (threadIdx.x >> 6) * WAVE_STAGE;
      wave_store_blocks<5>(tri_rec + p0 * 5, rec, mask, ws);
      wave_store_blocks<3 * (NA + 1)>(tri_attr + p0 * 3 * (NA + 1), attr, mask, ws);
    }
  }
  if (bsum) {  // uniform over the launch: the block's total; the clip launch adds the counts it makes
    const uint32_t t = block_sum_u32(c0);
    if (threadIdx.x == 0) bsum[bx] = t;
  }
  if (P.count_stats) block_partial(partial, cprims);  // uniform over the launch
}
template <int NA>
__global__ void __launch_bounds__(256) setup_kernel(draw_params P, const float4* __restrict__ vbuf, float4* __restrict__ tri_rec,
                                                     float4* __restrict__ tri_attr,
                                                     uint32_t* __restrict__ cnt, uint8_t* __restrict__ clip_flag,
                                                     uint32_t* __restrict__ counters, uint32_t* __restrict__ wide_list,
                                                     unsigned long long* __restrict__ partial, uint32_t* __restrict__ bsum,
                                                     uint4* __restrict__ pairs) {
  setup_body<NA>(P, vbuf, tri_rec, tri_attr, cnt, clip_flag, counters, wide_list, partial, bsum, pairs, blockIdx.x);
}

// ============================================================== clipping (slow path)
template <int NA>
__device__ __forceinline__ void lerp_vtx(vtx<NA>& o, const vtx<NA>& a, const vtx<NA>& b, float t, const draw_params& P) {
  o.r[0] = make_float4(a.r[0].x + (b.r[0].x - a.r[0].x) * t, a.r[0].y + (b.r[0].y - a.r[0].y) * t,
                       a.r[0].z + (b.r[0].z - a.r[0].z) * t, a.r[0].w + (b.r[0].w - a.r[0].w) * t);
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    o.r[i + 1] = a.r[i + 1];
    if (!(P.attr_mod[i] & AM_NOINTERPOLATION))
      o.r[i + 1] = make_float4(o.r[i + 1].x + (b.r[i + 1].x - a.r[i + 1].x) * t, o.r[i + 1].y + (b.r[i + 1].y - a.r[i + 1].y) * t,
                               o.r[i + 1].z + (b.r[i + 1].z - a.r[i + 1].z) * t, o.r[i + 1].w + (b.r[i + 1].w - a.r[i + 1].w) * t);
  }
}

// clip_triangle_to_poly_general + clip_solid_triangle (clipper.cpp:43-228) for primitive p
template <int NA>
__device__ uint32_t clip_primitive(const draw_params& P, uint32_t p, const float4* __restrict__ vbuf, float4* __restrict__ tri_rec,
                                   float4* __restrict__ tri_attr, int32_t* __restrict__ clip_slot,
                               float4* __restrict__ clip_verts, uint32_t* __restrict__ clip_hdr, uint32_t capacity,
                               uint32_t* __restrict__ counters, unsigned long long* __restrict__ stats) {
  vtx<NA> cv[2][5];
  uint32_t nc[2] = {3, 0};
  for (int i = 0; i < 3; ++i) load_vertex<NA>(P, vbuf, fetch_index(P, p, i), cv[0][i]);
  const float4 planes[2] = {make_float4(0.0f, 0.0f, 1.0f, 0.0f), make_float4(0.0f, 0.0f, -1.0f, 1.0f)};
  int src = 0, dst = 1;
  bool front = false;
  for (int pl = 0; pl < 2; ++pl) {
    nc[dst] = 0;
    float d0 = 0.0f;
    if (nc[src] != 0) d0 = dot4(planes[pl], cv[src][0].r[0]);
    for (uint32_t i = 0, j = 1; i < nc[src]; ++i, ++j) {
      j %= nc[src];
      float d1 = dot4(planes[pl], cv[src][j].r[0]);
      if (d0 >= 0.0f) {
        cv[dst][nc[dst]++] = cv[src][i];
        if (d1 < 0.0f) lerp_vtx<NA>(cv[dst][nc[dst]++], cv[src][i], cv[src][j], d0 / (d0 - d1), P);
      } else if (d1 >= 0.0f) {
        lerp_vtx<NA>(cv[dst][nc[dst]++], cv[src][j], cv[src][i], d1 / (d1 - d0), P);
      }
      d0 = d1;
    }
    if (pl == 0 && nc[dst] >= 3) {
      float px[3], py[3];
      for (int v = 0; v < 3; ++v) {
        float iaw = 1 / fabsf(cv[dst][v].r[0].w);
        px[v] = cv[dst][v].r[0].x * iaw;
        py[v] = cv[dst][v].r[0].y * iaw;
      }
      float ax = px[2] - px[0], ay = py[2] - py[0], bx = px[1] - px[0], by = py[1] - py[0];
      float area = ax * by - ay * bx;
      front = area > 0.0f;
      if (cull_fn(P, area)) return 0;
    }
    src ^= 1;
    dst ^= 1;
  }
  uint32_t n = nc[src];
  if (n < 3) return 0;
  atomicAdd(&stats[ST_CPRIMITIVES], static_cast<unsigned long long>(n - 2));
  uint32_t slot = atomicAdd(&counters[CT_CLIP_SLOTS], 1u);
  if (slot >= capacity) {
    atomicAdd(&counters[CT_CLIP_OVERFLOW], 1u);
    return 0;
  }
  clip_slot[p] = static_cast<int32_t>(slot);
  clip_hdr[slot] = n | (front ? 0x100u : 0u);
  float4* out = clip_verts + static_cast<size_t>(slot) * 5 * (NA + 1);
  for (uint32_t i = 0; i < n; ++i) {
    viewport_project<NA>(cv[src][i], P);  // once per polygon vertex, as for the unique vertices
    for (int r = 0; r <= NA; ++r) out[i * (NA + 1) + r] = cv[src][i].r[r];
  }
  uint32_t fans = 0;
  for (uint32_t t = 1; t + 1 < n; ++t) {
    const vtx<NA>& a = cv[src][0];
    const vtx<NA>& b = front ? cv[src][t] : cv[src][t + 1];
    const vtx<NA>& c = front ? cv[src][t + 1] : cv[src][t];
    tri_setup<NA> ts;
    triangle_info<NA>(a, b, c, ts);
    uint32_t id = 3 * p + (t - 1);
    if (!ts.valid) continue;
    write_tri_rec<NA>(tri_rec + tri_slot(P, id) * 5, ts);
    write_tri_attr<NA>(tri_attr + tri_slot(P, id) * 3 * (NA + 1), ts);
    fans |= 1u << (t - 1);
  }
  return fans;
}

// Clipping launch: a bounded grid strides over the primitives setup flagged (none, usually).  With
// `bsum` (single draws) the counts it makes are added to their 256-primitive block's total.
template <int NA>
__device__ __forceinline__ void clip_work(const draw_params& P, const float4* __restrict__ vbuf, float4* __restrict__ tri_rec,
                                          float4* __restrict__ tri_attr, uint32_t* __restrict__ cnt,
                                          const uint8_t* __restrict__ clip_flag, int32_t* __restrict__ clip_slot,
                                          float4* __restrict__ clip_verts, uint32_t* __restrict__ clip_hdr, uint32_t capacity,
                                          uint32_t* __restrict__ counters, unsigned long long* __restrict__ stats,
                                          const uint32_t* __restrict__ wide_list, uint32_t* __restrict__ bsum,
                                          uint32_t nclip, uint32_t nwide, uint32_t bx, uint32_t gx) {
  // triangles over many 64x64 tiles: one wave counts each one's records
  const uint32_t wave = (bx * blockDim.x + threadIdx.x) >> 6, waves = (gx * blockDim.x) >> 6;
  for (uint32_t w = wave; w < nwide; w += waves) {
    const uint32_t p = wide_list[w];
    float e[9], bb[4];
    read_tri_rec(tri_rec + static_cast<size_t>(p) * 5, e, bb);  // fan 0 of primitive p
    const uint32_t n = count_gtiles_wave(P, e, bb);
    if (__lane_id() == 0) {
      cnt[3 * p] = n;
      if (bsum) atomicAdd(&bsum[p / 256], n);
    }
  }
  if (nclip == 0) return;
  // lanes clip the flagged primitives among the wave's 64; the wave then counts the records of the
  // resulting triangles together (clipped triangles are few and often reach across the target)
  const int lane = __lane_id();
  for (uint32_t b = wave * 64; b < P.prim_count; b += waves * 64) {
    const uint32_t p = b + static_cast<uint32_t>(lane);
    uint32_t fans = 0;  // bit k: fan triangle 3p + k was set up
    if (p < P.prim_count && clip_flag[p])
      fans = clip_primitive<NA>(P, p, vbuf, tri_rec, tri_attr, clip_slot, clip_verts, clip_hdr, capacity, counters, stats);
    __threadfence();  // the fans' records are read back by every lane of the wave
    for (unsigned long long m = __ballot(fans != 0); m; m &= m - 1) {
      const int src = __builtin_ctzll(m);
      const uint32_t fs = static_cast<uint32_t>(__shfl(static_cast<int>(fans), src, 64));
      const uint32_t ps = b + static_cast<uint32_t>(src);
      for (int k = 0; k < 3; ++k) {
        if (!(fs & (1u << k))) continue;
        const uint32_t id = 3 * ps + k;
        float e[9], bb[4];
        read_tri_rec(tri_rec + tri_slot(P, id) * 5, e, bb);
        const uint32_t n = count_gtiles_wave(P, e, bb);
        if (lane == 0) {
          cnt[id] = n;
          if (bsum) atomicAdd(&bsum[ps / 256], n);
        }
      }
    }
  }
}

// counters[CT_TOTAL] = the sum of the block totals (every thread of the workgroup calls it).
__device__ __forceinline__ void record_total(const draw_params& P, const uint32_t* __restrict__ bsum,
                                             uint32_t* __restrict__ counters) {
  const uint32_t nb = (P.prim_count + 255) / 256;
  uint32_t t = 0;
  for (uint32_t i0 = 0; i0 < nb; i0 += 8 * blockDim.x) {
    uint32_t v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t i = i0 + k * blockDim.x + threadIdx.x;
      const uint32_t x = __hip_atomic_load(bsum + min(i, nb - 1u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      v[k] = i < nb ? x : 0u;  // no branch per load (see load_or_zero)
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) t += v[k];
  }
  t = block_sum_u32(t);
  if (threadIdx.x == 0) counters[CT_TOTAL] = t;
}

template <int NA>
__device__ __forceinline__ void clip_body(const draw_params& P, const float4* __restrict__ vbuf, float4* __restrict__ tri_rec,
                                          float4* __restrict__ tri_attr, uint32_t* __restrict__ cnt,
                                          const uint8_t* __restrict__ clip_flag, int32_t* __restrict__ clip_slot,
                                          float4* __restrict__ clip_verts, uint32_t* __restrict__ clip_hdr, uint32_t capacity,
                                          uint32_t* __restrict__ counters, unsigned long long* __restrict__ stats,
                                          const uint32_t* __restrict__ wide_list, uint32_t* __restrict__ bsum, uint32_t bx,
                                          uint32_t gx) {
  const uint32_t nclip = counters[CT_CLIP_PRIMS], nwide = counters[CT_WIDE];
  const bool flagged = nclip != 0 || nwide != 0;  // uniform over the launch
  if (flagged)
    clip_work<NA>(P, vbuf, tri_rec, tri_attr, cnt, clip_flag, clip_slot, clip_verts, clip_hdr, capacity, counters, stats,
                  wide_list, bsum, nclip, nwide, bx, gx);
  if (!bsum) return;
  // single draws: the record total, once every workgroup's counts are in the block totals (the last
  // workgroup to finish sums them; with nothing flagged, setup's totals are final and workgroup 0 does)
  if (flagged) {
    __shared__ uint32_t s_last;
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0) s_last = atomicAdd(&counters[CT_CLIP_DONE], 1u) == gx - 1 ? 1u : 0u;
    __syncthreads();
    if (!s_last) return;
    __threadfence();
  } else if (bx != 0) {
    return;
  }
  record_total(P, bsum, counters);
}
template <int NA>
__global__ void clip_kernel(draw_params P, const float4* __restrict__ vbuf, float4* __restrict__ tri_rec,
                            float4* __restrict__ tri_attr, uint32_t* __restrict__ cnt, const uint8_t* __restrict__ clip_flag, int32_t* __restrict__ clip_slot,
                            float4* __restrict__ clip_verts, uint32_t* __restrict__ clip_hdr, uint32_t capacity,
                            uint32_t* __restrict__ counters, unsigned long long* __restrict__ stats,
                            const uint32_t* __restrict__ wide_list, uint32_t* __restrict__ bsum) {
  clip_body<NA>(P, vbuf, tri_rec, tri_attr, cnt, clip_flag, clip_slot, clip_verts, clip_hdr, capacity, counters, stats,
                wide_list, bsum, blockIdx.x, gridDim.x);
}

// ============================================================== record emission
// off: exclusive scan of the per-triangle record counts; a triangle owns [off[id], off[id+1]).
// One thread per primitive, over its (at most 3) clipped triangles in fan order.  Records beyond
// `capacity` are dropped; the host compares the total with it and emits again.

// Records of one clipped triangle emitted by a whole wave: lanes take the triangle's 64x64 tiles in
// for_each_gtile's order, count each tile's GPU tiles with the same tests, and write at their
// wave-scanned offsets -- for triangles that reach many tiles, which one lane would walk serially.
__device__ __forceinline__ void emit_wide(const draw_params& P, const float4* __restrict__ tri_rec, uint32_t id,
                                          uint32_t first, uint32_t next, uint32_t capacity,
                                          uint32_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  const int lane = __lane_id();
  float e[9], bb[4];
  read_tri_rec(tri_rec + tri_slot(P, id) * 5, e, bb);
  tri_bin t;
  bin_setup(P, e, bb, t);
  const int sub = TILE / P.gt, w = t.ex - t.sx;
  const int R = (t.ex > t.sx && t.ey > t.sy) ? w * (t.ey - t.sy) : 0;
  uint32_t base = first;
  for (int t0 = 0; t0 < R; t0 += 64) {
    const int tt = t0 + lane;
    uint64_t m = 0;
    bool full = false;
    int x = 0, y = 0;
    if (tt < R) {
      x = t.sx + tt % w;
      y = t.sy + tt / w;
      m = tile_gmask(P, e, bb, t, x, y, full);
    }
    const uint32_t cnt = static_cast<uint32_t>(__popcll(m));
    const uint32_t incl = wave_incl_scan(cnt);
    uint32_t o = base + incl - cnt;
    for (; m; m &= m - 1) {
      const int b = __builtin_ctzll(m);
      if (o < next && o < capacity) {
        keys[o] = static_cast<uint32_t>((y * sub + b / sub) * P.gtiles_x + x * sub + b % sub);
        vals[o] = (id << 1) | (full ? 1u : 0u);
      }
      ++o;
    }
    base += static_cast<uint32_t>(__shfl(static_cast<int>(incl), 63, 64));
  }
}

// Records beyond which a triangle is emitted by its whole wave (so is any triangle over more than
// COUNT_WIDE 64x64 tiles).
constexpr uint32_t EMIT_WIDE = 64;

// Records of primitive p's fan triangles: triangle 3p+k owns [o[k], o[k+1]).  Every lane of the wave
// calls it (p >= prim_count: nothing of its own).
// pr: setup's first four (tile << 1 | full) pairs of fan triangle 0, pr.x == NO_PAIRS when it kept
// none (then, and for the other fan triangles, the tiles are walked again).
__device__ __forceinline__ void emit_records(const draw_params& P, const float4* __restrict__ tri_rec, uint32_t p,
                                             const uint32_t (&o)[4], uint4 pr, uint32_t capacity,
                                             uint32_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  uint32_t wide = 0;  // fan triangles left to the wave
  if (p < P.prim_count) {
    const uint32_t id3 = 3 * p;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const uint32_t id = id3 + k;
      const uint32_t first = o[k], next = o[k + 1];
      if (next == first) continue;
      if (k == 0 && pr.x != NO_PAIRS) {  // at most four records, as setup's walk found them
        const uint32_t v[4] = {pr.x, pr.y, pr.z, pr.w};
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i)
          if (first + i < next && first + i < capacity) {
            keys[first + i] = v[i] >> 1;
            vals[first + i] = (id << 1) | (v[i] & 1u);
          }
        continue;
      }
      if (next - first > EMIT_WIDE) {
        wide |= 1u << k;
        continue;
      }
      float e[9], bb[4];
      read_tri_rec(tri_rec + tri_slot(P, id) * 5, e, bb);
      if (bin_span(P, bb) > COUNT_WIDE) {  // few records over a large box: the walk is over the box
        wide |= 1u << k;
        continue;
      }
      uint32_t q = first;
      for_each_gtile(P, e, bb, [&](uint32_t g, bool full) {
        if (q < next && q < capacity) {  // the enumeration repeats the counting pass exactly
          keys[q] = g;
          vals[q] = (id << 1) | (full ? 1u : 0u);
        }
        ++q;
      });
    }
  }
  // every lane of the wave takes part in its lanes' wide triangles, one after another
  unsigned long long pending = __ballot(wide != 0);
  while (pending) {
    const int src = __ffsll(static_cast<long long>(pending)) - 1;
    pending &= pending - 1;
    const uint32_t ws = static_cast<uint32_t>(__shfl(static_cast<int>(wide), src, 64));
    const uint32_t ps = static_cast<uint32_t>(__shfl(static_cast<int>(p), src, 64));
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      if (!(ws & (1u << k))) continue;
      const uint32_t first = static_cast<uint32_t>(__shfl(static_cast<int>(o[k]), src, 64));
      const uint32_t next = static_cast<uint32_t>(__shfl(static_cast<int>(o[k + 1]), src, 64));
      emit_wide(P, tri_rec, 3 * ps + k, first, next, capacity, keys, vals);
    }
  }
}
// off: exclusive scan of the counts, followed by the total (batches)
__device__ __forceinline__ void emit_body(const draw_params& P, const float4* __restrict__ tri_rec,
                                          const uint32_t* __restrict__ off, const uint32_t* __restrict__ total,
                                          uint32_t capacity, uint32_t* __restrict__ keys, uint32_t* __restrict__ vals,
                                          uint32_t bx) {
  const uint32_t p = bx * blockDim.x + threadIdx.x;
  const uint32_t n = 3 * P.prim_count;
  uint32_t o[4] = {0, 0, 0, 0};
  if (p < P.prim_count) {
    const uint32_t id3 = 3 * p;
    o[0] = off[id3];
    o[1] = off[id3 + 1];
    o[2] = off[id3 + 2];
    o[3] = (id3 + 3 < n) ? off[id3 + 3] : *total;
  }
  emit_records(P, tri_rec, p, o, make_uint4(NO_PAIRS, NO_PAIRS, NO_PAIRS, NO_PAIRS), capacity, keys, vals);
}
// Single draws: the offsets come from the counts of the workgroup's 256 primitives (a workgroup
// scan) and the totals of the blocks before it, which setup and the clip launch left in `bsum`, so
// no scan of the counts runs: triangle id's first record is the sum of the counts of the triangles
// before it, as an exclusive scan of the counts gives it.
__global__ void __launch_bounds__(256) emit_kernel(draw_params P, const float4* __restrict__ tri_rec,
                                                   const uint32_t* __restrict__ cnt, const uint32_t* __restrict__ bsum,
                                                   const uint4* __restrict__ pairs, uint32_t capacity,
                                                   uint32_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  __shared__ uint32_t wtot[4], wbefore[4];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t p = blockIdx.x * 256 + tid;
  uint32_t c[3] = {0, 0, 0};
  uint4 pr = make_uint4(NO_PAIRS, NO_PAIRS, NO_PAIRS, NO_PAIRS);
  if (p < P.prim_count) {
    c[0] = cnt[3 * p];
    c[1] = cnt[3 * p + 1];
    c[2] = cnt[3 * p + 2];
    pr = pairs[p];
  }
  uint32_t before = 0;  // records of the blocks before this one
  for (uint32_t i0 = 0; i0 < blockIdx.x; i0 += 4 * 256) {
    uint32_t v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t i = i0 + k * 256 + tid;
      v[k] = load_or_zero(bsum, i, blockIdx.x);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) before += v[k];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) before += static_cast<uint32_t>(__shfl_xor(static_cast<int>(before), off, 64));
  const uint32_t t = c[0] + c[1] + c[2];
  const uint32_t incl = wave_incl_scan(t);
  if (lane == 63) {
    wtot[wave] = incl;
    wbefore[wave] = before;
  }
  __syncthreads();
  uint32_t o[4];
  o[0] = wbefore[0] + wbefore[1] + wbefore[2] + wbefore[3] + incl - t;
  for (uint32_t w = 0; w < wave; ++w) o[0] += wtot[w];
  o[1] = o[0] + c[0];
  o[2] = o[1] + c[1];
  o[3] = o[2] + c[2];
  emit_records(P, tri_rec, p, o, pr, capacity, keys, vals);
}

__global__ void fill_u32_kernel(uint32_t* p, uint32_t n, uint32_t v) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// ============================================================== scan (exclusive, u32)
constexpr int SCAN_PER_THREAD = 16;
static_assert(SCAN_PER_THREAD % 4 == 0, "scan blocks move as 16-byte words");
constexpr int SCAN_BLOCK = 256 * SCAN_PER_THREAD;  // elements per workgroup

// Exclusive scan of one SCAN_BLOCK-element block in place.  The block total goes to sums[block]
// (when sums is given); a single-block launch also stores it to *total.
__global__ void __launch_bounds__(256) scan_block_kernel(uint32_t* data, uint32_t n, uint32_t* sums, uint32_t* total) {
  __shared__ uint32_t wsum[4];
  // 64-bit positions: n may come within one block of 2^32
  const uint64_t base = static_cast<uint64_t>(blockIdx.x) * SCAN_BLOCK + threadIdx.x * SCAN_PER_THREAD;
  // a full block of 16-byte-aligned data moves as four 16-byte words per lane
  const bool vec = (static_cast<uint64_t>(blockIdx.x) + 1) * SCAN_BLOCK <= n && (reinterpret_cast<uintptr_t>(data) & 15) == 0;
  uint32_t v[SCAN_PER_THREAD];
  uint32_t t = 0;
  if (vec) {
    const uint4* d4 = reinterpret_cast<const uint4*>(data + base);
#pragma unroll
    for (int i = 0; i < SCAN_PER_THREAD / 4; ++i) {
      const uint4 q = d4[i];
      v[4 * i] = q.x;
      v[4 * i + 1] = q.y;
      v[4 * i + 2] = q.z;
      v[4 * i + 3] = q.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < SCAN_PER_THREAD; ++i) v[i] = (base + i < n) ? data[base + i] : 0u;
  }
#pragma unroll
  for (int i = 0; i < SCAN_PER_THREAD; ++i) t += v[i];
  const uint32_t incl = wave_incl_scan(t);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 63) wsum[wave] = incl;
  __syncthreads();
  uint32_t wprefix = 0;
  for (int w = 0; w < wave; ++w) wprefix += wsum[w];
  uint32_t run = wprefix + incl - t;
#pragma unroll
  for (int i = 0; i < SCAN_PER_THREAD; ++i) {
    const uint32_t x = v[i];
    v[i] = run;
    run += x;
  }
  if (vec) {
    uint4* d4 = reinterpret_cast<uint4*>(data + base);
#pragma unroll
    for (int i = 0; i < SCAN_PER_THREAD / 4; ++i) d4[i] = make_uint4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
  } else {
#pragma unroll
    for (int i = 0; i < SCAN_PER_THREAD; ++i)
      if (base + i < n) data[base + i] = v[i];
  }
  if (threadIdx.x == 255) {
    const uint32_t block_total = wprefix + incl;
    if (sums) sums[blockIdx.x] = block_total;
    if (total && gridDim.x == 1) *total = block_total;
  }
}

__global__ void __launch_bounds__(256) scan_add_kernel(uint32_t* data, uint32_t n, const uint32_t* sums) {
  const uint32_t add = sums[blockIdx.x];
  const uint64_t b0 = static_cast<uint64_t>(blockIdx.x) * SCAN_BLOCK;
#pragma unroll
  for (int k = 0; k < SCAN_PER_THREAD; ++k) {
    const uint64_t i = b0 + k * 256 + threadIdx.x;
    if (i < n) data[i] += add;
  }
}

size_t scan_tmp_size(uint32_t n) {
  size_t total = 0;
  uint64_t m = n;
  while (true) {
    const uint64_t nb = (m + SCAN_BLOCK - 1) / SCAN_BLOCK;
    if (nb <= 1) break;
    total += nb;
    m = nb;
  }
  return total + 4;
}

// Reduce-then-scan: blocks scan in place, the block totals are scanned the same way (one block up
// to SCAN_BLOCK^2 elements), then added back.  The top-level single block yields the total.
static void scan_rec(uint32_t* data, uint32_t n, uint32_t* tmp, uint32_t* total_dev, hipStream_t s) {
  const uint32_t nb = static_cast<uint32_t>((static_cast<uint64_t>(n) + SCAN_BLOCK - 1) / SCAN_BLOCK);
  if (nb <= 1) {
    hipLaunchKernelGGL(scan_block_kernel, dim3(1), dim3(256), 0, s, data, n, nullptr, total_dev);
    return;
  }
  uint32_t* sums = tmp;
  hipLaunchKernelGGL(scan_block_kernel, dim3(nb), dim3(256), 0, s, data, n, sums, nullptr);
  scan_rec(sums, nb, tmp + nb, total_dev, s);
  hipLaunchKernelGGL(scan_add_kernel, dim3(nb), dim3(256), 0, s, data, n, sums);
}

void launch_exclusive_scan(uint32_t* data, uint32_t n, uint32_t* tmp, uint32_t* total_dev, hipStream_t s) {
  scan_rec(data, n, tmp, total_dev, s);
}

// ============================================================== radix sort (stable LSD, 8-bit digits)
constexpr int SORT_BLOCK = 4096;  // 256 threads x 16 items

__global__ void __launch_bounds__(256) radix_hist_kernel(const uint32_t* __restrict__ keys, uint32_t n, int shift,
                                                          uint32_t nblocks, uint32_t* __restrict__ hist) {
  __shared__ uint32_t cnt[256];
  cnt[threadIdx.x] = 0;
  __syncthreads();
  uint32_t b0 = blockIdx.x * SORT_BLOCK;
  uint32_t end = min(n, b0 + SORT_BLOCK);
  for (uint32_t i = b0 + threadIdx.x; i < end; i += 256) atomicAdd(&cnt[(keys[i] >> shift) & 255u], 1u);
  __syncthreads();
  hist[threadIdx.x * nblocks + blockIdx.x] = cnt[threadIdx.x];
}

// Each wave ranks its 1024 consecutive items in 16 rounds of 64; a lane finds the lanes sharing its
// digit with eight ballots (one per digit bit), so ranks follow input order (stability) at a cost
// independent of how many digits a round holds.
__global__ void __launch_bounds__(256) radix_scatter_kernel(const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
                                                             uint32_t n, int shift, uint32_t nblocks,
                                                             const uint32_t* __restrict__ hist_scanned,
                                                             uint32_t* __restrict__ kout, uint32_t* __restrict__ vout) {
  __shared__ uint32_t wcnt[4][256];
  int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int i = threadIdx.x; i < 4 * 256; i += 256) (&wcnt[0][0])[i] = 0;
  __syncthreads();
  uint32_t base = blockIdx.x * SORT_BLOCK + wave * 1024;
  uint32_t rank[16], key[16], val[16];
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    uint32_t i = base + r * 64 + lane;
    bool valid = i < n;
    key[r] = valid ? kin[i] : 0u;
    val[r] = valid ? vin[i] : 0u;
    uint32_t d = (key[r] >> shift) & 255u;
    // m: the valid lanes holding this lane's digit, from one ballot per digit bit
    uint64_t m = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const bool bit = ((d >> b) & 1u) != 0;
      const uint64_t bal = __ballot(bit);
      m &= bit ? bal : ~bal;
    }
    const uint32_t before = valid ? wcnt[wave][d] : 0u;
    rank[r] = before + static_cast<uint32_t>(__popcll(m & lt));
    __builtin_amdgcn_wave_barrier();
    if (valid && (m & lt) == 0) wcnt[wave][d] = before + static_cast<uint32_t>(__popcll(m));  // lowest lane of the digit
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  {
    uint32_t d = threadIdx.x, s = 0;
    for (int w = 0; w < 4; ++w) {
      uint32_t c = wcnt[w][d];
      wcnt[w][d] = s;
      s += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    uint32_t i = base + r * 64 + lane;
    if (i < n) {
      uint32_t d = (key[r] >> shift) & 255u;
      uint32_t pos = hist_scanned[d * nblocks + blockIdx.x] + wcnt[wave][d] + rank[r];
      if (pos < n) {
        kout[pos] = key[r];
        vout[pos] = val[r];
      }
    }
  }
}

int launch_sort(const draw_buffers& B, uint32_t n, int bits, hipStream_t s) {
  int cur = 0;
  if (n == 0) return cur;
  uint32_t nblocks = (n + SORT_BLOCK - 1) / SORT_BLOCK;
  for (int shift = 0; shift < bits; shift += 8) {
    hipLaunchKernelGGL(radix_hist_kernel, dim3(nblocks), dim3(256), 0, s, B.keys[cur], n, shift, nblocks, B.hist);
    launch_exclusive_scan(B.hist, 256 * nblocks, B.scan_tmp, nullptr, s);
    hipLaunchKernelGGL(radix_scatter_kernel, dim3(nblocks), dim3(256), 0, s, B.keys[cur], B.vals[cur], n, shift, nblocks,
                       B.hist, B.keys[cur ^ 1], B.vals[cur ^ 1]);
    cur ^= 1;
  }
  return cur;
}

// [ts, te) of every GPU tile in the sorted records.  With T > 0 the thread at the last record of a
// tile (or before the first record) also writes the empty ranges of the tiles up to the next
// record's tile, so every tile is written exactly once without a separate clear (dense records).
// ---------------------------------------------------------------- one-pass bucket sort by GPU tile
// For the order-independent path the order of a tile's records is immaterial, so one counting pass
// replaces the stable radix passes: per-workgroup tile histograms in LDS, one scan of the
// tile-major histogram, and a scatter whose in-workgroup ranks come from LDS atomics.
constexpr int BUCKET_PER_THREAD = 16;
constexpr int BUCKET_ITEMS = 256 * BUCKET_PER_THREAD;  // records per workgroup
constexpr uint32_t BUCKET_MAX_TILES = 8192;

// PT records per thread: 256 * PT records per workgroup (the batched path tunes PT)
// Column of workgroup b in a tile's row of the bucket histogram: the workgroups of one XCD
// (b mod 8, as workgroups are dealt to the XCDs) take adjacent columns, so each histogram line is
// written from one XCD's L2.  Any order of the workgroups within a tile is valid here (the tile's
// records carry no order on this path); the map is a bijection on [0, nblocks).
__device__ __forceinline__ uint32_t bucket_column(uint32_t b, uint32_t nblocks) {
  const uint32_t q = nblocks / 8, r = nblocks % 8, x = b % 8;
  return x * q + min(x, r) + b / 8;
}
// The per-workgroup tile counts live in LDS for BUCKET_MAX_TILES tiles at a time: a target with more
// GPU tiles is counted range by range, each pass over the workgroup's keys taking the tiles of one
// range (the keys stay in registers).
template <int PT>
__device__ __forceinline__ void bucket_hist_body(const uint32_t* __restrict__ keys, uint32_t n, uint32_t T,
                                                 uint32_t nblocks, uint32_t* __restrict__ hist, uint32_t bx) {
  __shared__ uint32_t cnt[BUCKET_MAX_TILES];
  const uint32_t b0 = bx * (256 * PT);
  uint32_t k[PT];
#pragma unroll
  for (int j = 0; j < PT; ++j) {
    const uint32_t i = b0 + j * 256 + threadIdx.x;
    k[j] = i < n ? keys[i] : 0xFFFFFFFFu;
  }
  const uint32_t col = bucket_column(bx, nblocks);
  for (uint32_t r0 = 0; r0 < T; r0 += BUCKET_MAX_TILES) {
    const uint32_t tn = min(T - r0, BUCKET_MAX_TILES);
    if (r0) __syncthreads();  // the previous range's counts are written out
    for (uint32_t d = threadIdx.x; d < tn; d += 256) cnt[d] = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PT; ++j)
      if (k[j] - r0 < tn) atomicAdd(&cnt[k[j] - r0], 1u);  // also skips the 0xFFFFFFFF padding
    __syncthreads();
    for (uint32_t d = threadIdx.x; d < tn; d += 256) hist[(r0 + d) * nblocks + col] = cnt[d];
  }
}

// Only the tiles present in the workgroup's records fetch their (strided) offsets.  Positions at
// or beyond `limit` (the output's size) are dropped.
template <int PT>
__device__ __forceinline__ void bucket_scatter_body(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ vals,
                                                    uint32_t n, uint32_t T, uint32_t nblocks,
                                                    const uint32_t* __restrict__ hist_scanned, uint32_t* __restrict__ vout,
                                                    uint32_t limit, uint32_t bx) {
  __shared__ uint32_t off[BUCKET_MAX_TILES];
  const uint32_t b0 = bx * (256 * PT);
  uint32_t k[PT], v[PT];
#pragma unroll
  for (int j = 0; j < PT; ++j) {
    const uint32_t i = b0 + j * 256 + threadIdx.x;
    k[j] = i < n ? keys[i] : 0xFFFFFFFFu;
    v[j] = i < n ? vals[i] : 0u;
  }
  for (uint32_t r0 = 0; r0 < T; r0 += BUCKET_MAX_TILES) {
    const uint32_t tn = min(T - r0, BUCKET_MAX_TILES);
    if (r0) __syncthreads();  // the previous range's offsets are consumed
    for (uint32_t d = threadIdx.x; d < tn; d += 256) off[d] = 0xFFFFFFFFu;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PT; ++j)
      if (k[j] - r0 < tn) off[k[j] - r0] = 0u;  // mark the tiles present
    __syncthreads();
    for (uint32_t d = threadIdx.x; d < tn; d += 256)
      if (off[d] == 0u) off[d] = hist_scanned[(r0 + d) * nblocks + bucket_column(bx, nblocks)];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PT; ++j)
      if (k[j] - r0 < tn) {
        const uint32_t pos = atomicAdd(&off[k[j] - r0], 1u);
        if (pos < limit) vout[pos] = v[j];
      }
  }
}

// atomicAdd(&counters[key], 1) for every active lane, one atomic per distinct key of the wave;
// returns the lane's old value plus its rank among the lanes with the same key.
__device__ __forceinline__ uint32_t wave_counted_add(uint32_t* counters, uint32_t key) {
  const int lane = __lane_id();
  uint32_t result = 0;
  while (true) {
    const uint32_t k0 = __builtin_amdgcn_readfirstlane(key);
    const unsigned long long m = __ballot(key == k0);
    if (key == k0) {
      const uint32_t rank = static_cast<uint32_t>(__popcll(m & ((1ull << lane) - 1ull)));
      uint32_t old = 0;
      if (rank == 0) old = atomicAdd(&counters[k0], static_cast<uint32_t>(__popcll(m)));
      result = static_cast<uint32_t>(__shfl(static_cast<int>(old), __builtin_ctzll(m), 64)) + rank;
      break;
    }
  }
  return result;
}
// Record-count class of a GPU tile for the scheduling order: class 11 - floor(log2 n) (heaviest
// first, 2048 records and more in class 0), class 15 for an empty tile.
__device__ __forceinline__ uint32_t tile_class(uint32_t n) {
  if (n == 0) return 15u;
  const int lg = 31 - __clz(n);
  return static_cast<uint32_t>(min(max(11 - lg, 0), 14));
}

// tile t's records are [scanned[t * nblocks], scanned[(t + 1) * nblocks]) (`end` for the last tile)
__device__ __forceinline__ void bucket_range_body(const uint32_t* __restrict__ hist_scanned, uint32_t end, uint32_t T,
                                                  uint32_t nblocks, uint32_t* __restrict__ ts, uint32_t* __restrict__ te,
                                                  uint32_t t) {
  if (t >= T) return;
  ts[t] = hist_scanned[t * nblocks];
  te[t] = (t + 1 < T) ? hist_scanned[(t + 1) * nblocks] : end;
}

uint32_t bucket_hist_size(uint32_t T, uint32_t n) {
  return T * std::max<uint32_t>((n + BUCKET_ITEMS - 1) / BUCKET_ITEMS, 1);
}

// Counting sort of one draw's records by GPU tile (order-independent draws): the order within a tile
// is immaterial, so each workgroup of BUCKET_ITEMS records counts its tiles in LDS, noting the
// tiles it touches, and adds the counts of those tiles to the per-tile totals; one workgroup turns
// the totals into tile ranges; the scatter counts again, reserves its range in each touched tile
// with one atomic and places its records at the LDS ranks.  tile_count and tile_cursor are zero
// at the start of the draw.
// Counts the workgroup's records of tiles [r0, r0 + tn) in LDS (rank[j]: the record's rank among the
// workgroup's records of its tile) and lists the tiles it touches (relative to r0).
__device__ __forceinline__ void tile_count_lds(const uint32_t (&k)[BUCKET_PER_THREAD], uint32_t (&rank)[BUCKET_PER_THREAD],
                                               uint32_t r0, uint32_t tn, uint32_t* cnt, uint16_t* touched,
                                               uint32_t* ntouched) {
  for (uint32_t d = threadIdx.x; d < tn; d += 256) cnt[d] = 0;
  if (threadIdx.x == 0) *ntouched = 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < BUCKET_PER_THREAD; ++j)
    if (k[j] - r0 < tn) {  // also skips the 0xFFFFFFFF padding
      rank[j] = atomicAdd(&cnt[k[j] - r0], 1u);
      if (rank[j] == 0) touched[atomicAdd(ntouched, 1u)] = static_cast<uint16_t>(k[j] - r0);
    }
  __syncthreads();
}
__device__ __forceinline__ void tile_load_keys(const uint32_t* __restrict__ keys, uint32_t n, uint32_t b0,
                                               uint32_t (&k)[BUCKET_PER_THREAD]) {
#pragma unroll
  for (int j = 0; j < BUCKET_PER_THREAD; ++j) {
    const uint32_t i = b0 + j * 256 + threadIdx.x;
    k[j] = i < n ? keys[i] : 0xFFFFFFFFu;
  }
}
__global__ void __launch_bounds__(256) tile_count_kernel(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ count,
                                                         uint32_t cap, uint32_t T, uint32_t* __restrict__ tile_count) {
  __shared__ uint32_t cnt[BUCKET_MAX_TILES];
  __shared__ uint16_t touched[BUCKET_ITEMS];
  __shared__ uint32_t ntouched;
  const uint32_t n = min(*count, cap);
  const uint32_t b0 = blockIdx.x * BUCKET_ITEMS;
  if (b0 >= n) return;
  uint32_t k[BUCKET_PER_THREAD], rank[BUCKET_PER_THREAD];
  tile_load_keys(keys, n, b0, k);
  for (uint32_t r0 = 0; r0 < T; r0 += BUCKET_MAX_TILES) {
    const uint32_t tn = min(T - r0, BUCKET_MAX_TILES);
    if (r0) __syncthreads();  // the previous range's touched tiles are consumed
    tile_count_lds(k, rank, r0, tn, cnt, touched, &ntouched);
    for (uint32_t i = threadIdx.x; i < ntouched; i += 256) {
      const uint32_t t = touched[i];
      atomicAdd(&tile_count[r0 + t], cnt[t]);
    }
  }
}
// counters[key] += the number of valid lanes with this lane's key (< 16), one LDS atomic per distinct
// key; returns the counter's old value plus the lane's rank among them.  Lanes with equal keys are
// matched by four ballots, one per key bit.  All lanes of the wave call it.
__device__ __forceinline__ uint32_t wave_counted_add16(uint32_t* counters, uint32_t key, bool valid) {
  const int lane = __lane_id();
  uint64_t m = __ballot(valid);
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const bool bit = ((key >> b) & 1u) != 0;
    const uint64_t bal = __ballot(bit);
    m &= bit ? bal : ~bal;
  }
  const uint64_t lt = (1ull << lane) - 1ull;
  uint32_t old = 0;
  if (valid && (m & lt) == 0) old = atomicAdd(&counters[key], static_cast<uint32_t>(__popcll(m)));
  const int leader = valid ? __builtin_ctzll(m) : lane;
  old = static_cast<uint32_t>(__shfl(static_cast<int>(old), leader, 64));
  return old + static_cast<uint32_t>(__popcll(m & lt));
}

// One workgroup: tile ranges from the totals (exclusive prefix, BUCKET_MAX_TILES tiles per step), the
// tiles per record-count class, and, when `order` is given, the tiles' scheduling order: tiles of
// class c after every tile of the classes before c, within a class in the atomics' order (tiles are
// independent, so the order never changes a pixel).
__global__ void __launch_bounds__(1024) tile_prefix_kernel(const uint32_t* __restrict__ tile_count, uint32_t T,
                                                          uint32_t* __restrict__ ts, uint32_t* __restrict__ te,
                                                          uint32_t* __restrict__ counters, uint32_t* __restrict__ order) {
  constexpr int PER = BUCKET_MAX_TILES / 1024;
  __shared__ uint32_t wsum[16];
  __shared__ uint32_t classes[16];
  const uint32_t tid = threadIdx.x;
  if (tid < 16) classes[tid] = 0;
  uint32_t carry = 0;  // records of the tiles before this step
  for (uint32_t base = 0; base < T; base += BUCKET_MAX_TILES) {
    const uint32_t t0 = base + tid * PER;
    uint32_t c[PER], sum = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      c[i] = load_or_zero(tile_count, t0 + i, T);
      sum += c[i];
    }
    const uint32_t incl = wave_incl_scan(sum);
    if (base) __syncthreads();  // the previous step's wave sums are read
    if ((tid & 63) == 63) wsum[tid >> 6] = incl;
    __syncthreads();
    uint32_t run = carry + incl - sum, step = 0;
    for (uint32_t w = 0; w < 16; ++w) {
      if (w < (tid >> 6)) run += wsum[w];
      step += wsum[w];
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (t0 + i < T) {
        ts[t0 + i] = run;
        te[t0 + i] = run + c[i];
      }
      run += c[i];
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) (void)wave_counted_add16(classes, tile_class(c[i]), t0 + i < T);
    carry += step;
  }
  __syncthreads();
  if (tid < 16) counters[CT_CLASS + tid] = classes[tid];
  if (!order) return;
  // classes[] becomes each class's next position
  if (tid == 0) {
    uint32_t b = 0;
    for (int k = 0; k < 16; ++k) {
      const uint32_t n = classes[k];
      classes[k] = b;
      b += n;
    }
  }
  __syncthreads();
  for (uint32_t base = 0; base < T; base += BUCKET_MAX_TILES) {
    const uint32_t t0 = base + tid * PER;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const bool valid = t0 + i < T;
      const uint32_t pos = wave_counted_add16(classes, tile_class(load_or_zero(tile_count, t0 + i, T)), valid);
      if (valid) order[pos] = t0 + i;
    }
  }
}
// The same for targets of at most PREFIX_MAX_TILES tiles, one workgroup per PREFIX_TILES tiles and
// no communication between them: every workgroup reads all T tile totals (8 per thread at 1080p),
// from which it takes the records of the tiles before its own, the tiles of each record-count class
// in the whole target and before its own tiles, and writes its tiles' ranges and scheduling
// positions.  The order is class by class (heaviest first), by tile within a class.
constexpr uint32_t PREFIX_TILES = 1024;
constexpr uint32_t PREFIX_MAX_TILES = 65536;
__global__ void __launch_bounds__(1024) tile_prefix_par_kernel(const uint32_t* __restrict__ tile_count, uint32_t T,
                                                              uint32_t* __restrict__ ts, uint32_t* __restrict__ te,
                                                              uint32_t* __restrict__ counters, uint32_t* __restrict__ order) {
  __shared__ uint32_t w_all[16][16], w_before[16][16], w_mine[16][16];  // [wave][class]
  __shared__ uint32_t w_rec[16], w_scan[16], c_base[16], s_start[16], s_pos[16][16];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, bx = blockIdx.x;
  const uint32_t nj = (T + PREFIX_TILES - 1) / PREFIX_TILES;  // at most 64
  // this lane's tiles per class, one 8-bit field per class (classes 0-7 in [0], 8-15 in [1]): all of
  // them, and those before the workgroup's
  unsigned long long all[2] = {0, 0}, before[2] = {0, 0};
  uint32_t rec_before = 0, mine = 0;
  for (uint32_t j0 = 0; j0 < nj; j0 += 8) {
    uint32_t v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const uint32_t i = (j0 + q) * PREFIX_TILES + tid;
      v[q] = load_or_zero(tile_count, i, T);
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const uint32_t j = j0 + q;  // uniform
      if (j >= nj) break;
      const bool valid = j * PREFIX_TILES + tid < T;
      const uint32_t c = tile_class(v[q]);
      if (j < bx) rec_before += v[q];
      if (j == bx) mine = v[q];
      const unsigned long long one = valid ? 1ull << (8 * (c & 7)) : 0ull;
      all[c >> 3] += one;
      if (j < bx) before[c >> 3] += one;
    }
  }
  const uint32_t t = bx * PREFIX_TILES + tid;
  const bool mine_valid = t < T;
  const uint32_t cm = tile_class(mine);
  // rank among the wave's own tiles of the same class (four ballots, one per class bit)
  uint64_t m = __ballot(mine_valid);
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const bool bit = ((cm >> b) & 1u) != 0;
    const uint64_t bal = __ballot(bit);
    m &= bit ? bal : ~bal;
  }
  const uint32_t rank = static_cast<uint32_t>(__popcll(m & ((1ull << lane) - 1ull)));
  unsigned long long mine_f[2] = {0, 0};
  mine_f[cm >> 3] = mine_valid ? 1ull << (8 * (cm & 7)) : 0ull;
  // the wave's per-class sums: the 8-bit fields widened to 16 bits (4 classes per word, at most
  // 64 lanes x 64 chunks per class), added over the wave
  unsigned long long wa[4], wb[4], wm[4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const unsigned long long lo = 0x00FF00FF00FF00FFull;
    wa[2 * h] = all[h] & lo;
    wa[2 * h + 1] = (all[h] >> 8) & lo;
    wb[2 * h] = before[h] & lo;
    wb[2 * h + 1] = (before[h] >> 8) & lo;
    wm[2 * h] = mine_f[h] & lo;
    wm[2 * h + 1] = (mine_f[h] >> 8) & lo;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      wa[w] += __shfl_xor(wa[w], off, 64);
      wb[w] += __shfl_xor(wb[w], off, 64);
      wm[w] += __shfl_xor(wm[w], off, 64);
    }
  // class k = 8h + 2f + e lives in word 2h + e, 16-bit field f (fields of a word: classes of one parity)
  auto field = [](const unsigned long long (&w)[4], uint32_t k) -> uint32_t {
    const bool h = (k >> 3) != 0, e = (k & 1) != 0;
    const unsigned long long x = h ? (e ? w[3] : w[2]) : (e ? w[1] : w[0]);  // selects, no indexing
    return static_cast<uint32_t>((x >> (16 * ((k & 7) >> 1))) & 0xFFFFull);
  };
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) rec_before += static_cast<uint32_t>(__shfl_xor(static_cast<int>(rec_before), off, 64));
  const uint32_t incl = wave_incl_scan(mine);
  if (lane < 16) {
    w_all[wave][lane] = field(wa, lane);
    w_before[wave][lane] = field(wb, lane);
    w_mine[wave][lane] = field(wm, lane);
  }
  if (lane == 0) w_rec[wave] = rec_before;
  if (lane == 63) w_scan[wave] = incl;
  __syncthreads();
  // Per-wave and per-class bases, each a fixed-length sum over the 16 waves (unrolled, the loads
  // issued together):
  //   c_base[k]     tiles of classes < k in the target + tiles of class k before the workgroup's
  //   s_start[w]    records of the tiles before the workgroup's + of waves < w's tiles
  //   s_pos[w][k]   c_base[k] + this workgroup's class-k tiles in waves < w
  if (tid < 64) {
    const uint32_t k = tid & 15;
    uint32_t tot = 0, bef = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      tot += w_all[w][k];
      bef += w_before[w][k];
    }
    uint32_t below = tot;  // inclusive scan over the 16 classes, then exclusive
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
      const uint32_t y = static_cast<uint32_t>(__shfl_up(static_cast<int>(below), off, 16));
      if (k >= static_cast<uint32_t>(off)) below += y;
    }
    below -= tot;
    if (tid < 16) {
      c_base[k] = below + bef;
      if (bx == 0) counters[CT_CLASS + k] = tot;
    }
  } else if (tid < 80) {
    const uint32_t w = tid - 64;
    uint32_t rec = 0, pre = 0;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      rec += w_rec[v];
      pre += static_cast<uint32_t>(v) < w ? w_scan[v] : 0u;
    }
    s_start[w] = rec + pre;
  }
  __syncthreads();
  if (tid < 256) {
    const uint32_t w = tid >> 4, k = tid & 15;
    uint32_t pre = 0;
#pragma unroll
    for (int v = 0; v < 16; ++v) pre += static_cast<uint32_t>(v) < w ? w_mine[v][k] : 0u;
    s_pos[w][k] = c_base[k] + pre;
  }
  __syncthreads();
  if (mine_valid) {
    const uint32_t start = s_start[wave] + incl - mine;
    ts[t] = start;
    te[t] = start + mine;
    order[s_pos[wave][cm] + rank] = t;
  }
}
__global__ void __launch_bounds__(256) tile_scatter_kernel(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ vals,
                                                           const uint32_t* __restrict__ count, uint32_t cap, uint32_t T,
                                                           const uint32_t* __restrict__ ts, uint32_t* __restrict__ tile_cursor,
                                                           uint32_t* __restrict__ vout) {
  __shared__ uint32_t cnt[BUCKET_MAX_TILES];
  __shared__ uint16_t touched[BUCKET_ITEMS];
  __shared__ uint32_t ntouched;
  const uint32_t n = min(*count, cap);
  const uint32_t b0 = blockIdx.x * BUCKET_ITEMS;
  if (b0 >= n) return;
  uint32_t k[BUCKET_PER_THREAD], rank[BUCKET_PER_THREAD];
  tile_load_keys(keys, n, b0, k);
  for (uint32_t r0 = 0; r0 < T; r0 += BUCKET_MAX_TILES) {
    const uint32_t tn = min(T - r0, BUCKET_MAX_TILES);
    if (r0) __syncthreads();  // the previous range's positions are consumed
    tile_count_lds(k, rank, r0, tn, cnt, touched, &ntouched);
    // this workgroup's range in each touched tile; cnt[t] becomes its first position
    for (uint32_t i = threadIdx.x; i < ntouched; i += 256) {
      const uint32_t t = touched[i];
      cnt[t] = ts[r0 + t] + atomicAdd(&tile_cursor[r0 + t], cnt[t]);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < BUCKET_PER_THREAD; ++j)
      if (k[j] - r0 < tn) vout[cnt[k[j] - r0] + rank[j]] = vals[b0 + j * 256 + threadIdx.x];
  }
}

bool bucket_sort_applicable(const draw_params& P) { return P.gtiles_x > 0 && P.gtiles_y > 0; }
bool launch_bucket_sort(const draw_params& P, const draw_buffers& B, uint32_t cap, uint32_t* order, hipStream_t s) {
  const uint32_t T = static_cast<uint32_t>(P.gtiles_x * P.gtiles_y);
  if (!bucket_sort_applicable(P)) return false;
  const uint32_t* count = B.counters + CT_TOTAL;
  const uint32_t nblocks = std::max<uint32_t>((cap + BUCKET_ITEMS - 1) / BUCKET_ITEMS, 1);
  hipLaunchKernelGGL(tile_count_kernel, dim3(nblocks), dim3(256), 0, s, B.keys[0], count, cap, T, B.tile_count);
  if (order && T <= PREFIX_MAX_TILES)
    hipLaunchKernelGGL(tile_prefix_par_kernel, dim3((T + PREFIX_TILES - 1) / PREFIX_TILES), dim3(1024), 0, s, B.tile_count, T,
                       B.tstart, B.tend, B.counters, order);
  else
    hipLaunchKernelGGL(tile_prefix_kernel, dim3(1), dim3(1024), 0, s, B.tile_count, T, B.tstart, B.tend, B.counters, order);
  hipLaunchKernelGGL(tile_scatter_kernel, dim3(nblocks), dim3(256), 0, s, B.keys[0], B.vals[0], count, cap, T, B.tstart,
                     B.tile_count + T, B.vals[1]);
  return true;
}

__global__ void tile_range_kernel(const uint32_t* __restrict__ keys, uint32_t n, uint32_t T, uint32_t* __restrict__ ts,
                                  uint32_t* __restrict__ te) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  // T == 0: the ranges were cleared beforehand, only the non-empty tiles are written
  uint32_t k = keys[i];
  if (i == 0 && T) {
    for (uint32_t t = 0; t < k; ++t) ts[t] = te[t] = 0;
  }
  if (i == 0 || keys[i - 1] != k) ts[k] = i;
  if (i == n - 1 || keys[i + 1] != k) {
    te[k] = i + 1;
    const uint32_t next = !T ? k + 1 : ((i == n - 1) ? T : keys[i + 1]);
    for (uint32_t t = k + 1; t < next; ++t) ts[t] = te[t] = i + 1;
  }
}

// Scheduling order of the GPU tiles, heaviest first so that the longest tiles start early.  Tiles
// are independent, so the order never changes a pixel.  One workgroup buckets the tiles by record
// count / 8 (heaviest bucket first) with LDS counters.
__device__ __forceinline__ uint32_t tile_bucket(const uint32_t* ts, const uint32_t* te, uint32_t t) {
  return 255u - min((te[t] - ts[t]) >> 3, 255u);
}
__device__ __forceinline__ void tile_order_body(const uint32_t* __restrict__ ts, const uint32_t* __restrict__ te,
                                                uint32_t T, uint32_t* __restrict__ order) {
  __shared__ uint32_t cnt[256];
  __shared__ uint32_t wtot[4];
  const uint32_t tid = threadIdx.x;
  if (tid < 256) cnt[tid] = 0;
  __syncthreads();
  for (uint32_t t = tid; t < T; t += blockDim.x) (void)wave_counted_add(cnt, tile_bucket(ts, te, t));
  __syncthreads();
  // exclusive scan of the 256 bucket counts by the first four waves
  uint32_t c = 0, incl = 0;
  if (tid < 256) {
    c = cnt[tid];
    incl = wave_incl_scan(c);
    if ((tid & 63) == 63) wtot[tid >> 6] = incl;
  }
  __syncthreads();
  if (tid < 256) {
    uint32_t before = 0;
    for (uint32_t w = 0; w < (tid >> 6); ++w) before += wtot[w];
    cnt[tid] = before + incl - c;
  }
  __syncthreads();
  for (uint32_t t = tid; t < T; t += blockDim.x) order[wave_counted_add(cnt, tile_bucket(ts, te, t))] = t;
}
__global__ void __launch_bounds__(1024) tile_order_kernel(const uint32_t* __restrict__ ts, const uint32_t* __restrict__ te,
                                                          uint32_t T, uint32_t* __restrict__ order) {
  tile_order_body(ts, te, T, order);
}

__global__ void tile_class_count_kernel(const uint32_t* __restrict__ ts, const uint32_t* __restrict__ te, uint32_t T,
                                        uint32_t* __restrict__ counters) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < T) (void)wave_counted_add(counters + CT_CLASS, tile_class(te[t] - ts[t]));
}
// Tiles of class c take the positions after every tile of the classes before c; within a class the
// order is the atomics' (tiles are independent, so the order never changes a pixel).
__global__ void tile_class_order_kernel(const uint32_t* __restrict__ ts, const uint32_t* __restrict__ te, uint32_t T,
                                        uint32_t* __restrict__ counters, uint32_t* __restrict__ order) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= T) return;
  const uint32_t c = tile_class(te[t] - ts[t]);
  uint32_t base = 0;
  for (uint32_t k = 0; k < c; ++k) base += counters[CT_CLASS + k];
  order[base + wave_counted_add(counters + CT_CURSOR, c)] = t;
}
void launch_tile_order(const draw_params& P, const draw_buffers& B, uint32_t* order, bool counted, hipStream_t s) {
  const uint32_t T = static_cast<uint32_t>(P.gtiles_x * P.gtiles_y);
  if (!T) return;
  if (!counted) hipLaunchKernelGGL(tile_class_count_kernel, dim3((T + 255) / 256), dim3(256), 0, s, B.tstart, B.tend, T, B.counters);
  hipLaunchKernelGGL(tile_class_order_kernel, dim3((T + 255) / 256), dim3(256), 0, s, B.tstart, B.tend, T, B.counters, order);
}

void launch_fill_u32(uint32_t* p, uint32_t n, uint32_t v, hipStream_t s) {
  if (n) hipLaunchKernelGGL(fill_u32_kernel, dim3((n + 255) / 256), dim3(256), 0, s, p, n, v);
}

void launch_tile_ranges(const draw_params& P, const draw_buffers& B, int which, uint32_t n, hipStream_t s) {
  uint32_t T = static_cast<uint32_t>(P.gtiles_x * P.gtiles_y);
  if (!T) return;
  if (n < 4 * T) {  // sparse records: clear every range first, so no thread walks a long empty run
    hipLaunchKernelGGL(fill_u32_kernel, dim3((T + 255) / 256), dim3(256), 0, s, B.tstart, T, 0u);
    hipLaunchKernelGGL(fill_u32_kernel, dim3((T + 255) / 256), dim3(256), 0, s, B.tend, T, 0u);
    if (n) hipLaunchKernelGGL(tile_range_kernel, dim3((n + 255) / 256), dim3(256), 0, s, B.keys[which], n, 0u, B.tstart, B.tend);
    return;
  }
  hipLaunchKernelGGL(tile_range_kernel, dim3((n + 255) / 256), dim3(256), 0, s, B.keys[which], n, T, B.tstart, B.tend);
}

// ============================================================== host launchers
void launch_reduce_partials(const unsigned long long* partial, uint32_t n, unsigned long long* stats, int slot, hipStream_t s) {
  hipLaunchKernelGGL(reduce_partials_kernel, dim3(1), dim3(256), 0, s, partial, n, stats, slot);
}

void launch_vs(const draw_params& P, float4* vbuf, uint32_t* counters, uint32_t* tiles, size_t ntiles, hipStream_t s) {
  uint32_t n = P.nverts + 1;
  hipLaunchKernelGGL(vs_kernel, dim3((n + 255) / 256), dim3(256), 0, s, P, vbuf, counters, tiles,
                     static_cast<uint32_t>(ntiles));
}

void launch_setup(const draw_params& P, const draw_buffers& B, hipStream_t s) {
  if (P.prim_count == 0) return;
  dim3 grid((P.prim_count + 255) / 256);
#define SRX_SETUP(NA) \
  hipLaunchKernelGGL(setup_kernel<NA>, grid, dim3(256), 0, s, P, B.vbuf, B.tri_rec, B.tri_attr, B.cnt, B.clip_flag, B.counters, \
                     B.wide_list, B.partial, B.bsum, B.pairs)
  SRX_NA_DISPATCH(P.nattr, SRX_SETUP)
#undef SRX_SETUP
  if (P.count_stats)
    launch_reduce_partials(B.partial, grid.x, B.stats, ST_CPRIMITIVES, s);
}

void launch_clip(const draw_params& P, const draw_buffers& B, hipStream_t s) {
  if (P.prim_count == 0) return;
  dim3 grid(std::min<uint32_t>((P.prim_count + 255) / 256, 256));  // up to 1024 waves in 256-lane workgroups
#define SRX_CLIP(NA)                                                                                                     \
  hipLaunchKernelGGL(clip_kernel<NA>, grid, dim3(256), 0, s, P, B.vbuf, B.tri_rec, B.tri_attr, B.cnt, B.clip_flag, B.clip_slot, \
                     B.clip_verts, B.clip_hdr, B.clip_capacity, B.counters, B.stats, B.wide_list, B.bsum)
  SRX_NA_DISPATCH(P.nattr, SRX_CLIP)
#undef SRX_CLIP
}

void launch_emit(const draw_params& P, const draw_buffers& B, uint32_t capacity, hipStream_t s) {
  const uint32_t n = P.prim_count;
  if (!n) return;
  hipLaunchKernelGGL(emit_kernel, dim3((n + 255) / 256), dim3(256), 0, s, P, B.tri_rec, B.cnt, B.bsum, B.pairs,
                     capacity, B.keys[0], B.vals[0]);
}

// ============================================================== clears, resolve, mip generation
// surface::fill with the converted colour: the texel bytes are built once and stored 16 bytes at a
// time (texel sizes 4, 8 and 16 tile a 16-byte word; RGB32F takes the per-texel path).
__global__ void clear_kernel(surface_desc s, float4 v) {
  const size_t n = static_cast<size_t>(s.w) * s.h * s.samples;
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int es = pf_size(s.pf);
  if (es == 12) {
    if (i < n) store_texel(s.pf, s.data + i * 12, v);
    return;
  }
  const uint4 w = fill_words(s.pf, v);
  const size_t words = n * es / 16, tail = n * es % 16;
  if (i < words) reinterpret_cast<uint4*>(s.data)[i] = w;
  if (i == 0 && tail) {  // whole texels (es divides 16): the tail starts a fresh 16-byte word
    const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
    for (size_t b = 0; b < tail; b += 4) *reinterpret_cast<uint32_t*>(s.data + words * 16 + b) = ws[b / 4];
  }
}

// depth and/or stencil of every RG32F sample; both at once are 16-byte stores of two samples
__global__ void clear_ds_kernel(surface_desc s, uint32_t flags, float depth, uint32_t stencil) {
  const size_t n = static_cast<size_t>(s.w) * s.h * s.samples;
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (flags == 3) {
    const uint32_t d = __float_as_uint(depth);
    if (i < n / 2) reinterpret_cast<uint4*>(s.data)[i] = make_uint4(d, stencil, d, stencil);
    if (i == 0 && (n & 1)) {
      float* p = reinterpret_cast<float*>(s.data + (n - 1) * 8);
      p[0] = depth;
      p[1] = __uint_as_float(stencil);
    }
    return;
  }
  if (i >= n) return;
  float* p = reinterpret_cast<float*>(s.data + i * 8);
  if (flags & 1) p[0] = depth;
  if (flags & 2) p[1] = __uint_as_float(stencil);
}

// surface::resolve (surface.cpp:123-140): sum samples in order, then multiply by 1/S
__global__ void resolve_kernel(surface_desc src, surface_desc dst) {
  int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
  if (x >= src.w) return;
  float4 c = make_float4(0, 0, 0, 0);
  for (int s = 0; s < src.samples; ++s) {
    float4 t = load_texel(src.pf, sample_addr(src, x, y, s));
    c = make_float4(c.x + t.x, c.y + t.y, c.z + t.z, c.w + t.w);
  }
  float inv = 1 / static_cast<float>(src.samples);
  store_texel(dst.pf, sample_addr(dst, x, y, 0), make_float4(c.x * inv, c.y * inv, c.z * inv, c.w * inv));
}

// The same for 4-sample RGBA8 into RGBA8: one 16-byte load per pixel.
__global__ void resolve_rgba8x4_kernel(surface_desc src, surface_desc dst) {
  const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= static_cast<size_t>(src.w) * src.h) return;
  const uint4 q = reinterpret_cast<const uint4*>(src.data)[i];
  const uint32_t w[4] = {q.x, q.y, q.z, q.w};
  float4 c = make_float4(0, 0, 0, 0);
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const uint32_t u = w[s];
    const float4 t = make_float4(static_cast<float>(u & 0xFF) * (1.0f / 255), static_cast<float>((u >> 8) & 0xFF) * (1.0f / 255),
                                 static_cast<float>((u >> 16) & 0xFF) * (1.0f / 255), static_cast<float>(u >> 24) * (1.0f / 255));
    c = make_float4(c.x + t.x, c.y + t.y, c.z + t.z, c.w + t.w);
  }
  const float inv = 1 / 4.0f;
  store_texel(PF_RGBA8, dst.data + i * 4, make_float4(c.x * inv, c.y * inv, c.z * inv, c.w * inv));
}

// surface::make_mip_surface (surface.cpp:53-92); odd-size edge reads clamp to the last texel
__global__ void mip_kernel(surface_desc src, surface_desc dst, int filter) {
  int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
  if (x >= dst.w) return;
  for (int s = 0; s < dst.samples; ++s) {
    int x0 = x * 2, y0 = y * 2, x1 = min(x0 + 1, src.w - 1), y1 = min(y0 + 1, src.h - 1);
    float4 c;
    if (filter == FILTER_POINT) {
      c = load_texel(src.pf, sample_addr(src, x0, y0, s));
    } else {
      float4 c0 = load_texel(src.pf, sample_addr(src, x0, y0, s)), c1 = load_texel(src.pf, sample_addr(src, x1, y0, s));
      float4 c2 = load_texel(src.pf, sample_addr(src, x0, y1, s)), c3 = load_texel(src.pf, sample_addr(src, x1, y1, s));
      c = make_float4(((c0.x + c1.x) + c2.x) + c3.x, ((c0.y + c1.y) + c2.y) + c3.y, ((c0.z + c1.z) + c2.z) + c3.z,
                      ((c0.w + c1.w) + c2.w) + c3.w);
      c = make_float4(c.x * 0.25f, c.y * 0.25f, c.z * 0.25f, c.w * 0.25f);
    }
    store_texel(dst.pf, sample_addr(dst, x, y, s), c);
  }
}

// ============================================================== batched jobs
// Every stage of a batch of independent draws is one launch: each workgroup looks up its job and
// its index within the job's grid (stage_map) and runs the single-draw kernel body on the job's
// parameters and buffers.  Record counts are read on the device (from the batch-wide scan of the
// per-triangle counts), clamped to the capacities the batch was prepared with, so a replay whose
// geometry changed stays in bounds and reports the overflow through the status word.

__global__ void batch_reset_kernel(uint32_t* __restrict__ counters, uint32_t n, uint32_t* __restrict__ cnt_tail,
                                   uint32_t* __restrict__ hist_tail, uint32_t* __restrict__ status) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) counters[i] = 0;
  if (i == 0) {
    *cnt_tail = 0;
    *hist_tail = 0;
    *status = 0;
  }
}

__global__ void __launch_bounds__(256) fill_batch_kernel(const fill_item* __restrict__ items, stage_map m) {
  uint32_t lb, nb;
  const fill_item& it = items[stage_job(m, lb, nb)];
  const size_t i = static_cast<size_t>(lb) * 256 + threadIdx.x;
  const uint4 w = fill_words(it.pf, it.value);
  if (i < it.words) reinterpret_cast<uint4*>(it.data)[i] = w;
  if (i == 0 && it.tail) {
    const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
    for (uint32_t b = 0; b < it.tail; b += 4) *reinterpret_cast<uint32_t*>(it.data + it.words * 16 + b) = ws[b / 4];
  }
}

__global__ void __launch_bounds__(256) resolve_batch_kernel(const resolve_item* __restrict__ items, stage_map m) {
  uint32_t lb, nb;
  const resolve_item& it = items[stage_job(m, lb, nb)];
  const surface_desc src = it.src, dst = it.dst;
  const size_t i = static_cast<size_t>(lb) * 256 + threadIdx.x;
  if (i >= static_cast<size_t>(src.w) * src.h) return;
  const int x = static_cast<int>(i % src.w), y = static_cast<int>(i / src.w);
  float4 c = make_float4(0, 0, 0, 0);
  for (int smp = 0; smp < src.samples; ++smp) {
    const float4 t = load_texel(src.pf, sample_addr(src, x, y, smp));
    c = make_float4(c.x + t.x, c.y + t.y, c.z + t.z, c.w + t.w);
  }
  const float inv = 1 / static_cast<float>(src.samples);
  store_texel(dst.pf, sample_addr(dst, x, y, 0), make_float4(c.x * inv, c.y * inv, c.z * inv, c.w * inv));
}

__global__ void __launch_bounds__(256) vs_batch_kernel(const batch_job* __restrict__ jobs, stage_map m) {
  uint32_t lb, nb;
  const batch_job& J = jobs[stage_job(m, lb, nb)];
  vs_body(J.P, J.B.vbuf, lb);
}

template <int NA>
__global__ void __launch_bounds__(256) setup_batch_kernel(const batch_job* __restrict__ jobs, stage_map m) {
  uint32_t lb, nb;
  const batch_job& J = jobs[stage_job(m, lb, nb)];
  setup_body<NA>(J.P, J.B.vbuf, J.B.tri_rec, J.B.tri_attr, J.B.cnt, J.B.clip_flag, J.B.counters, J.B.wide_list, J.B.partial,
                 nullptr, nullptr, lb);
}

template <int NA>
__global__ void clip_batch_kernel(const batch_job* __restrict__ jobs, stage_map m) {
  uint32_t lb, nb;
  const batch_job& J = jobs[stage_job(m, lb, nb)];
  clip_body<NA>(J.P, J.B.vbuf, J.B.tri_rec, J.B.tri_attr, J.B.cnt, J.B.clip_flag, J.B.clip_slot, J.B.clip_verts,
                J.B.clip_hdr, J.B.clip_capacity, J.B.counters, J.B.stats, J.B.wide_list, nullptr, lb, nb);
}

// The job's counts are followed by the next job's first scanned count (or the batch total): the
// end of its last triangle's records.
__global__ void __launch_bounds__(256) emit_batch_kernel(const batch_job* __restrict__ jobs, stage_map m, uint32_t capacity) {
  uint32_t lb, nb;
  const batch_job& J = jobs[stage_job(m, lb, nb)];
  emit_body(J.P, J.B.tri_rec, J.B.cnt, J.B.cnt + 3 * J.P.prim_count, capacity, J.B.keys[0], J.B.vals[0], lb);
}

// The job's records [begin, begin + n): its scanned counts clamped to the record capacity and to the
// records its binning workgroups cover.
__device__ __forceinline__ void job_records(const batch_job& J, uint32_t capacity, uint32_t items, uint32_t& begin,
                                            uint32_t& n) {
  const uint32_t b = min(J.B.cnt[0], capacity), e = min(J.B.cnt[3 * J.P.prim_count], capacity);
  begin = b;
  n = min(e - b, J.bucket_blocks * items);
}

template <int PT>
__global__ void __launch_bounds__(256) bucket_hist_batch_kernel(const batch_job* __restrict__ jobs, stage_map m,
                                                                uint32_t capacity) {
  uint32_t lb, nb, begin, n;
  const batch_job& J = jobs[stage_job(m, lb, nb)];
  job_records(J, capacity, 256 * PT, begin, n);
  bucket_hist_body<PT>(J.B.keys[0] + begin, n, J.tiles, J.bucket_blocks, J.B.hist, lb);
}

template <int PT>
__global__ void __launch_bounds__(256) bucket_scatter_batch_kernel(const batch_job* __restrict__ jobs, stage_map m,
                                                                   uint32_t capacity) {
  uint32_t lb, nb, begin, n;
  const batch_job& J = jobs[stage_job(m, lb, nb)];
  job_records(J, capacity, 256 * PT, begin, n);
  bucket_scatter_body<PT>(J.B.keys[0] + begin, J.B.vals[0] + begin, n, J.tiles, J.bucket_blocks, J.B.hist, J.B.vals[1],
                          capacity, lb);
}

// The job's histogram is followed by the next job's first scanned entry (or the batch total).
__global__ void __launch_bounds__(256) bucket_range_batch_kernel(const batch_job* __restrict__ jobs, stage_map m) {
  uint32_t lb, nb;
  const batch_job& J = jobs[stage_job(m, lb, nb)];
  bucket_range_body(J.B.hist, J.B.hist[J.tiles * J.bucket_blocks], J.tiles, J.bucket_blocks, J.B.tstart, J.B.tend,
                    lb * 256 + threadIdx.x);
}

__global__ void __launch_bounds__(1024) tile_order_batch_kernel(const batch_job* __restrict__ jobs) {
  const batch_job& J = jobs[blockIdx.x];
  tile_order_body(J.B.tstart, J.B.tend, J.tiles, const_cast<uint32_t*>(J.B.order));
}

// status bit 0: a job's records exceeded the capacity it was prepared with; bit 1: clip overflow
__global__ void batch_check_kernel(const batch_job* __restrict__ jobs, uint32_t njobs, uint32_t capacity, uint32_t items,
                                   uint32_t* __restrict__ status) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= njobs) return;
  const batch_job& J = jobs[j];
  const uint32_t b = J.B.cnt[0], e = J.B.cnt[3 * J.P.prim_count];
  uint32_t st = 0;
  if (e > capacity || e - b > J.bucket_blocks * items) st |= 1u;
  if (J.B.counters[CT_CLIP_OVERFLOW]) st |= 2u;
  if (st) atomicOr(status, st);
}

// records[j] of every job (unclamped), for sizing a batch
__global__ void batch_counts_kernel(const batch_job* __restrict__ jobs, uint32_t njobs, uint32_t* __restrict__ out) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= njobs) return;
  const batch_job& J = jobs[j];
  out[j] = J.B.cnt[3 * J.P.prim_count] - J.B.cnt[0];
  out[njobs + j] = J.B.counters[CT_CLIP_OVERFLOW];
}
void launch_batch_counts(const batch_job* jobs, uint32_t njobs, uint32_t* out, hipStream_t s) {
  if (njobs) hipLaunchKernelGGL(batch_counts_kernel, dim3((njobs + 255) / 256), dim3(256), 0, s, jobs, njobs, out);
}

void launch_batch_reset(uint32_t* counters, uint32_t n, uint32_t* cnt_tail, uint32_t* hist_tail, uint32_t* status,
                        hipStream_t s) {
  hipLaunchKernelGGL(batch_reset_kernel, dim3((std::max<uint32_t>(n, 1) + 255) / 256), dim3(256), 0, s, counters, n,
                     cnt_tail, hist_tail, status);
}
void launch_fill_batch(const fill_item* items, stage_map m, uint32_t blocks, hipStream_t s) {
  if (blocks) hipLaunchKernelGGL(fill_batch_kernel, dim3(blocks), dim3(256), 0, s, items, m);
}
void launch_resolve_batch(const resolve_item* items, stage_map m, uint32_t blocks, hipStream_t s) {
  if (blocks) hipLaunchKernelGGL(resolve_batch_kernel, dim3(blocks), dim3(256), 0, s, items, m);
}
void launch_vs_batch(const batch_job* jobs, stage_map m, uint32_t blocks, hipStream_t s) {
  if (blocks) hipLaunchKernelGGL(vs_batch_kernel, dim3(blocks), dim3(256), 0, s, jobs, m);
}
void launch_setup_batch(int na, const batch_job* jobs, stage_map m, uint32_t blocks, hipStream_t s) {
  if (!blocks) return;
#define SRX_SETUP_B(NA) hipLaunchKernelGGL(setup_batch_kernel<NA>, dim3(blocks), dim3(256), 0, s, jobs, m)
  SRX_NA_DISPATCH_BATCH(na, SRX_SETUP_B)
#undef SRX_SETUP_B
}
void launch_clip_batch(int na, const batch_job* jobs, stage_map m, uint32_t blocks, hipStream_t s) {
  if (!blocks) return;
#define SRX_CLIP_B(NA) hipLaunchKernelGGL(clip_batch_kernel<NA>, dim3(blocks), dim3(64), 0, s, jobs, m)
  SRX_NA_DISPATCH_BATCH(na, SRX_CLIP_B)
#undef SRX_CLIP_B
}
void launch_emit_batch(const batch_job* jobs, stage_map m, uint32_t blocks, uint32_t capacity, hipStream_t s) {
  if (blocks) hipLaunchKernelGGL(emit_batch_kernel, dim3(blocks), dim3(256), 0, s, jobs, m, capacity);
}
bool batch_bin_items_valid(int pt) { return pt == 8 || pt == 16 || pt == 32 || pt == 64; }
void launch_bucket_batch(int pt, int phase, const batch_job* jobs, stage_map m, uint32_t blocks, uint32_t capacity,
                         hipStream_t s) {
  if (!blocks) return;
#define SRX_BUCKET_B(PT)                                                                                          \
  if (phase == 0)                                                                                                  \
    hipLaunchKernelGGL(bucket_hist_batch_kernel<PT>, dim3(blocks), dim3(256), 0, s, jobs, m, capacity);          \
  else                                                                                                             \
    hipLaunchKernelGGL(bucket_scatter_batch_kernel<PT>, dim3(blocks), dim3(256), 0, s, jobs, m, capacity)
  switch (pt) {
  case 8: SRX_BUCKET_B(8); break;
  case 32: SRX_BUCKET_B(32); break;
  case 64: SRX_BUCKET_B(64); break;
  default: SRX_BUCKET_B(16); break;
  }
#undef SRX_BUCKET_B
}
void launch_range_batch(const batch_job* jobs, stage_map m, uint32_t blocks, hipStream_t s) {
  if (blocks) hipLaunchKernelGGL(bucket_range_batch_kernel, dim3(blocks), dim3(256), 0, s, jobs, m);
}
void launch_tile_order_batch(const batch_job* jobs, uint32_t njobs, hipStream_t s) {
  if (njobs) hipLaunchKernelGGL(tile_order_batch_kernel, dim3(njobs), dim3(1024), 0, s, jobs);
}
void launch_batch_check(const batch_job* jobs, uint32_t njobs, uint32_t capacity, int pt, uint32_t* status, hipStream_t s) {
  if (njobs)
    hipLaunchKernelGGL(batch_check_kernel, dim3((njobs + 255) / 256), dim3(256), 0, s, jobs, njobs, capacity,
                       static_cast<uint32_t>(256 * pt), status);
}

void launch_clear(const surface_desc& s, float4 v, hipStream_t st) {
  const size_t n = static_cast<size_t>(s.w) * s.h * s.samples;
  const size_t threads = pf_size(s.pf) == 12 ? n : std::max<size_t>(n * pf_size(s.pf) / 16, 1);
  if (n) hipLaunchKernelGGL(clear_kernel, dim3(static_cast<unsigned>((threads + 255) / 256)), dim3(256), 0, st, s, v);
}
void launch_clear_ds(const surface_desc& s, uint32_t flags, float depth, uint32_t stencil, hipStream_t st) {
  const size_t n = static_cast<size_t>(s.w) * s.h * s.samples;
  const size_t threads = flags == 3 ? std::max<size_t>(n / 2, 1) : n;
  if (n) hipLaunchKernelGGL(clear_ds_kernel, dim3(static_cast<unsigned>((threads + 255) / 256)), dim3(256), 0, st, s, flags, depth, stencil);
}
void launch_resolve(const surface_desc& src, const surface_desc& dst, hipStream_t st) {
  if (src.pf == PF_RGBA8 && dst.pf == PF_RGBA8 && src.samples == 4 && dst.samples == 1 && src.w == dst.w && src.h == dst.h) {
    const size_t n = static_cast<size_t>(src.w) * src.h;
    if (n) hipLaunchKernelGGL(resolve_rgba8x4_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, st, src, dst);
    return;
  }
  hipLaunchKernelGGL(resolve_kernel, dim3((src.w + 255) / 256, src.h), dim3(256), 0, st, src, dst);
}
void launch_mip(const surface_desc& src, const surface_desc& dst, int filter, hipStream_t st) {
  hipLaunchKernelGGL(mip_kernel, dim3((dst.w + 255) / 256, dst.h), dim3(256), 0, st, src, dst, filter);
}

}  // namespace srx
