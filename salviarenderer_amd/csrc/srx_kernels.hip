// HIP kernels of the Salvia rasterization pipeline for MI355X (gfx950).
//
// Draw pipeline (one HIP stream per renderer):
//   vs_kernel       vertex fetch + vertex shader, one thread per vertex    (stream_assembler.cpp,
//                   default_vertex_cache.cpp: the shader runs once per vertex instead of per cache miss)
//   setup_kernel    index fetch, near/far trivial accept, cull, winding, viewport transform and
//                   triangle setup, one thread per primitive; emits the (GPU tile, triangle) records of
//                   triangles on few tiles                                  (clipper.cpp, rasterizer.cpp:864-945)
//   clip_kernel     Sutherland-Hodgman near/far clipping for the few primitives that need it; emits the
//                   records of the clipped triangles and of those on many tiles
//   tile_ranges     tile ranges and classes from the record counts per tile
//   tile_scatter    scheduling order, parts of split tiles, records to their tiles' lists; in-order draws then
//                   sort each list (tile_sort), so it is in primitive order (the reference's per-tile
//                   std::sort, rasterizer.cpp:947-994)
//   inorder_kernel  (srx_inorder.hip) one workgroup per GPU tile, one thread per pixel; evaluates the
//                   reference's 64->16->4->sample decision chain (rasterizer.cpp:298-773) for the records of
//                   the tile's list, then every pixel's own in order: depth-stencil tests, pixel shader and
//                   blending (framebuffer.cpp)
//   raster_kernel   (srx_raster.hip) the same with one thread per 2x2 quad, for statistics queries, SASL
//                   pixel shaders, 32-pixel tiles and NOT_EQUAL depth.  Opaque early-Z draws defer the
//                   pixel shader to one pass over the final per-sample winners.
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
__device__ __forceinline__ void bin_edges(const float* e, tri_bin& t) {
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
__device__ __forceinline__ void bin_setup(const draw_params& P, const float* e, const float* bb, tri_bin& t) {
  const int tx = P.tiles_x, ty = P.tiles_y;
  t.sx = min(fast_floori(std_max(0.0f, bb[0]) / TILE), tx);
  t.sy = min(fast_floori(std_max(0.0f, bb[2]) / TILE), ty);
  t.ex = min(fast_ceili(std_max(0.0f, bb[1]) / TILE) + 1, tx);
  t.ey = min(fast_ceili(std_max(0.0f, bb[3]) / TILE) + 1, ty);
  t.small = (t.sx + 1 == t.ex) && (t.sy + 1 == t.ey);
  t.regions = (t.ex - t.sx) * (t.ey - t.sy) <= REGION_TEST_TILES;
  bin_edges(e, t);
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
// Batches: triangles over more than this many 64x64 tiles are counted by a whole wave (clip launch), not by
// setup's one lane, and emitted by a whole wave.  (Single draws emit as they set up; their rule is SMALL_SPAN.)
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

// The same for a triangle whose walk has been set up, keeping the first four GPU tiles for_each_gtile
// visits, packed as tile << 1 | full.
__device__ __forceinline__ uint32_t count_gtiles_pairs(const draw_params& P, const float* e, const float* bb,
                                                       const tri_bin& t, uint32_t (&k)[4]) {
  const int sub = TILE / P.gt;
  uint32_t n = 0;
  for (int y = t.sy; y < t.ey; ++y)
    for (int x = t.sx; x < t.ex; ++x) {
      bool full;
      uint64_t m = tile_gmask(P, e, bb, t, x, y, full);
      const uint32_t c = static_cast<uint32_t>(__popcll(m));
      for (uint32_t i = n; m && i < 4; m &= m - 1, ++i) {
        const int b = __builtin_ctzll(m);
        const uint32_t g = static_cast<uint32_t>((y * sub + b / sub) * P.gtiles_x + x * sub + b % sub);
        const uint32_t v = (g << 1) | (full ? 1u : 0u);
        if (i == 0) k[0] = v;
        else if (i == 1) k[1] = v;
        else if (i == 2) k[2] = v;
        else k[3] = v;
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
// Primitive p of the draw: near/far trivial accept, cull, winding, viewport transform, triangle setup.
// Sets the clip flag; returns whether the primitive gave a set-up triangle.
template <int NA>
__device__ __forceinline__ bool setup_primitive(const draw_params& P, const float4* __restrict__ vbuf, uint32_t p,
                                                uint8_t* __restrict__ clip_flag, uint32_t* __restrict__ counters,
                                                unsigned long long& cprims, tri_setup<NA>& t) {
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
    return false;
  }
  const bool front = compute_front(v[0].r[0], v[1].r[0], v[2].r[0]);
  if (cull_fn(P, front ? 1.0f : -1.0f)) return false;
  cprims = 1;
  // winding normalisation (clipper.cpp:59-65) by selects
  vtx<NA> o[3] = {v[0], vsel<NA>(front, v[1], v[2]), vsel<NA>(front, v[2], v[1])};
#pragma unroll
  for (int i = 0; i < 3; ++i) viewport_project<NA>(o[i], P);
  triangle_info<NA>(o[0], o[1], o[2], t);
  return t.valid;
}
// The fan-0 slots of the wave's 64 consecutive primitives (first of the block: bx * 256) are
// consecutive: the set-up triangles' words are stored coalesced.
template <int NA>
__device__ __forceinline__ void store_setup(const float4 (&rec)[5], const float4 (&attr)[3 * (NA + 1)], bool have,
                                            float4* __restrict__ tri_rec, float4* __restrict__ tri_attr, uint32_t bx,
                                            float4* stage) {
  const uint64_t mask = __ballot(have);
  if (!mask) return;
  const size_t p0 = static_cast<size_t>(bx) * 256 + (threadIdx.x & ~63u);
  float4* ws = stage + (threadIdx.x >> 6) * WAVE_STAGE;
  wave_store_blocks<5>(tri_rec + p0 * 5, rec, mask, ws);
  wave_store_blocks<3 * (NA + 1)>(tri_attr + p0 * 3 * (NA + 1), attr, mask, ws);
}

// Batches: counts each triangle's records (emitted at offsets from a scan of the counts).
template <int NA>
__device__ __forceinline__ void setup_count_body(const draw_params& P, const draw_buffers& B, uint32_t bx) {
  __shared__ float4 stage[4 * WAVE_STAGE];
  const uint32_t p = bx * 256 + threadIdx.x;
  unsigned long long cprims = 0;
  float4 rec[5], attr[3 * (NA + 1)];  // this lane's setup words, stored by the whole wave below
  bool have = false;
  if (p < P.prim_count) {
    uint32_t c0 = 0;  // records of fan triangle 0
    tri_setup<NA> t;
    have = setup_primitive<NA>(P, B.vbuf, p, B.clip_flag, B.counters, cprims, t);
    if (have) {
      tri_rec_words<NA>(t, rec);
      tri_attr_words<NA>(t, attr);
      float e[9], bb[4];
      for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) e[i * 3 + j] = t.e[i][j];
      for (int i = 0; i < 4; ++i) bb[i] = t.bb[i];
      if (bin_span(P, bb) > COUNT_WIDE)
        B.wide_list[atomicAdd(&B.counters[CT_WIDE], 1u)] = p;  // counted in the clip launch
      else
        c0 = count_gtiles(P, e, bb);
    }
    B.cnt[3 * p] = c0;
    B.cnt[3 * p + 1] = 0;
    B.cnt[3 * p + 2] = 0;
  }
  store_setup<NA>(rec, attr, have, B.tri_rec, B.tri_attr, bx, stage);
}

// ---------------------------------------------------------------- records of single draws
// A record is (GPU tile, triangle id << 1 | full, rank among the tile's records).  Records are emitted
// as triangles are set up, at positions taken from the draw's cursor (counters[CT_TOTAL]) a workgroup
// at a time, in no particular order: the rank comes from the tile's count, so the tiles' lists need no
// counting pass afterwards, and draws that need primitive order sort each tile's list.  Records
// beyond `capacity` are counted and dropped (the host compares the total with it and repeats).
//
// A triangle is emitted by the lane that set it up when its box lies on at most four GPU tiles and nine
// 64x64 tiles (a box inside one 64x64 tile spans four of them, see bin_setup); any other goes to the
// wide list, whose (triangle, 64x64 tile) pairs the clip launch spreads over all lanes.  Walking up to
// 32 64x64 tiles in one lane, and emitting long lists by the lane's wave one triangle after another,
// took 117 + 72 + 342 us of a 2,000-triangle draw at 512x512, which leaves 32 waves to do it; setup now
// takes 7 and the clip launch 31 us there.  What bounds the clip launch is the tiles' counts: 330k
// device atomics take 14 us however they are spread.
constexpr int SMALL_SPAN = 9;
__device__ __forceinline__ void put_record(const draw_buffers& B, uint32_t capacity, uint32_t pos, uint32_t tile,
                                           uint32_t val, uint32_t rank) {
  if (pos < capacity) {
    B.keys[0][pos] = tile;
    B.vals[0][pos] = val;
    B.keys[1][pos] = rank;
  }
}

// Ranks of one record per lane (of lanes with `valid`) in their tiles.  Lanes on the same tile are
// matched in the wave and their tile's count is taken with one atomic: consecutive triangles lie on the
// same few tiles, where an atomic per record serialises (590k records: 400 us).  Lanes still unmatched
// after RANK_ROUNDS tiles take their own (scattered triangles: their atomics do not meet).
constexpr int RANK_ROUNDS = 16;
__device__ __forceinline__ uint32_t take_ranks(const draw_buffers& B, uint32_t slot_shift, uint32_t tile, bool valid) {
  const int lane = __lane_id();
  int leader = lane;
  uint32_t rank = 0, n = 1;
  bool open = valid;
  for (int it = 0; it < RANK_ROUNDS; ++it) {
    const uint64_t left = __ballot(open);
    if (!left) break;
    const int first = __builtin_ctzll(left);
    const uint32_t t0 = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(tile), first));
    const bool same = open && tile == t0;
    const uint64_t m = __ballot(same);
    if (same) {
      leader = first;
      rank = static_cast<uint32_t>(__popcll(m & ((1ull << lane) - 1ull)));
      n = static_cast<uint32_t>(__popcll(m));
      open = false;
    }
  }
  uint32_t old = 0;
  if (valid && leader == lane) old = atomicAdd(&B.tile_count[tile_slot(tile, slot_shift)], n);
  return static_cast<uint32_t>(__shfl(static_cast<int>(old), leader, 64)) + rank;
}

// One workgroup: 256 primitives.
template <int NA>
__global__ void __launch_bounds__(256) setup_kernel(draw_params P, draw_buffers B, uint32_t capacity, uint32_t slot_shift) {
  __shared__ float4 stage[4 * WAVE_STAGE];
  __shared__ uint32_t wtot[4], s_base, s_wide;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, bx = blockIdx.x;
  const uint32_t p = bx * 256 + tid;
  unsigned long long cprims = 0;
  uint32_t c = 0;     // records this lane emits (its triangle's, when it is small)
  bool wide = false;  // left to the clip launch
  uint32_t kp[4] = {0, 0, 0, 0};
  {
    float4 rec[5], attr[3 * (NA + 1)];
    bool have = false;
    if (p < P.prim_count) {
      tri_setup<NA> t;
      have = setup_primitive<NA>(P, B.vbuf, p, B.clip_flag, B.counters, cprims, t);
      if (have) {
        tri_rec_words<NA>(t, rec);
        tri_attr_words<NA>(t, attr);
        float e[9], bb[4];
        for (int i = 0; i < 3; ++i)
          for (int j = 0; j < 3; ++j) e[i * 3 + j] = t.e[i][j];
        for (int i = 0; i < 4; ++i) bb[i] = t.bb[i];
        tri_bin w;
        bin_setup(P, e, bb, w);
        if (w.ex > w.sx && w.ey > w.sy) {
          const float inv = 1.0f / static_cast<float>(P.gt);
          const float gw = floorf(bb[1] * inv) - floorf(bb[0] * inv) + 1.0f, gh = floorf(bb[3] * inv) - floorf(bb[2] * inv) + 1.0f;
          wide = !(gw * gh <= 4.0f) || (w.ex - w.sx) * (w.ey - w.sy) > SMALL_SPAN;
          if (!wide) {
            c = count_gtiles_pairs(P, e, bb, w, kp);
            if (c > 4) {  // the corner tests accept tiles beyond the box of a triangle far below a pixel
              wide = true;
              c = 0;
            }
          }
        }
      }
    }
    store_setup<NA>(rec, attr, have, B.tri_rec, B.tri_attr, bx, stage);
  }
  const uint32_t incl = wave_incl_scan(c | (wide ? 0x10000u : 0u));
  if (lane == 63) wtot[wave] = incl;
  __syncthreads();  // the staging area is stored
  uint32_t before = 0, total = 0;
#pragma unroll
  for (uint32_t w = 0; w < 4; ++w) {
    if (w < wave) before += wtot[w];
    total += wtot[w];
  }
  const uint32_t off = before + incl - (c | (wide ? 0x10000u : 0u));
  const uint32_t nrec = total & 0xFFFFu;
  if (tid == 0 && total) {
    // the record cursor and the wide list's length are one 64-bit word
    const unsigned long long old =
        atomicAdd(reinterpret_cast<unsigned long long*>(B.counters + CT_TOTAL),
                  static_cast<unsigned long long>(nrec) | (static_cast<unsigned long long>(total >> 16) << 32));
    s_base = static_cast<uint32_t>(old);
    s_wide = static_cast<uint32_t>(old >> 32);
  }
  uint32_t rank[4];
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) {
    rank[i] = 0;
    if (__ballot(i < c)) rank[i] = take_ranks(B, slot_shift, kp[i] >> 1, i < c);
  }
  __syncthreads();
  if (nrec) {
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i)
      if (i < c) put_record(B, capacity, s_base + (off & 0xFFFFu) + i, kp[i] >> 1, (3 * p) << 1 | (kp[i] & 1u), rank[i]);
  }
  if (wide && s_wide + (off >> 16) < P.prim_count) B.wide_list[s_wide + (off >> 16)] = p;
  if (P.count_stats) block_partial(B.partial, cprims);  // uniform over the launch
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

// Batches: the clip launch counts the records of the triangles it clips and of those on the wide list.
template <int NA>
__device__ __forceinline__ void clip_count_body(const draw_params& P, const draw_buffers& B, uint32_t bx, uint32_t gx) {
  const uint32_t nclip = B.counters[CT_CLIP_PRIMS], nwide = B.counters[CT_WIDE];
  // triangles over many 64x64 tiles: one wave counts each one's records
  const uint32_t wave = (bx * blockDim.x + threadIdx.x) >> 6, waves = (gx * blockDim.x) >> 6;
  for (uint32_t w = wave; w < nwide; w += waves) {
    const uint32_t p = B.wide_list[w];
    float e[9], bb[4];
    read_tri_rec(B.tri_rec + static_cast<size_t>(p) * 5, e, bb);  // fan 0 of primitive p
    const uint32_t n = count_gtiles_wave(P, e, bb);
    if (__lane_id() == 0) B.cnt[3 * p] = n;
  }
  if (nclip == 0) return;
  // lanes clip the flagged primitives among the wave's 64; the wave then counts the records of the
  // resulting triangles together (clipped triangles are few and often reach across the target)
  const int lane = __lane_id();
  for (uint32_t b = wave * 64; b < P.prim_count; b += waves * 64) {
    const uint32_t p = b + static_cast<uint32_t>(lane);
    uint32_t fans = 0;  // bit k: fan triangle 3p + k was set up
    if (p < P.prim_count && B.clip_flag[p])
      fans = clip_primitive<NA>(P, p, B.vbuf, B.tri_rec, B.tri_attr, B.clip_slot, B.clip_verts, B.clip_hdr, B.clip_capacity,
                                B.counters, B.stats);
    __threadfence();  // the fans' records are read back by every lane of the wave
    for (unsigned long long m = __ballot(fans != 0); m; m &= m - 1) {
      const int src = __builtin_ctzll(m);
      const uint32_t fs = static_cast<uint32_t>(__shfl(static_cast<int>(fans), src, 64));
      const uint32_t ps = b + static_cast<uint32_t>(src);
      for (int k = 0; k < 3; ++k) {
        if (!(fs & (1u << k))) continue;
        const uint32_t id = 3 * ps + k;
        float e[9], bb[4];
        read_tri_rec(B.tri_rec + tri_slot(P, id) * 5, e, bb);
        const uint32_t n = count_gtiles_wave(P, e, bb);
        if (lane == 0) B.cnt[id] = n;
      }
    }
  }
}

// The workgroup emits the records of its lanes' triangles (`has`: lane's triangle `id`, set up in
// B.tri_rec): their (triangle, 64x64 tile) pairs are numbered consecutively and taken one per lane, so
// a triangle over the whole target and a hundred small ones fill the lanes alike.  The records of
// WIDE_STEP pairs per lane then take their positions together and are listed in LDS, so that consecutive
// lanes write consecutive records and no lane waits for another's longer list.  Every thread of the
// workgroup calls it.
constexpr uint32_t WIDE_STEP = 4;
constexpr uint32_t WIDE_LIST = 4096;  // records listed at a time
struct wide_lds {
  uint16_t list[WIDE_LIST];  // pair << 4 | GPU tile of the pair's 64x64 tile
  float4 tri[256 * 4];  // edges, bounding box, first 64x64 tile and columns, id
  uint2 pair[256 * WIDE_STEP];  // a pair's first GPU tile; GPU tile mask | full << 16 | owner lane << 17
  uint32_t pre[256];  // pairs of the lanes up to and including this one
  uint32_t wsum[4], base;
};
__device__ __forceinline__ void emit_wide(const draw_params& P, const draw_buffers& B, uint32_t capacity,
                                          uint32_t slot_shift, bool has, uint32_t id, wide_lds& L) {
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t R = 0;
  if (has) {
    float e[9], bb[4];
    read_tri_rec(B.tri_rec + tri_slot(P, id) * 5, e, bb);
    tri_bin t;
    bin_setup(P, e, bb, t);
    if (t.ex > t.sx && t.ey > t.sy) R = static_cast<uint32_t>((t.ex - t.sx) * (t.ey - t.sy));
    L.tri[tid * 4] = make_float4(e[0], e[1], e[2], e[3]);
    L.tri[tid * 4 + 1] = make_float4(e[4], e[5], e[6], e[7]);
    L.tri[tid * 4 + 2] = make_float4(e[8], bb[0], bb[1], bb[2]);
    // at most 129 64x64 tiles a side (targets are at most 8192 wide)
    L.tri[tid * 4 + 3] = make_float4(bb[3], __uint_as_float(static_cast<uint32_t>(t.sx) | (static_cast<uint32_t>(t.sy) << 10) |
                                                            (static_cast<uint32_t>(t.ex - t.sx) << 20)),
                                     __uint_as_float(id), __uint_as_float((t.small ? 1u : 0u) | (t.regions ? 2u : 0u)));
  }
  const uint32_t incl = wave_incl_scan(R);
  if (lane == 63) L.wsum[wave] = incl;
  __syncthreads();
  uint32_t before = 0, total = 0;
#pragma unroll
  for (uint32_t w = 0; w < 4; ++w) {
    if (w < wave) before += L.wsum[w];
    total += L.wsum[w];
  }
  L.pre[tid] = before + incl;
  __syncthreads();
  const int sub = TILE / P.gt;
  for (uint32_t q0 = 0; q0 < total; q0 += 256 * WIDE_STEP) {
    uint32_t n = 0;  // records of this lane's pairs
#pragma unroll 1
    for (uint32_t u = 0; u < WIDE_STEP; ++u) {
      const uint32_t q = q0 + u * 256 + tid;
      uint2 pr = make_uint2(0, 0);
      if (q < total) {
        uint32_t o = 0;  // the first lane with q < pre[o]
#pragma unroll
        for (uint32_t step = 128; step; step >>= 1)
          if (L.pre[o + step - 1] <= q) o += step;
        const uint32_t local = q - (o ? L.pre[o - 1] : 0u);
        const float4 a = L.tri[o * 4], b = L.tri[o * 4 + 1], c = L.tri[o * 4 + 2], d = L.tri[o * 4 + 3];
        const float e[9] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, c.x}, bb[4] = {c.y, c.z, c.w, d.x};
        const uint32_t box = __float_as_uint(d.y), flags = __float_as_uint(d.w);
        const uint32_t w = box >> 20;
        tri_bin t;
        t.small = (flags & 1u) != 0;
        t.regions = (flags & 2u) != 0;
        bin_edges(e, t);
        const int x = static_cast<int>((box & 1023u) + local % w), y = static_cast<int>(((box >> 10) & 1023u) + local / w);
        bool full;
        const uint32_t m = static_cast<uint32_t>(tile_gmask(P, e, bb, t, x, y, full));  // GPU tiles of 16 or 32 pixels
        n += __popc(m);
        pr = make_uint2(static_cast<uint32_t>(y * sub * P.gtiles_x + x * sub), m | (full ? 0x10000u : 0u) | (o << 17));
      }
      L.pair[u * 256 + tid] = pr;
    }
    const uint32_t in = wave_incl_scan(n);
    if (lane == 63) L.wsum[wave] = in;
    __syncthreads();
    uint32_t pos = in - n, all = 0;
#pragma unroll
    for (uint32_t w = 0; w < 4; ++w) {
      if (w < wave) pos += L.wsum[w];
      all += L.wsum[w];
    }
    if (tid == 0 && all) {
      L.base = atomicAdd(&B.counters[CT_TOTAL], all);
      if (L.base > ~all) B.counters[CT_OVERRUN] = 1;
    }
    __syncthreads();
    const uint32_t base = L.base;
    for (uint32_t w0 = 0; w0 < all; w0 += WIDE_LIST) {
      uint32_t at = pos - w0;  // this lane's next entry of the window (wraps below it)
#pragma unroll 1
      for (uint32_t u = 0; u < WIDE_STEP; ++u)
        for (uint32_t m = L.pair[u * 256 + tid].y & 0xFFFFu; m; m &= m - 1, ++at)
          if (at < WIDE_LIST) L.list[at] = static_cast<uint16_t>(((u * 256 + tid) << 4) | static_cast<uint32_t>(__builtin_ctz(m)));
      __syncthreads();
      const uint32_t nw = min(all - w0, WIDE_LIST);
      for (uint32_t r0 = 0; r0 < nw; r0 += 1024) {
        uint32_t tile[4], val[4], rank[4];
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {  // four ranks in flight
          const uint32_t r = r0 + i * 256 + tid;
          const uint32_t en = L.list[min(r, nw - 1)];
          const uint2 pr = L.pair[en >> 4];
          const int b = static_cast<int>(en & 15u);
          tile[i] = pr.x + static_cast<uint32_t>((b / sub) * P.gtiles_x + b % sub);
          val[i] = (__float_as_uint(L.tri[(pr.y >> 17) * 4 + 3].z) << 1) | ((pr.y >> 16) & 1u);
          rank[i] = r < nw ? atomicAdd(&B.tile_count[tile_slot(tile[i], slot_shift)], 1u) : 0u;
        }
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
          const uint32_t r = r0 + i * 256 + tid;
          if (r < nw) put_record(B, capacity, base + w0 + r, tile[i], val[i], rank[i]);
        }
      }
      __syncthreads();
    }
    __syncthreads();  // the sums, the base and the pairs are used again
  }
}

// Single draws: emits the records of the wide list's triangles, then clips the flagged primitives and
// emits theirs.  A draw with neither returns at once.
template <int NA>
__global__ void __launch_bounds__(256) clip_kernel(draw_params P, draw_buffers B, uint32_t capacity, uint32_t slot_shift) {
  __shared__ wide_lds L;
  const uint32_t nclip = B.counters[CT_CLIP_PRIMS], nwide = min(B.counters[CT_WIDE], P.prim_count);
  const uint32_t tid = threadIdx.x;
  const uint32_t per = min(max((nwide + gridDim.x - 1) / gridDim.x, 1u), 256u);  // triangles per workgroup and turn
  for (uint32_t g = blockIdx.x * per; g < nwide; g += gridDim.x * per) {
    const bool has = tid < min(per, nwide - g);
    emit_wide(P, B, capacity, slot_shift, has, has ? 3 * B.wide_list[g + tid] : 0u, L);
    __syncthreads();
  }
  if (nclip == 0) return;
  for (uint32_t b = blockIdx.x * 256; b < P.prim_count; b += gridDim.x * 256) {
    const uint32_t p = b + tid;
    uint32_t fans = 0;  // bit k: fan triangle 3p + k was set up
    if (p < P.prim_count && B.clip_flag[p])
      fans = clip_primitive<NA>(P, p, B.vbuf, B.tri_rec, B.tri_attr, B.clip_slot, B.clip_verts, B.clip_hdr, B.clip_capacity,
                                B.counters, B.stats);
    for (uint32_t k = 0; k < 3; ++k) {
      const bool has = ((fans >> k) & 1u) != 0;
      if (!__syncthreads_or(has)) continue;
      emit_wide(P, B, capacity, slot_shift, has, 3 * p + k, L);
      __syncthreads();
    }
  }
}

// ============================================================== record emission (batches)
// off: exclusive scan of the per-triangle record counts; a triangle owns [off[id], off[id+1]).
// One thread per primitive, over its (at most 3) clipped triangles in fan order.  Records beyond
// `capacity` are dropped; the batch's status word reports them.

// Records of one clipped triangle emitted by a whole wave: lanes take the triangle's 64x64 tiles in
// for_each_gtile's order, count each tile's GPU tiles with the same tests, and write at their
// wave-scanned offsets -- for triangles that reach many tiles, which one lane would walk serially.
__device__ __forceinline__ void emit_wave(const draw_params& P, const float4* __restrict__ tri_rec, uint32_t id,
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
__device__ __forceinline__ void emit_records(const draw_params& P, const float4* __restrict__ tri_rec, uint32_t p,
                                             const uint32_t (&o)[4], uint32_t capacity,
                                             uint32_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  uint32_t wide = 0;  // fan triangles left to the wave
  if (p < P.prim_count) {
    const uint32_t id3 = 3 * p;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const uint32_t id = id3 + k;
      const uint32_t first = o[k], next = o[k + 1];
      if (next == first) continue;
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
      emit_wave(P, tri_rec, 3 * ps + k, first, next, capacity, keys, vals);
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
  emit_records(P, tri_rec, p, o, capacity, keys, vals);
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

// ---------------------------------------------------------------- one-pass bucket sort by GPU tile
// Batches: the order of a tile's records is immaterial, so one counting pass bins them: per-workgroup
// tile histograms in LDS, one scan of the tile-major histogram, and a scatter whose in-workgroup
// ranks come from LDS atomics.
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

// ---------------------------------------------------------------- tile ranges of single draws
// Each tile's range of the lists and its place in its record-count class, both from cursors a wave takes
// its share of at once: neither the ranges nor the tiles of a class need an order, so no workgroup
// waits for another's counts.  The lists' launch, which knows every class's count, makes the scheduling
// order of the places.  (A scan over all counts took 12 us whatever the number of tiles.)
constexpr uint32_t PLACE_BITS = 28;  // a place: class << PLACE_BITS | rank (targets have at most 2^18 GPU tiles)
__global__ void __launch_bounds__(256) tile_ranges_kernel(const uint32_t* __restrict__ tile_count, uint32_t T, uint32_t N,
                                                          uint32_t shift, uint32_t* __restrict__ ts, uint32_t* __restrict__ te,
                                                          uint32_t* __restrict__ counters, uint32_t* __restrict__ place) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  const int lane = __lane_id();
  const uint32_t t = slot_tile(i, shift);
  const bool valid = i < N && t < T;
  const uint32_t n = valid ? tile_count[i] : 0u;
  const uint32_t incl = wave_incl_scan(n);
  const uint32_t all = static_cast<uint32_t>(__shfl(static_cast<int>(incl), 63, 64));
  uint32_t base = 0;
  if (lane == 0 && all) base = atomicAdd(&counters[CT_CURSOR], all);
  // lanes of the same class, matched by one ballot per class bit
  const uint32_t c = tile_class(n);
  uint64_t m = __ballot(valid);
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const bool bit = ((c >> b) & 1u) != 0;
    const uint64_t bal = __ballot(bit);
    m &= bit ? bal : ~bal;
  }
  const int leader = valid ? __builtin_ctzll(m) : lane;
  uint32_t old = 0;
  if (valid && leader == lane) old = atomicAdd(&counters[CT_CLASS + c], static_cast<uint32_t>(__popcll(m)));
  const uint32_t at = static_cast<uint32_t>(__shfl(static_cast<int>(old), leader, 64)) +
                      static_cast<uint32_t>(__popcll(m & ((1ull << lane) - 1ull)));
  base = static_cast<uint32_t>(__shfl(static_cast<int>(base), 0, 64));
  if (valid) {
    ts[t] = base + incl - n;
    te[t] = base + incl;
    place[t] = (c << PLACE_BITS) | at;
    if (n >= VIS_PART_SMALL) atomicAdd(&counters[CT_STEP + vis_step(n)], 1u);
  }
}
// The scheduling order, the parts of split tiles and the mail (workgroups of the tiles), and the records to their
// tiles' lists (the others): position = first record of the tile + rank in it.
constexpr uint32_t SCATTER_PER_THREAD = 4;
__global__ void __launch_bounds__(256) tile_scatter_kernel(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ vals,
                                                           const uint32_t* __restrict__ ranks,
                                                           const uint32_t* __restrict__ counters, uint32_t cap,
                                                           const uint32_t* __restrict__ ts, const uint32_t* __restrict__ te,
                                                           uint32_t* __restrict__ vout,
                                                           uint32_t T, const uint32_t* __restrict__ place,
                                                           uint32_t* __restrict__ order, bool split, uint32_t prims,
                                                           uint32_t tile_cost, uint32_t* __restrict__ ct_parts,
                                                           uint32_t* __restrict__ ct_merges, uint4* __restrict__ parts,
                                                           uint4* __restrict__ merges, draw_mail* mail, uint32_t seq) {
  const uint32_t total = record_total(counters);
  const bool may_split = split && total <= cap;  // with more records the tables' bounds do not hold
  const uint32_t part = may_split ? vis_part(prims, total, busy_tiles(counters, T), tile_cost) : 0u;
  if (blockIdx.x == 0 && threadIdx.x < 64) {  // the counts are final; the host waits for seq
    uint32_t split_tiles = 0;
    if (may_split && counters[CT_CLASS] + counters[CT_CLASS + 1])  // a tile of VIS_PART_SMALL records or more
      for (uint32_t k = vis_step(part + 1) + threadIdx.x; k < VIS_STEPS; k += 64) split_tiles += counters[CT_STEP + k];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) split_tiles += static_cast<uint32_t>(__shfl_xor(static_cast<int>(split_tiles), off, 64));
    if (threadIdx.x == 0) {
      mail->total = total;
      mail->merges = split_tiles;
      mail->clip_overflow = counters[CT_CLIP_OVERFLOW];
      __hip_atomic_store(&mail->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
  const uint32_t tile_blocks = (T + 255) / 256;
  if (blockIdx.x < tile_blocks) {
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    if (t >= T) return;
    const uint32_t c = place[t] >> PLACE_BITS;
    uint32_t at = place[t] & ((1u << PLACE_BITS) - 1u);
#pragma unroll
    for (uint32_t k = 0; k + 1 < TILE_CLASSES; ++k) at += k < c ? counters[CT_CLASS + k] : 0u;
    order[at] = t;
    const uint32_t len = may_split ? te[t] - ts[t] : 0u;
    if (may_split && len > part) {
      const uint32_t np = (len + part - 1) / part;
      const uint32_t e = atomicAdd(ct_parts, np);
      merges[atomicAdd(ct_merges, 1u)] = make_uint4(t, np, e, 0u);
      for (uint32_t k = 0; k < np; ++k) parts[e + k] = make_uint4(t, k, np, 0u);
    }
    return;
  }
  const uint32_t n = min(total, cap);
  const uint32_t b0 = (blockIdx.x - tile_blocks) * (256 * SCATTER_PER_THREAD);
  if (b0 >= n) return;
  uint32_t k[SCATTER_PER_THREAD], v[SCATTER_PER_THREAD], r[SCATTER_PER_THREAD];
#pragma unroll
  for (uint32_t j = 0; j < SCATTER_PER_THREAD; ++j) {  // clamped indices: no branch per load
    const uint32_t i = min(b0 + j * 256 + threadIdx.x, n - 1);
    k[j] = keys[i];
    v[j] = vals[i];
    r[j] = ranks[i];
  }
#pragma unroll
  for (uint32_t j = 0; j < SCATTER_PER_THREAD; ++j) {
    const uint32_t pos = ts[k[j]] + r[j];
    if (b0 + j * 256 + threadIdx.x < n && pos < cap) vout[pos] = v[j];  // beyond cap: the draw is emitted again
  }
}

// Each tile's list in ascending order (primitive order: a triangle is on a tile once), from `in` to `out`, one
// workgroup per tile.  Lists of up to SORT_LDS records are sorted in LDS.  A longer one is partitioned by the
// leading 8 bits of its values (a histogram, then every record to its bucket in the other buffer, in any
// order: the values are distinct), runs of buckets that fit are sorted in LDS, and a bucket that does not fit
// is partitioned by its next 8 bits, back into the first buffer.  Every level reads its records twice, and
// three levels leave buckets of at most 256 values, so the time grows with the list's length (blended
// triangles on the same 16 tiles: 100,000 of them 9.7 ms a frame, 300,000 29, a million small ones 19; with
// windows of SORT_LDS records, each found by reading the whole list, 14.6, 72 and 93).  Sorting the lists costs in-order draws a pass over their records; two stable radix
// passes over all records (by tile) took 50 us of a 32k-triangle draw at 1280x720.
constexpr uint32_t SORT_LDS = 2048, SORT_LEVELS = 3, SORT_FLIGHT = 8;
struct sort_space {
  uint32_t a[SORT_LDS];
  uint32_t hist[256];
  uint32_t start[SORT_LEVELS][257];  // the buckets of a level's partition
  uint32_t wsum[4];
};
__device__ __forceinline__ void sort_lds(uint32_t* a, uint32_t n) {
  uint32_t m = 2;
  while (m < n) m <<= 1;  // uniform
  for (uint32_t i = n + threadIdx.x; i < m; i += 256) a[i] = 0xFFFFFFFFu;
  for (uint32_t k = 2; k <= m; k <<= 1)
    for (uint32_t j = k >> 1; j; j >>= 1) {
      __syncthreads();
      for (uint32_t t = threadIdx.x; t < m / 2; t += 256) {
        const uint32_t i = ((t & ~(j - 1)) << 1) | (t & (j - 1));  // bit j clear
        const uint32_t x = a[i], y = a[i + j];
        if ((x > y) == ((i & k) == 0)) {
          a[i] = y;
          a[i + j] = x;
        }
      }
    }
  __syncthreads();
}
// f(x[i]) for i < n, SORT_FLIGHT loads of a lane in flight.
template <class F>
__device__ __forceinline__ void sort_each(const uint32_t* x, uint32_t n, F&& f) {
  for (uint32_t i0 = threadIdx.x; i0 < n; i0 += 256 * SORT_FLIGHT) {
    uint32_t v[SORT_FLIGHT];
#pragma unroll
    for (uint32_t j = 0; j < SORT_FLIGHT; ++j) v[j] = x[min(i0 + j * 256, n - 1)];
#pragma unroll
    for (uint32_t j = 0; j < SORT_FLIGHT; ++j)
      if (i0 + j * 256 < n) f(v[j]);
  }
}
// Sorts x[0, n), n > SORT_LDS, whose values agree above bit shift + 8, into o, the buffer that holds x on odd
// levels and y on even ones.
template <uint32_t LEVEL>
__device__ __forceinline__ void sort_long(uint32_t* x, uint32_t* y, uint32_t* o, uint32_t n, uint32_t shift, sort_space& L) {
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t* start = L.start[LEVEL];
  while (true) {
    L.hist[tid] = 0;
    __syncthreads();
    sort_each(x, n, [&](uint32_t v) { atomicAdd(&L.hist[(v >> shift) & 255u], 1u); });
    __syncthreads();
    const uint32_t c = L.hist[tid];
    if (!__syncthreads_or(c == n) || shift == 0) break;
    shift = shift > 8 ? shift - 8 : 0;  // all in one bucket: by the next bits
  }
  const uint32_t c = L.hist[tid], incl = wave_incl_scan(c);
  if (lane == 63) L.wsum[wave] = incl;
  __syncthreads();
  uint32_t before = 0;
#pragma unroll
  for (uint32_t w = 0; w < 4; ++w)
    if (w < wave) before += L.wsum[w];
  start[tid + 1] = before + incl;
  if (tid == 0) start[0] = 0;
  L.hist[tid] = before + incl - c;
  __syncthreads();
  sort_each(x, n, [&](uint32_t v) { y[atomicAdd(&L.hist[(v >> shift) & 255u], 1u)] = v; });
  __syncthreads();  // the buckets are written
  uint32_t b = 0;
  while (b < 256) {
    const uint32_t s = start[b];
    uint32_t e = b;
    while (e < 256 && start[e + 1] - s <= SORT_LDS) ++e;  // uniform
    if (e > b) {
      const uint32_t m = start[e] - s;
      if (m) {
        for (uint32_t i = tid; i < m; i += 256) L.a[i] = y[s + i];
        sort_lds(L.a, m);
        for (uint32_t i = tid; i < m; i += 256) o[s + i] = L.a[i];
        __syncthreads();
      }
      b = e;
    } else {
      if constexpr (LEVEL + 1 < SORT_LEVELS)
        sort_long<LEVEL + 1>(y + s, x + s, o + s, start[b + 1] - s, shift > 8 ? shift - 8 : 0, L);
      ++b;
    }
  }
}
// bits: the values lie below 1 << bits.
__global__ void __launch_bounds__(256) tile_sort_kernel(const uint32_t* __restrict__ ts, const uint32_t* __restrict__ te,
                                                        const uint32_t* __restrict__ order, const uint32_t* __restrict__ counters,
                                                        uint32_t cap, uint32_t bits, uint32_t* in, uint32_t* out) {
  __shared__ sort_space L;
  if (record_total(counters) > cap) return;  // records were dropped: the draw is emitted again
  const uint32_t t = order[blockIdx.x], t0 = ts[t], n = te[t] - t0, tid = threadIdx.x;
  if (n > SORT_LDS) {
    sort_long<0>(in + t0, out + t0, out + t0, n, bits > 8 ? bits - 8 : 0, L);
    return;
  }
  if (n == 0) return;
  for (uint32_t i = tid; i < n; i += 256) L.a[i] = in[t0 + i];
  if (n > 1) sort_lds(L.a, n);
  for (uint32_t i = tid; i < n; i += 256) out[t0 + i] = L.a[i];
}

void launch_tile_ranges(const draw_params& P, const draw_buffers& B, hipStream_t s) {
  const uint32_t T = static_cast<uint32_t>(P.gtiles_x * P.gtiles_y);
  if (!T) return;
  const uint32_t N = tile_slots(T), shift = tile_slot_shift(T);
  hipLaunchKernelGGL(tile_ranges_kernel, dim3((N + 255) / 256), dim3(256), 0, s, B.tile_count, T, N, shift, B.tstart, B.tend,
                     B.counters, reinterpret_cast<uint32_t*>(B.partial));
}
void launch_tile_lists(const draw_params& P, const draw_buffers& B, uint32_t cap, uint32_t* order, bool sorted, draw_mail* mail,
                       uint32_t seq, hipStream_t s) {
  const uint32_t T = static_cast<uint32_t>(P.gtiles_x * P.gtiles_y);
  if (!T) return;
  const uint32_t per = 256 * SCATTER_PER_THREAD;
  hipLaunchKernelGGL(tile_scatter_kernel, dim3((T + 255) / 256 + (std::max<uint32_t>(cap, 1) + per - 1) / per), dim3(256), 0, s, B.keys[0], B.vals[0],
                     B.keys[1], B.counters, cap, B.tstart, B.tend, B.vals[1], T, reinterpret_cast<const uint32_t*>(B.partial),
                     order, B.vis_split, P.prim_count, B.tile_cost, B.counters + CT_PARTS,
                     B.counters + CT_MERGES, B.vis_parts, B.vis_merges, mail, seq);
  if (sorted) {
    uint32_t bits = 1;  // the values are below 6 * prim_count
    while (bits < 32 && (6ull * P.prim_count) >> bits) ++bits;
    hipLaunchKernelGGL(tile_sort_kernel, dim3(T), dim3(256), 0, s, B.tstart, B.tend, B.order, B.counters, cap, bits, B.vals[1],
                       B.vals[0]);
  }
}

// Batches: scheduling order of the GPU tiles, heaviest first so that the longest tiles start early.  Tiles
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
void launch_fill_u32(uint32_t* p, uint32_t n, uint32_t v, hipStream_t s) {
  if (n) hipLaunchKernelGGL(fill_u32_kernel, dim3((n + 255) / 256), dim3(256), 0, s, p, n, v);
}

void launch_reduce_partials(const unsigned long long* partial, uint32_t n, unsigned long long* stats, int slot, hipStream_t s) {
  hipLaunchKernelGGL(reduce_partials_kernel, dim3(1), dim3(256), 0, s, partial, n, stats, slot);
}

void launch_vs(const draw_params& P, float4* vbuf, uint32_t* counters, uint32_t* tiles, size_t ntiles, hipStream_t s) {
  uint32_t n = P.nverts + 1;
  hipLaunchKernelGGL(vs_kernel, dim3((n + 255) / 256), dim3(256), 0, s, P, vbuf, counters, tiles,
                     static_cast<uint32_t>(ntiles));
}

void launch_setup(const draw_params& P, const draw_buffers& B, uint32_t capacity, hipStream_t s) {
  if (P.prim_count == 0) return;
  dim3 grid((P.prim_count + 255) / 256);
  const uint32_t shift = tile_slot_shift(static_cast<uint32_t>(P.gtiles_x * P.gtiles_y));
#define SRX_SETUP(NA) hipLaunchKernelGGL(setup_kernel<NA>, grid, dim3(256), 0, s, P, B, capacity, shift)
  SRX_NA_DISPATCH(P.nattr, SRX_SETUP)
#undef SRX_SETUP
  if (P.count_stats) launch_reduce_partials(B.partial, grid.x, B.stats, ST_CPRIMITIVES, s);
}

// Workgroups of the clip launch: enough to fill the GPU four deep when every triangle is on the wide
// list, few enough that a draw with none (they return at once) loses nothing measurable.
void launch_clip(const draw_params& P, const draw_buffers& B, uint32_t capacity, hipStream_t s) {
  if (P.prim_count == 0) return;
  dim3 grid(std::min<uint32_t>((P.prim_count + 3) / 4, 1024));
  const uint32_t shift = tile_slot_shift(static_cast<uint32_t>(P.gtiles_x * P.gtiles_y));
#define SRX_CLIP(NA) hipLaunchKernelGGL(clip_kernel<NA>, grid, dim3(256), 0, s, P, B, capacity, shift)
  SRX_NA_DISPATCH(P.nattr, SRX_CLIP)
#undef SRX_CLIP
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
  setup_count_body<NA>(J.P, J.B, lb);
}

template <int NA>
__global__ void clip_batch_kernel(const batch_job* __restrict__ jobs, stage_map m) {
  uint32_t lb, nb;
  const batch_job& J = jobs[stage_job(m, lb, nb)];
  clip_count_body<NA>(J.P, J.B, lb, nb);
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
