// Run-time compilation of SASL pixel shaders to gfx950 code: the reference JIT-compiles SASL
// through LLVM to host code (sasl/src/codegen, salvia/src/core/renderer.cpp compile()); here the
// register program is translated to HIP C++ -- straight-line code with the quad's registers in
// VGPRs, every operand, swizzle and write mask resolved at translation time and the masks of
// if/loops kept in variables -- and compiled with hiprtc into the deferred SASL shading kernel
// (one lane per pixel, a quad in 4 lanes; the interpreter, sasl_shade_kernel in srx_kernels.hip,
// runs a quad per thread).  The translation
// performs the same fp32 operations in the same order as the interpreter (srx_sasl_exec.h), with
// the same numerics flags, so both give identical results.  Modules are cached per program,
// attribute count, sample count and device.
#include <hip/hiprtc.h>

#include <map>
#include <memory>
#include <mutex>
#include <sstream>

#include "srx_runtime_internal.h"
#include "srx_jit_sources.gen.h"  // the device headers' text, generated by the build

namespace srx_rt {
namespace {

const char* const kComp = "xyzw";

// Component k of an operand read through its swizzle, in the lane's own pixel.
std::string opnd_comp(uint8_t o, uint8_t swz, int k) {
  const int c = (swz >> (2 * k)) & 3;
  std::ostringstream s;
  if (o >= SASL_CONST) s << "K[" << (o - SASL_CONST) << "]." << kComp[c];
  else s << "R[" << int(o) << "]." << kComp[c];
  return s.str();
}

// The translated kernel runs one pixel per lane, a 2x2 quad in 4 consecutive lanes (pixel index =
// lane & 3, as in the reference's package): every lane of a quad takes the same path (the
// execution masks are the quad's), ddx/ddy read the neighbour pixel's value by a lane shuffle
// within the quad, and the masks of conditions are gathered from the four lanes.
std::string translate(const sasl_program& p, int NA, int S) {
  std::ostringstream o;
  o << "typedef __hip_internal::uint8_t uint8_t;\n"
       "typedef __hip_internal::uint16_t uint16_t;\n"
       "typedef __hip_internal::int32_t int32_t;\n"
       "typedef __hip_internal::uint32_t uint32_t;\n"
       "typedef __hip_internal::int64_t int64_t;\n"
       "typedef __hip_internal::uint64_t uint64_t;\n"
       "#include \"srx_sasl_exec.h\"\n"
       "namespace srx { __constant__ float c_ewa[256]; }\n"
       "using namespace srx;\n"
       "__device__ __forceinline__ float4 jit_tex(const draw_params& P, const ps_samplers* __restrict__ SM, int slot, float u,\n"
       "    float v, float dxu, float dxv, float dyu, float dyv) {\n"
       "  if (!P.has_sampler[slot]) return make_float4(0.0f, 0.0f, 0.0f, 0.0f);\n"
       "  const sampler_desc_dev& sp = SM->s[slot];\n"
       "  return sample_grad(sp, u, v, dxu, dxv, dyu, dyv);\n"
       "}\n"
       "// the quad's mask of lanes whose bit b is set\n"
       "__device__ __forceinline__ uint32_t quad_bits(uint32_t b) {\n"
       "  b |= static_cast<uint32_t>(__shfl_xor(static_cast<int>(b), 1, 4));\n"
       "  b |= static_cast<uint32_t>(__shfl_xor(static_cast<int>(b), 2, 4));\n"
       "  return b;\n"
       "}\n";
  const int NR = std::max<int>(1, static_cast<int>(p.nregs));
  o << "extern \"C\" __global__ void __launch_bounds__(256) sasl_jit_shade(draw_params P, const ps_samplers* __restrict__ SM,\n"
       "    const float4* __restrict__ tri_attr, const uint32_t* __restrict__ vis) {\n"
       "  constexpr int NA = "
    << NA << ", S = " << S << ";\n"
    << "  (void)S;\n"
    << "  // (quad, winning triangle) items of this 16x16 tile: at most 4 * S distinct winners per quad\n"
       "  __shared__ uint2 items[64 * 4 * S];\n"
       "  __shared__ uint32_t wins[256 * S];\n"
       "  __shared__ uint32_t nitems;\n"
       "  if (threadIdx.x == 0) nitems = 0u;\n"
       "  __syncthreads();\n"
       "  const int pi = threadIdx.x & 3;\n"
       "  const int tw = static_cast<int>(P.target_w), th = static_cast<int>(P.target_h);\n"
       "  {  // phase A: each quad lists its distinct winners (the first pending one of its lowest pixel first)\n"
       "    const int qd = threadIdx.x >> 2;\n"
       "    const int px0 = blockIdx.x * 16 + (qd & 7) * 2, py0 = blockIdx.y * 16 + (qd >> 3) * 2;\n"
       "    const int x = px0 + (pi & 1), y = py0 + (pi >> 1);\n"
       "    const bool in = px0 < tw && py0 < th && x < tw && y < th;\n"
       "    const size_t vbase = (static_cast<size_t>(y) * tw + x) * S;\n";
  for (int k = 0; k < S; ++k)
    o << "    uint32_t w" << k << " = in ? vis[vbase + " << k << "] : NO_WINNER;\n    wins[threadIdx.x * S + " << k << "] = w" << k
      << ";\n";
  o << "    for (;;) {\n"
       "      uint32_t mine = NO_WINNER;\n";
  for (int k = 0; k < S; ++k) o << "      if (mine == NO_WINNER) mine = w" << k << ";\n";
  o << "      const uint32_t c0 = static_cast<uint32_t>(__shfl(static_cast<int>(mine), 0, 4));\n"
       "      const uint32_t c1 = static_cast<uint32_t>(__shfl(static_cast<int>(mine), 1, 4));\n"
       "      const uint32_t c2 = static_cast<uint32_t>(__shfl(static_cast<int>(mine), 2, 4));\n"
       "      const uint32_t c3 = static_cast<uint32_t>(__shfl(static_cast<int>(mine), 3, 4));\n"
       "      const uint32_t cur = c0 != NO_WINNER ? c0 : c1 != NO_WINNER ? c1 : c2 != NO_WINNER ? c2 : c3;\n"
       "      if (cur >= 3u * P.prim_count) break;\n"
       "      if (pi == 0) items[atomicAdd(&nitems, 1u)] = make_uint2(static_cast<uint32_t>(qd), cur);\n";
  for (int k = 0; k < S; ++k) o << "      if (w" << k << " == cur) w" << k << " = NO_WINNER;\n";
  o << "    }\n"
       "  }\n"
       "  __syncthreads();\n"
       "  const uint32_t n_items = nitems;\n"
       "  const float4* __restrict__ K = reinterpret_cast<const float4*>(P.sasl->consts);\n"
       "  // phase B: each 4-lane group shades the next item (the program runs on the item's whole quad)\n"
       "  for (uint32_t it = threadIdx.x >> 2; it < n_items; it += 64u) {\n"
       "    const uint2 item = items[it];\n"
       "    const int qd = static_cast<int>(item.x);\n"
       "    const uint32_t cur = item.y;\n"
       "    const int px0 = blockIdx.x * 16 + (qd & 7) * 2, py0 = blockIdx.y * 16 + (qd >> 3) * 2;\n"
       "    const int x = px0 + (pi & 1), y = py0 + (pi >> 1);\n";
  for (int k = 0; k < S; ++k) o << "    const uint32_t w" << k << " = wins[(qd * 4 + pi) * S + " << k << "];\n";
  o << "    attr_setup<NA> at;\n"
       "    load_attr<NA>(P, tri_attr, cur, at);\n"
       "    const quad_lazy<NA> q(at, P, px0, py0);\n"
       "    float4 R["
    << NR << "];\n";
  for (int r = 0; r < NR; ++r) o << "    R[" << r << "] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);\n";
  o << "    { const float iw = q.inv_w(pi);\n";
  for (uint32_t k = 0; k < p.ninputs; ++k) {
    const sasl_input& in = p.inputs[k];
    o << "      { const float4 v = q.reg(" << (in.attr + 1) << ", pi, iw); R[" << int(in.reg) << "] = make_float4(v.x, "
      << (in.ncomp > 1 ? "v.y" : "0.0f") << ", " << (in.ncomp > 2 ? "v.z" : "0.0f") << ", " << (in.ncomp > 3 ? "v.w" : "0.0f")
      << "); }\n";
  }
  o << "    }\n";
  o << "    uint32_t exec = 15u, steps = 0u;\n";
  for (int d = 0; d < SASL_MAX_DEPTH; ++d)
    o << "    uint32_t fs" << d << " = 0u, fc" << d << " = 0u, fm" << d << " = 0u, fb" << d << " = 0u;\n";

  // the if/loop frames open before each instruction
  std::vector<std::pair<bool, int>> stack;  // (is loop, depth index)
  auto innermost_loop = [&](size_t below) -> std::string {
    for (size_t i = below; i-- > 0;)
      if (stack[i].first) return "fb" + std::to_string(stack[i].second);
    return "0u";
  };
  auto cond = [&](const sasl_inst& in) {
    return "quad_bits((" + opnd_comp(in.a, in.sa, 0) + " != 0.0f) ? (1u << pi) : 0u)";
  };
  for (uint32_t i = 0; i < p.ninst; ++i) {
    const sasl_inst& in = p.code[i];
    o << "  L" << i << ": {\n";
    const int top = stack.empty() ? -1 : stack.back().second;
    switch (in.op) {
    case SOP_IF: {
      const int d = static_cast<int>(stack.size());
      o << "    const uint32_t c = " << cond(in) << ";\n    fs" << d << " = exec; fc" << d << " = c; exec &= c;\n"
        << "    if (!exec) goto L" << in.target << ";\n";
      stack.push_back({false, d});
      break;
    }
    case SOP_ELSE:
      o << "    fs" << top << " &= ~" << innermost_loop(stack.size() - 1) << "; exec = fs" << top << " & ~fc" << top
        << " & 15u;\n    if (!exec) goto L" << in.target << ";\n";
      break;
    case SOP_ENDIF:
      stack.pop_back();
      o << "    exec = fs" << top << " & ~" << innermost_loop(stack.size()) << " & 15u;\n";
      break;
    case SOP_LOOP: {
      const int d = static_cast<int>(stack.size());
      o << "    fs" << d << " = exec; fm" << d << " = exec; fb" << d << " = 0u;\n";
      stack.push_back({true, d});
      break;
    }
    case SOP_LTEST:
      o << "    exec = fm" << top << " & " << (in.imm ? std::string("15u") : "(" + cond(in) + ")") << "; fb" << top
        << " = 0u;\n    if (!exec) goto L" << in.target << ";\n";
      break;
    case SOP_DTEST:
      o << "    exec = fm" << top << " & (" << cond(in) << "); fb" << top << " = 0u; fm" << top << " = exec;\n"
        << "    if (exec) { if (++steps > " << SASL_STEP_LIMIT << "u) goto Lend; goto L" << in.target << "; }\n";
      break;
    case SOP_DBODY: o << "    exec = fm" << top << ";\n"; break;
    case SOP_LSAVE: o << "    fm" << top << " = exec;\n"; break;
    case SOP_JMP: o << "    if (++steps > " << SASL_STEP_LIMIT << "u) goto Lend;\n    goto L" << in.target << ";\n"; break;
    case SOP_LEND:
      stack.pop_back();
      o << "    exec = fs" << top << ";\n";
      break;
    case SOP_BREAK: o << "    " << innermost_loop(stack.size()) << " |= exec; exec = 0u;\n"; break;
    case SOP_NOP: break;
    default: {
      // every component of the result first, then the (masked) write
      const bool masked = (in.wmask & SASL_WM_MASKED) != 0;
      if (in.op == SOP_TEX)  // tex2Dgrad_ps samples the executing pixels only
        o << "    float4 tq = make_float4(0.0f, 0.0f, 0.0f, 0.0f);\n    if ((exec >> pi) & 1u) tq = jit_tex(P, SM, "
          << int(in.imm) << ", " << opnd_comp(in.a, in.sa, 0) << ", " << opnd_comp(in.a, in.sa, 1) << ", "
          << opnd_comp(in.b, in.sb, 0) << ", " << opnd_comp(in.b, in.sb, 1) << ", " << opnd_comp(in.c, in.sc, 0) << ", "
          << opnd_comp(in.c, in.sc, 1) << ");\n";
      for (int k = 0; k < 4; ++k) {
        if (!((in.wmask >> k) & 1)) continue;
        const std::string a = opnd_comp(in.a, in.sa, k), b = opnd_comp(in.b, in.sb, k);
        std::string e;
        switch (in.op) {
        case SOP_MOV: e = a; break;
        case SOP_ADD: e = "(" + a + " + " + b + ")"; break;
        case SOP_SUB: e = "(" + a + " - " + b + ")"; break;
        case SOP_MUL: e = "(" + a + " * " + b + ")"; break;
        case SOP_DIV: e = "(" + a + " / " + b + ")"; break;
        case SOP_NEG: e = "(-" + a + ")"; break;
        case SOP_SLT: e = "(" + a + " < " + b + " ? " + a + " : " + b + ")"; break;
        case SOP_SGT: e = "(" + a + " > " + b + " ? " + a + " : " + b + ")"; break;
        case SOP_SGE: e = "(" + a + " >= " + b + " ? " + a + " : " + b + ")"; break;
        case SOP_SLE: e = "(" + a + " <= " + b + " ? " + a + " : " + b + ")"; break;
        case SOP_CLT: e = "(" + a + " < " + b + " ? 1.0f : 0.0f)"; break;
        case SOP_CGT: e = "(" + a + " > " + b + " ? 1.0f : 0.0f)"; break;
        case SOP_CLE: e = "(" + a + " <= " + b + " ? 1.0f : 0.0f)"; break;
        case SOP_CGE: e = "(" + a + " >= " + b + " ? 1.0f : 0.0f)"; break;
        case SOP_CEQ: e = "(" + a + " == " + b + " ? 1.0f : 0.0f)"; break;
        case SOP_CNE: e = "(" + a + " != " + b + " ? 1.0f : 0.0f)"; break;
        case SOP_ABS: e = "fabsf(" + a + ")"; break;
        case SOP_SQRT: e = "sqrtf(" + a + ")"; break;
        case SOP_FN1: e = "sasl_fn1(" + std::to_string(in.imm) + ", " + a + ")"; break;
        case SOP_FN2: e = "sasl_fn2(" + std::to_string(in.imm) + ", " + a + ", " + b + ")"; break;
        case SOP_DOT:
          e = "0.0f";
          for (int j = 0; j < in.imm; ++j) e = "(" + e + " + (" + opnd_comp(in.a, in.sa, j) + " * " + opnd_comp(in.b, in.sb, j) + "))";
          break;
        case SOP_CROSS:
          if (k == 3) {
            e = "0.0f";
          } else {
            const int j1 = (k + 1) % 3, j2 = (k + 2) % 3;
            e = "((" + opnd_comp(in.a, in.sa, j1) + " * " + opnd_comp(in.b, in.sb, j2) + ") - (" + opnd_comp(in.a, in.sa, j2) +
                " * " + opnd_comp(in.b, in.sb, j1) + "))";
          }
          break;
        case SOP_DDX:  // p1 - p0 for the top row, p3 - p2 for the bottom: the partner is lane ^ 1
        case SOP_DDY:  // p2 - p0, p3 - p1 per column: the partner is lane ^ 2
        {
          const int m = in.op == SOP_DDX ? 1 : 2;
          o << "    const float v" << k << " = " << a << ", n" << k << " = __shfl_xor(v" << k << ", " << m << ", 4);\n";
          e = "((pi & " + std::to_string(m) + ") ? (v" + std::to_string(k) + " - n" + std::to_string(k) + ") : (n" +
              std::to_string(k) + " - v" + std::to_string(k) + "))";
          break;
        }
        case SOP_TEX: e = std::string("tq.") + kComp[k]; break;
        default: e = "0.0f"; break;
        }
        o << "    const float t" << k << " = " << e << ";\n";
      }
      o << (masked ? "    if ((exec >> pi) & 1u) {" : "    {");
      for (int k = 0; k < 4; ++k)
        if ((in.wmask >> k) & 1) o << " R[" << int(in.dst) << "]." << kComp[k] << " = t" << k << ";";
      o << " }\n";
      break;
    }
    }
    o << "  }\n";
  }
  o << "  Lend:;\n";
  // colour target 0 of this lane's pixel to the samples the triangle won
  int c0 = -1;
  for (uint32_t k = 0; k < p.noutputs; ++k)
    if (p.outputs[k].target == 0) c0 = static_cast<int>(k);
  if (c0 < 0) {
    o << "    const float4 c = make_float4(0.0f, 0.0f, 0.0f, 0.0f);\n";
  } else {
    const sasl_output& so = p.outputs[c0];
    o << "    const float4 v = R[" << int(so.reg) << "];\n"
      << "    const float4 c = make_float4(v.x, " << (so.ncomp > 1 ? "v.y" : "0.0f") << ", " << (so.ncomp > 2 ? "v.z" : "0.0f")
      << ", " << (so.ncomp > 3 ? "v.w" : "0.0f") << ");\n";
  }
  for (int k = 0; k < S; ++k)
    o << "    if (w" << k << " == cur) store_texel(P.color.pf, sample_addr(P.color, x, y, " << k << "), c);\n";
  o << "  }\n}\n";
  return o.str();
}

struct jit_entry {
  hipModule_t mod = nullptr;
  hipFunction_t fn = nullptr;
  bool failed = false;
};

std::mutex g_jit_mu;
std::map<std::string, jit_entry> g_jit;

std::string jit_key(const sasl_program& p, int NA, int S, int device) {
  sasl_program k = p;
  std::memset(k.consts, 0, sizeof k.consts);  // constants are read at run time
  std::string s(reinterpret_cast<const char*>(&k), sizeof k);
  s += static_cast<char>(NA);
  s += static_cast<char>(S);
  s.append(reinterpret_cast<const char*>(&device), sizeof device);
  return s;
}

int32_t compile_module(const std::string& src, jit_entry& e) {
  hiprtcProgram prog;
  if (hiprtcCreateProgram(&prog, src.c_str(), "sasl_jit.hip", kJitHeaderCount, kJitHeaderText, kJitHeaderName) != HIPRTC_SUCCESS)
    return fail(SRX_FAILED, "hiprtcCreateProgram");
  const char* opts[] = {"--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off", "-fno-fast-math",
                        "-fno-gpu-flush-denormals-to-zero", "-fhip-fp32-correctly-rounded-divide-sqrt",
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"};
  const hiprtcResult r = hiprtcCompileProgram(prog, static_cast<int>(sizeof opts / sizeof opts[0]), opts);
  if (r != HIPRTC_SUCCESS) {
    size_t n = 0;
    hiprtcGetProgramLogSize(prog, &n);
    std::string log(n, '\0');
    if (n) hiprtcGetProgramLog(prog, &log[0]);
    hiprtcDestroyProgram(&prog);
    return fail(SRX_FAILED, ("SASL shader compilation: " + log.substr(0, 2000)).c_str());
  }
  size_t n = 0;
  hiprtcGetCodeSize(prog, &n);
  std::vector<char> code(n);
  hiprtcGetCode(prog, code.data());
  hiprtcDestroyProgram(&prog);
  HIPCHK(hipModuleLoadData(&e.mod, code.data()));
  HIPCHK(hipModuleGetFunction(&e.fn, e.mod, "sasl_jit_shade"));
  hipDeviceptr_t ewa = nullptr;
  size_t bytes = 0;
  HIPCHK(hipModuleGetGlobal(&ewa, &bytes, e.mod, "_ZN3srx5c_ewaE"));
  float t[256];
  make_ewa(t);
  HIPCHK(hipMemcpyHtoD(ewa, t, sizeof t));
  return SRX_OK;
}

}  // namespace

std::string sasl_jit_source(const sasl_program& p, int NA, int S) { return translate(p, NA, S); }

bool sasl_jit_enabled() {
  const char* v = std::getenv("SRX_SASL_JIT");
  return !(v && v[0] == '0');
}

int32_t sasl_jit_launch(const sasl_program& prog, const draw_params& P, const draw_buffers& B, int device, hipStream_t s,
                        bool allow_compile, bool* launched) {
  *launched = false;
  if (!sasl_jit_enabled()) return SRX_OK;
  const int NA = std::max(1, std::min(P.nattr, MAX_ATTRS));
  const int S = P.samples;
  jit_entry* e;
  {
    std::lock_guard<std::mutex> lk(g_jit_mu);
    const std::string key = jit_key(prog, NA, S, device);
    auto it = g_jit.find(key);
    if (it == g_jit.end() && !allow_compile) return SRX_OK;  // compiling allocates: the interpreter shades
    e = &g_jit[key];
    if (!e->fn && !e->failed) {
      // the module compiles while the stream's earlier work proceeds
      if (compile_module(translate(prog, NA, S), *e) != SRX_OK) e->failed = true;
    }
    if (e->failed) return SRX_OK;  // the interpreter kernel shades instead
  }
  draw_params Pk = P;
  const ps_samplers* sm = B.samplers;
  const float4* ta = B.tri_attr;
  const uint32_t* vis = B.vis;
  void* args[] = {&Pk, &sm, &ta, &vis};
  HIPCHK(hipModuleLaunchKernel(e->fn, static_cast<unsigned>(P.gtiles_x), static_cast<unsigned>(P.gtiles_y), 1, 256, 1, 1, 0, s,
                               args, nullptr));
  *launched = true;
  return SRX_OK;
}

}  // namespace srx_rt
