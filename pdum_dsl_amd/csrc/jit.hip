// Runtime specialization of elementwise programs with hipRTC.
//
// The interpreter (ew.h) runs any program but pays a decode and a
// VGPR-indexed register access per instruction. Here a program is turned
// into a straight-line evaluator (one C++ statement per instruction,
// registers as named floats, constants and opcodes baked in, strides still
// read from the program at run time), spliced into the same kernel bodies
// (contract_core.h) and compiled by hipRTC for gfx950 with the library's own
// flags. Compiled modules are cached per (device, generated source) for the
// life of the process; a failed compile is remembered and the caller uses
// the interpreter kernels instead.
#include <hip/hiprtc.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "common.h"
#include "contract_core.h"
#include "contract_host.h"
#include "jit.h"
#include "jit_sources.h"  // generated by the build: the text of dev.h, ew.h, contract_core.h, pdhip.h

namespace pdh {
namespace {

std::atomic<int> g_mode{-1};  // -1: not read yet
std::atomic<int64_t> g_compiled{0}, g_launched{0}, g_failed{0};

struct Entry {
  hipModule_t mod = nullptr;
  hipFunction_t fn[kJitFns] = {};
  bool ok = false;
};
std::mutex g_mu;
std::unordered_map<std::string, Entry> g_cache;

// The entry of each request under a short key of exactly what the generated
// source depends on, so that a launch does not generate the source again to
// look it up (6 us a call). A source has few keys, and entries stay put in
// the map above. Guarded by g_mu.
std::unordered_map<std::string, const Entry*> g_by_request;

template <typename T>
void key_add(std::string& k, const T& v) {
  k.append(reinterpret_cast<const char*>(&v), sizeof(T));
}

// What gen_eval reads of a program: its instructions, and which views are
// contiguous along the last dim.
void key_program(std::string& k, const pdh_ew_program& p) {
  key_add(k, p.n_insns);
  key_add(k, p.ndim);
  key_add(k, p.out_reg);
  uint32_t contiguous = p.out_stride[p.ndim - 1] == 1 ? 1u : 0u;
  for (int i = 0; i < PDH_EW_MAX_OPERANDS; ++i) contiguous |= p.in_stride[i][p.ndim - 1] == 1 ? 2u << i : 0u;
  key_add(k, contiguous);
  for (int i = 0; i < p.n_insns; ++i) {
    const pdh_ew_insn& in = p.insns[i];
    const uint8_t b[5] = {in.op, in.dst, in.a, in.b, in.c};
    key_add(k, b);
    key_add(k, in.imm);
  }
}

std::string request_key(char what, int dev, int dt, int lay, int red, int f32_mode) {
  std::string k;
  k.reserve(256);
  k.push_back(what);
  for (const int v : {dev, dt, lay, red, f32_mode}) key_add(k, v);
  return k;
}

// The entry of request `key` into fns; false when there is none (or the interpreter runs it). known: whether there is one.
bool find_request(const std::string& key, hipFunction_t fns[kJitFns], bool* known) {
  std::lock_guard<std::mutex> lock(g_mu);
  const auto it = g_by_request.find(key);
  *known = it != g_by_request.end();
  if (!*known || !it->second->ok) return false;
  for (int i = 0; i < kJitFns; ++i) fns[i] = it->second->fn[i];
  return true;
}

const char* dt_name(int dt) { return dt == PDH_F32 ? "PDH_F32" : dt == PDH_BF16 ? "PDH_BF16" : "PDH_F16"; }

std::string fmt_float(float v) {
  char buf[64];
  std::snprintf(buf, sizeof(buf), "%af", static_cast<double>(v));  // hex float: exact
  if (v != v) return "__builtin_nanf(\"\")";
  if (v == __builtin_inff()) return "__builtin_inff()";
  if (v == -__builtin_inff()) return "(-__builtin_inff())";
  return buf;
}

// The generated evaluator: the Eval policy of contract_core.h.
std::string gen_eval(const pdh_ew_program& p, int dt, const char* name = "GenEval") {
  const int nd = p.ndim;
  std::string s;
  // fp32 with every read operand and the output contiguous along the last
  // dim: each operand's EPT = 4 values in one 16-byte load when es == 1
  bool vec = dt == PDH_F32 && p.out_stride[nd - 1] == 1;
  for (int i = 0; i < p.n_insns; ++i)
    if (p.insns[i].op == PDH_EW_LOAD && p.in_stride[p.insns[i].a][nd - 1] != 1) vec = false;
  s += std::string("namespace pdh {\nstruct ") + name + " {\n  static constexpr bool kVec = " +
       (vec ? "true" : "false") + ";\n  static constexpr int kStoreRun = 16;\n  template <int EPT>\n";
  s += "  static __device__ __forceinline__ void run(const pdh_ew_program& p, const EwOperands& ops, int,\n";
  s += "      const int (&c0)[PDH_EW_MAX_DIMS], const float (&acc)[EPT], float (&res)[EPT], int es) {\n";
  s += "    (void)p; (void)ops; (void)acc; (void)c0; (void)es;\n";
  bool used[PDH_EW_MAX_OPERANDS] = {};
  for (int i = 0; i < p.n_insns; ++i)
    if (p.insns[i].op == PDH_EW_LOAD) used[p.insns[i].a] = true;
  for (int k = 0; k < PDH_EW_MAX_OPERANDS; ++k) {
    if (!used[k]) continue;
    s += "    const int off" + std::to_string(k) + " = 0";
    for (int d = 0; d < nd; ++d)
      s += " + c0[" + std::to_string(d) + "] * static_cast<int>(p.in_stride[" + std::to_string(k) + "][" +
           std::to_string(d) + "])";
    s += ";\n    const int st" + std::to_string(k) + " = es * static_cast<int>(p.in_stride[" + std::to_string(k) +
         "][" + std::to_string(nd - 1) + "]);\n";
    const std::string K = std::to_string(k);
    s += "    float v" + K + "[EPT];\n";
    const bool vec16 = dt != PDH_F32 && p.in_stride[k][nd - 1] == 1;
    if (vec16) {  // runs of four 16-bit values in one 8-byte load each where this lane's run is 8-byte aligned
      const std::string cv = dt == PDH_BF16 ? "bf16_to_f32" : "f16_to_f32";
      s += "    if constexpr (EPT % 4 == 0) {\n      const uint16_t* h" + K + " = static_cast<const uint16_t*>(ops.p[" + K +
           "]) + off" + K + ";\n      if (es == 1 && (reinterpret_cast<uintptr_t>(h" + K +
           ") & 7) == 0) {\n#pragma unroll\n        for (int q = 0; q < EPT / 4; ++q) {\n          const u32x2 t" + K +
           " = *reinterpret_cast<const u32x2*>(h" + K + " + 4 * q);\n          v" + K + "[4 * q] = " + cv +
           "(static_cast<uint16_t>(t" + K + "[0])); v" + K + "[4 * q + 1] = " + cv + "(static_cast<uint16_t>(t" + K +
           "[0] >> 16)); v" + K + "[4 * q + 2] = " + cv + "(static_cast<uint16_t>(t" + K + "[1])); v" + K +
           "[4 * q + 3] = " + cv + "(static_cast<uint16_t>(t" + K + "[1] >> 16));\n        }\n      } else {\n"
           "#pragma unroll\n        for (int e = 0; e < EPT; ++e) v" + K + "[e] = ld_dt<" + dt_name(dt) + ">(ops.p[" +
           K + "], off" + K + " + e * st" + K + ");\n      }\n    } else {\n";
    }
    if (vec)
      s += "    if constexpr (EPT % 4 == 0) {\n      if (es == 1) {\n#pragma unroll\n        for (int q = 0; q < EPT / 4; ++q) {\n"
           "          const f32x4u t" + K + " = *reinterpret_cast<const f32x4u*>(static_cast<const float*>(ops.p[" + K +
           "]) + off" + K + " + 4 * q);\n          v" + K + "[4 * q] = t" + K + "[0]; v" + K + "[4 * q + 1] = t" + K +
           "[1]; v" + K + "[4 * q + 2] = t" + K + "[2]; v" + K + "[4 * q + 3] = t" + K +
           "[3];\n        }\n      } else {\n#pragma unroll\n        for (int e = 0; e < EPT; ++e) v" + K +
           "[e] = ld_dt<PDH_F32>(ops.p[" + K + "], off" + K + " + e * st" + K + ");\n      }\n    } else {\n";
    s += "#pragma unroll\n    for (int e = 0; e < EPT; ++e) v" + K + "[e] = ld_dt<" + dt_name(dt) + ">(ops.p[" + K +
         "], off" + K + " + e * st" + K + ");\n";
    if (vec || vec16) s += "    }\n";
  }
  s += "#pragma unroll\n    for (int e = 0; e < EPT; ++e) {\n      float ";
  for (int r = 0; r < PDH_EW_MAX_REGS; ++r) s += "r" + std::to_string(r) + (r + 1 < PDH_EW_MAX_REGS ? " = 0.f, " : " = 0.f;\n");
  auto R = [](int r) { return "r" + std::to_string(r); };
  for (int i = 0; i < p.n_insns; ++i) {
    const pdh_ew_insn& in = p.insns[i];
    const std::string d = R(in.dst), a = R(in.a), b = R(in.b), c = R(in.c);
    std::string rhs;
    switch (in.op) {
      case PDH_EW_LOAD: {
        const std::string k = std::to_string(in.a);
        rhs = "v" + k + "[e]";
        break;
      }
      case PDH_EW_ACC: rhs = "acc[e]"; break;
      case PDH_EW_CONST: rhs = fmt_float(in.imm); break;
      case PDH_EW_IOTA:
        rhs = "static_cast<float>(c0[" + std::to_string(in.a) + "] + static_cast<int>(p.start[" + std::to_string(in.a) +
              "])" + (in.a == nd - 1 ? " + e * es" : "") + ")";
        break;
      case PDH_EW_NEG: rhs = "-" + a; break;
      case PDH_EW_EXP: rhs = "expf(" + a + ")"; break;
      case PDH_EW_LOG: rhs = "logf(" + a + ")"; break;
      case PDH_EW_SQRT: rhs = "sqrtf(" + a + ")"; break;
      case PDH_EW_TANH: rhs = "pdh_tanh(" + a + ")"; break;
      case PDH_EW_SIN: rhs = "sinf(" + a + ")"; break;
      case PDH_EW_COS: rhs = "cosf(" + a + ")"; break;
      case PDH_EW_ABS: rhs = "fabsf(" + a + ")"; break;
      case PDH_EW_FLOOR: rhs = "floorf(" + a + ")"; break;
      case PDH_EW_RBF16: rhs = "bf16_to_f32(f32_to_bf16(" + a + "))"; break;
      case PDH_EW_RF16: rhs = "f16_to_f32(f32_to_f16(" + a + "))"; break;
      case PDH_EW_ADD: rhs = a + " + " + b; break;
      case PDH_EW_SUB: rhs = a + " - " + b; break;
      case PDH_EW_MUL: rhs = a + " * " + b; break;
      case PDH_EW_DIV: rhs = a + " / " + b; break;
      case PDH_EW_MAX: rhs = "pdh::nan_max(" + a + ", " + b + ")"; break;
      case PDH_EW_MIN: rhs = "pdh::nan_min(" + a + ", " + b + ")"; break;
      case PDH_EW_EQ: rhs = "(" + a + " == " + b + " ? 1.f : 0.f)"; break;
      case PDH_EW_NE: rhs = "(" + a + " != " + b + " ? 1.f : 0.f)"; break;
      case PDH_EW_LT: rhs = "(" + a + " < " + b + " ? 1.f : 0.f)"; break;
      case PDH_EW_LE: rhs = "(" + a + " <= " + b + " ? 1.f : 0.f)"; break;
      case PDH_EW_GT: rhs = "(" + a + " > " + b + " ? 1.f : 0.f)"; break;
      case PDH_EW_GE: rhs = "(" + a + " >= " + b + " ? 1.f : 0.f)"; break;
      default: rhs = "(" + a + " != 0.f ? " + b + " : " + c + ")"; break;  // PDH_EW_WHERE
    }
    s += "      " + d + " = " + rhs + ";\n";
  }
  s += "      res[e] = " + R(p.out_reg) + ";\n    }\n  }\n};\n}  // namespace pdh\n";
  return s;
}

std::string kernels_src(JitKind kind, int dt, int lay, int red, int f32_mode) {
  const std::string D = dt_name(dt);
  if (kind == JitKind::MapChain)
    return "extern \"C\" __global__ __launch_bounds__(256) void pdh_jit_k0(pdh_ew_program p, pdh::EwOperands ops, "
           "void* out, uint32_t total) { pdh::map_chain_body<" + D + ", 4, pdh::GenEval>(p, ops, out, total); }\n"
           "extern \"C\" __global__ __launch_bounds__(256) void pdh_jit_k1(pdh_ew_program p, pdh::EwOperands ops, "
           "void* out, uint32_t total) { pdh::map_chain_body<" + D + ", 1, pdh::GenEval>(p, ops, out, total); }\n";
  if (dt == PDH_F32 && f32_mode == 0)
    return "extern \"C\" __global__ __launch_bounds__(256) void pdh_jit_k0(pdh::ContractArgs a, pdh_ew_program p, "
           "pdh::EwOperands ops) { pdh::contract_f32_body<pdh::GenEval, " + std::to_string(red) + ">(a, p, ops); }\n";
  if (dt == PDH_F32) {
    const std::string ns = std::to_string(f32_mode), nl = ns + ", " + std::to_string(lay);
    const std::string rd = ", " + std::to_string(red);
    return "extern \"C\" __global__ __launch_bounds__(256, 2) void pdh_jit_k0(pdh::ContractArgs a, pdh_ew_program p, "
           "pdh::EwOperands ops) { __shared__ __attribute__((aligned(1024))) unsigned char "
           "smem[pdh::split_lds<64, " + ns + ">()]; pdh::contract_split_body<PDH_F32, 64, " + nl +
           ", pdh::GenEval" + rd + ">(a, p, ops, smem); }\n"
           "extern \"C\" __global__ __launch_bounds__(256, 2) void pdh_jit_k1(pdh::ContractArgs a, pdh_ew_program p, "
           "pdh::EwOperands ops) { __shared__ __attribute__((aligned(1024))) unsigned char "
           "smem[pdh::split_lds<32, " + ns + ">()]; pdh::contract_split_body<PDH_F32, 32, " + nl +
           ", pdh::GenEval" + rd + ">(a, p, ops, smem); }\n";
  }
  // 16-bit: 128 x 128 tiles, 64 x 64 tiles, the finish of a k split
  const std::string args = "(pdh::ContractArgs a, pdh_ew_program p, pdh::EwOperands ops";
  auto tile = [&](const char* name, const std::string& wm) {
    return std::string("extern \"C\" __global__ __launch_bounds__(256, 2) void ") + name + args +
           ") { __shared__ __attribute__((aligned(1024))) unsigned char smem[pdh::contract_lds<" + wm +
           ">()]; pdh::contract_mfma_body<" + D + ", " + wm + ", pdh::GenEval" +
           (lay != 0 ? ", " + std::to_string(lay) : "") + ">(a, p, ops, smem); }\n";
  };
  return tile("pdh_jit_k0", "64") + tile("pdh_jit_k1", "32") +
         "extern \"C\" __global__ __launch_bounds__(256) void pdh_jit_k2" + args + ", const float* ws) { "
         "pdh::contract_finish_body<" + D + ", pdh::GenEval>(a, p, ops, ws); }\n";
}

// Kernels in a contraction's module.
int contract_kernels(JitKind kind, int dt, int f32_mode) {
  return kind == JitKind::MapChain ? 2 : (dt != PDH_F32 ? 3 : (f32_mode != 0 ? 2 : 1));
}

bool compile_code(const std::string& src, std::vector<char>* code, std::string* err) {
  const char* hdrs[] = {kJitSrcDevH, kJitSrcEwH, kJitSrcCoreH, kJitSrcPdhipH};
  const char* names[] = {"dev.h", "ew.h", "contract_core.h", "pdhip.h"};
  hiprtcProgram prog;
  if (hiprtcCreateProgram(&prog, src.c_str(), "pdh_jit.hip", 4, hdrs, names) != HIPRTC_SUCCESS) {
    *err = "hiprtcCreateProgram failed";
    return false;
  }
  // the library's own code-generation flags (packed fp32 arithmetic off)
  const char* opts[] = {"--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops"};
  const hiprtcResult rc = hiprtcCompileProgram(prog, 7, opts);
  if (rc != HIPRTC_SUCCESS) {
    size_t n = 0;
    hiprtcGetProgramLogSize(prog, &n);
    std::string log(n, '\0');
    if (n) hiprtcGetProgramLog(prog, &log[0]);
    *err = "hipRTC compile failed: " + log.substr(0, 600);
    hiprtcDestroyProgram(&prog);
    return false;
  }
  size_t n = 0;
  hiprtcGetCodeSize(prog, &n);
  code->resize(n);
  hiprtcGetCode(prog, code->data());
  hiprtcDestroyProgram(&prog);
  return true;
}

std::string full_source(JitKind kind, const pdh_ew_program& p, int dt, int lay, int red, int f32_mode) {
  return "#include \"contract_core.h\"\n" + gen_eval(p, dt) + kernels_src(kind, dt, lay, red, f32_mode);
}

std::string reduce_source(const pdh_ew_program& ps, const pdh_ew_program& pe, int dt) {
  const std::string D = dt_name(dt);
  return "#include \"contract_core.h\"\n" + gen_eval(ps, dt, "GenEval") + gen_eval(pe, dt, "GenEvalE") +
         "extern \"C\" __global__ __launch_bounds__(256) void pdh_jit_k0(pdh_ew_program ps, pdh_ew_program pe, "
         "pdh::EwOperands ops, void* out, int nk, int rows, int reducer) { pdh::reduce_rows_body<" + D +
         ", pdh::GenEval, pdh::GenEvalE>(ps, pe, ops, out, nk, rows, reducer); }\n"
         "extern \"C\" __global__ __launch_bounds__(1024) void pdh_jit_k1(pdh_ew_program ps, pdh_ew_program pe, "
         "pdh::EwOperands ops, void* out, int nk, int rows, int reducer) { __shared__ float "
         "part[pdh::kColOut * pdh::kColK]; (void)nk; "
         "pdh::reduce_cols_body<" + D + ", pdh::GenEval, pdh::GenEvalE>(ps, pe, ops, out, rows, reducer, part); }\n";
}

// The fp32 contraction with operand prologues: the epilogue's evaluator, one
// per computed operand (GenProA, GenProB; an absent one is a stub the kernel
// never calls) and the prologue kernels of the fp32 mode.
std::string pro_source(const pdh_ew_program& pe, const pdh_ew_program* pa, const pdh_ew_program* pb, int lay, int dt,
                       int f32_mode) {
  const char* stub = "namespace pdh {\nstruct %s {\n  static constexpr bool kVec = false;\n  static constexpr int "
                     "kStoreRun = 16;\n  template <int EPT>\n  static __device__ __forceinline__ void run(const "
                     "pdh_ew_program&, const EwOperands&, int, const int (&)[PDH_EW_MAX_DIMS], const float (&)[EPT], "
                     "float (&res)[EPT], int) {\n    for (int e = 0; e < EPT; ++e) res[e] = 0.f;\n  }\n};\n}  // "
                     "namespace pdh\n";
  auto stub_of = [&](const char* name) {
    char buf[1024];
    std::snprintf(buf, sizeof(buf), stub, name);
    return std::string(buf);
  };
  std::string s = "#include \"contract_core.h\"\n" + gen_eval(pe, dt) +
                  (pa ? gen_eval(*pa, dt, "GenProA") : stub_of("GenProA")) +
                  (pb ? gen_eval(*pb, dt, "GenProB") : stub_of("GenProB"));
  const std::string args = "(pdh::ContractArgs a, pdh_ew_program p, pdh::EwOperands ops, pdh::ContractPro pa, "
                           "pdh::ContractPro pb)";
  if (dt == PDH_F32 && f32_mode == 0)
    return s + "extern \"C\" __global__ __launch_bounds__(256) void pdh_jit_k0" + args +
           " { pdh::contract_f32_body<pdh::GenEval, -1, pdh::GenProA, pdh::GenProB, true>(a, p, ops, &pa, &pb); }\n";
  // 16-bit storage: one bf16 plane (the operands' values rounded to bf16)
  const int ns = dt == PDH_F32 ? f32_mode : 1;
  const std::string nl = std::to_string(ns) + ", " + std::to_string(lay);
  std::string k;
  for (int small = 0; small < 2; ++small) {
    const std::string wm = small ? "32" : "64";
    k += "extern \"C\" __global__ __launch_bounds__(256, 2) void pdh_jit_k" + std::to_string(small) + args +
         " { __shared__ __attribute__((aligned(1024))) unsigned char smem[pdh::split_lds<" + wm + ", " +
         std::to_string(ns) + ">()]; pdh::contract_split_body<" + dt_name(dt) + ", " + wm + ", " + nl +
         ", pdh::GenEval, -1, pdh::GenProA, pdh::GenProB, true>(a, p, ops, smem, &pa, &pb); }\n";
  }
  return s + k;
}

bool compile(const std::string& src, int count, Entry* out, std::string* err) {
  std::vector<char> code;
  if (!compile_code(src, &code, err)) return false;
  if (hipModuleLoadData(&out->mod, code.data()) != hipSuccess) {
    *err = "hipModuleLoadData failed";
    return false;
  }
  for (int i = 0; i < count; ++i) {
    const std::string name = "pdh_jit_k" + std::to_string(i);
    if (hipModuleGetFunction(&out->fn[i], out->mod, name.c_str()) != hipSuccess) {
      *err = "hipModuleGetFunction failed";
      return false;
    }
  }
  return true;
}

}  // namespace

bool jit_enabled() {
  int m = g_mode.load();
  if (m < 0) {
    const char* env = std::getenv("PDH_JIT");
    m = (env != nullptr && std::strcmp(env, "0") == 0) ? 0 : 1;
    g_mode.store(m);
  }
  return m == 1;
}

namespace {

// The entry of `src` (compiled on its first request) into fns, kept under `key` for the next one.
bool get(const std::string& key, int dev, const std::string& src, int count, hipFunction_t fns[kJitFns]) {
  const std::string skey = std::to_string(dev) + "|" + src;
  std::lock_guard<std::mutex> lock(g_mu);
  auto it = g_cache.find(skey);
  if (it == g_cache.end()) {
    Entry e;
    std::string err;
    e.ok = compile(src, count, &e, &err);
    if (e.ok)
      ++g_compiled;
    else {
      ++g_failed;
      std::fprintf(stderr, "libpdhip: runtime specialization unavailable, the interpreter runs this program (%s)\n",
                   err.c_str());
    }
    it = g_cache.emplace(skey, e).first;
  }
  g_by_request.emplace(key, &it->second);
  if (!it->second.ok) return false;
  for (int i = 0; i < kJitFns; ++i) fns[i] = it->second.fn[i];
  return true;
}

}  // namespace

// The specialized kernels for program p (jit.h), or false when the
// interpreter must run it.
bool jit_get(JitKind kind, const pdh_ew_program& p, int dt, hipFunction_t fns[kJitFns], int lay, int red,
             int f32_mode) {
  if (!jit_enabled()) return false;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  std::string key = request_key(kind == JitKind::MapChain ? 'm' : 'c', dev, dt, lay, red, f32_mode);
  key_program(key, p);
  bool known;
  const bool found = find_request(key, fns, &known);
  return known ? found
               : get(key, dev, full_source(kind, p, dt, lay, red, f32_mode), contract_kernels(kind, dt, f32_mode),
                     fns);
}

// The specialized row-reduce kernels for (summand, epilogue): fns[0] one
// wave per output, fns[1] the column variant; or false.
bool jit_get_reduce(const pdh_ew_program& ps, const pdh_ew_program& pe, int dt, hipFunction_t fns[kJitFns]) {
  if (!jit_enabled()) return false;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  std::string key = request_key('r', dev, dt, 0, 0, 0);
  key_program(key, ps);
  key_program(key, pe);
  bool known;
  const bool found = find_request(key, fns, &known);
  return known ? found : get(key, dev, reduce_source(ps, pe, dt), 2, fns);
}

// The fp32 prologue kernels specialized for (epilogue, prologues): fns[0] the
// 128 x 128-tile kernel (or the VALU one in fp32 mode 0), fns[1] the
// 64 x 64-tile one; or false.
bool jit_get_pro(const pdh_ew_program& pe, const pdh_ew_program* pa, const pdh_ew_program* pb, hipFunction_t fns[kJitFns],
                 int lay, int dt, int f32_mode) {
  if (!jit_enabled()) return false;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  std::string key = request_key('p', dev, dt, lay, (pa != nullptr ? 1 : 0) | (pb != nullptr ? 2 : 0), f32_mode);
  key_program(key, pe);
  if (pa != nullptr) key_program(key, *pa);
  if (pb != nullptr) key_program(key, *pb);
  bool known;
  const bool found = find_request(key, fns, &known);
  return known ? found : get(key, dev, pro_source(pe, pa, pb, lay, dt, f32_mode),
                           dt != PDH_F32 || f32_mode != 0 ? 2 : 1, fns);
}

void jit_count_launch() { ++g_launched; }

}  // namespace pdh

using namespace pdh;

extern "C" int pdh_ew_set_jit(int enable) {
  const int prev = jit_enabled() ? 1 : 0;
  g_mode.store(enable ? 1 : 0);
  return prev;
}

extern "C" void pdh_ew_jit_stats(int64_t* stats3) {
  if (!stats3) return;
  stats3[0] = g_compiled.load();
  stats3[1] = g_launched.load();
  stats3[2] = g_failed.load();
}

extern "C" size_t pdh_ew_jit_source(const pdh_ew_program* prog, int kind, int dtype, char* buf, size_t n) {
  if (!prog || prog->n_insns < 1 || prog->n_insns > PDH_EW_MAX_INSNS || prog->ndim < 1 || prog->ndim > PDH_EW_MAX_DIMS ||
      kind < 0 || kind > 7)
    return 0;
  const std::string src = full_source(kind == 0 ? JitKind::MapChain : JitKind::Contract, *prog, dtype,
                                      kind > 1 && kind < 5 ? kind - 1 : 0, kind >= 5 ? kind - 5 : -1,
                                      f32_contract_mode());
  if (buf && n) {
    const size_t k = src.size() < n - 1 ? src.size() : n - 1;
    std::memcpy(buf, src.data(), k);
    buf[k] = '\0';
  }
  return src.size();
}

extern "C" int pdh_ew_jit_compile(const pdh_ew_program* prog, int kind, int dtype) {
  PDH_REQUIRE(prog && prog->n_insns >= 1 && prog->n_insns <= PDH_EW_MAX_INSNS && prog->ndim >= 1 &&
                  prog->ndim <= PDH_EW_MAX_DIMS && kind >= 0 && kind <= 7,
              PDH_EINVAL, "pdh_ew_jit_compile: malformed program or kind");
  std::vector<char> code;
  std::string err;
  PDH_REQUIRE(compile_code(full_source(kind == 0 ? JitKind::MapChain : JitKind::Contract, *prog, dtype,
                                       kind > 1 && kind < 5 ? kind - 1 : 0, kind >= 5 ? kind - 5 : -1,
                                      f32_contract_mode()),
                           &code, &err),
              PDH_ELAUNCH, "%s", err.c_str());
  return PDH_OK;
}
