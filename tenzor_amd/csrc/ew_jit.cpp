// Generated single-pass chain and reduction kernels (K1 fast path).
//
// The reference fuses an elementwise chain at compile time into one loop
// (codegen.zig:15-205 FusedElementwiseKernel: the ops of the chain applied
// in post-order per element, patterns.zig:43-63).  Here the same happens at
// run time: a chain program (ew_program.h) is turned into straight-line HIP
// source - every leaf loaded up front through its broadcast projection with
// the projection kind baked in, every op inlined with its tag as a
// constant - compiled once per program shape with hipRTC for the device's
// architecture, and cached.  Pointers, shapes, divisors and constant values
// stay run-time kernel arguments (the EwProgram struct itself), so programs
// that differ only in those share one kernel.
//
// The op semantics and the program layout are the exact text the
// interpreter kernels are compiled from (ew_shared.inc, stringified below).
#include "ew_program.h"

#ifndef TZH_EMULATION
#include <hip/hiprtc.h>
#else
#include <dlfcn.h>
#include <unistd.h>

#include <cstdio>
#include <cstdlib>
#endif

#include <cstring>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

namespace tzh_ew {
namespace {

#define TZH_EW_SHARED(...) #__VA_ARGS__
const char kSharedSrc[] =
#include "ew_shared.inc"
    ;
#undef TZH_EW_SHARED

#define TZH_JIT_OPS(X)                                                                                    \
    X(TZH_OP_NEG) X(TZH_OP_ABS) X(TZH_OP_EXP) X(TZH_OP_LOG) X(TZH_OP_SQRT) X(TZH_OP_RSQRT) X(TZH_OP_SIN)   \
    X(TZH_OP_COS) X(TZH_OP_TANH) X(TZH_OP_SIGMOID) X(TZH_OP_RELU) X(TZH_OP_GELU) X(TZH_OP_SILU)           \
    X(TZH_OP_SOFTPLUS) X(TZH_OP_FLOOR) X(TZH_OP_CEIL) X(TZH_OP_ROUND) X(TZH_OP_ADD) X(TZH_OP_SUB)         \
    X(TZH_OP_MUL) X(TZH_OP_DIV) X(TZH_OP_POW) X(TZH_OP_MAX) X(TZH_OP_MIN) X(TZH_OP_SUM) X(TZH_OP_MEAN) X(TZH_OP_PROD)                  \
    X(TZH_OP_REDUCE_MAX) X(TZH_OP_REDUCE_MIN)

std::string prelude() {
    std::string s = "typedef float tzh_f32x4 __attribute__((ext_vector_type(4)));\n"
                    "typedef double tzh_f64x2 __attribute__((ext_vector_type(2)));\n"
                    "enum {";
#define TZH_JIT_ENUM(name) s += std::string(#name) + " = " + std::to_string((int)name) + ", ";
    TZH_JIT_OPS(TZH_JIT_ENUM)
#undef TZH_JIT_ENUM
    s += "};\n";
    s += kSharedSrc;
    s += "\n";
    return s;
}

// Offset expression of leaf j for the flat output index held in `var`.
std::string offset_fn(const EwProgram &p, int j) {
    const EwLeaf &lf = p.leaves[j];
    const std::string L = "p.leaves[" + std::to_string(j) + "]";
    std::string b = "__device__ __forceinline__ long long off" + std::to_string(j) +
                    "(const EwProgram &p, long long flat) {\n";
    if (p.small) {
        b += "    unsigned f = (unsigned)flat;\n";
        if (!lf.general) {
            if (lf.div != 1) b += "    f = fast_div(" + L + ".fdiv, f);\n";
            if (lf.mod <= (long long)0xffffffff) b += "    f = f - fast_div(" + L + ".fmod, f) * " + L + ".fmod.d;\n";
            b += "    return f;\n";
        } else {
            b += "    unsigned off = 0, rem = f, q;\n";
            for (int d = p.ndim - 1; d >= 0; d--) {
                const std::string D = std::to_string(d);
                b += "    q = fast_div(p.fshape[" + D + "], rem);\n";
                if (lf.strides[d] != 0)
                    b += "    off += (rem - q * p.fshape[" + D + "].d) * (unsigned)" + L + ".strides[" + D + "];\n";
                b += "    rem = q;\n";
            }
            b += "    return off;\n";
        }
    } else {
        if (!lf.general) {
            b += "    return (flat / " + L + ".div) % " + L + ".mod;\n";
        } else {
            b += "    long long off = 0, rem = flat;\n";
            for (int d = p.ndim - 1; d >= 0; d--) {
                const std::string D = std::to_string(d);
                if (lf.strides[d] != 0) b += "    off += (rem % p.shape[" + D + "]) * " + L + ".strides[" + D + "];\n";
                b += "    rem /= p.shape[" + D + "];\n";
            }
            b += "    return off;\n";
        }
    }
    b += "}\n";
    return b;
}

// Leaf loads for outputs flat .. flat+W-1 into L<j><sfx>[W].  `flat` is the
// name of the index expression in the generated code.
std::string loads(const EwProgram &p, const char *T, int W, bool vec16, const std::string &sfx,
                  const std::string &flat) {
    std::string b;
    const std::string WS = std::to_string(W);
    for (int j = 0; j < p.n_leaves; j++) {
        const std::string J = std::to_string(j), LJ = "L" + J + sfx;
        const std::string ptr = "((const " + std::string(T) + " *)p.leaves[" + J + "].ptr)";
        b += "        " + std::string(T) + " " + LJ + "[" + WS + "];\n";
        const int mode = W == 1 ? VEC_PER_ELEM : p.leaves[j].vec;
        if (mode == VEC_CONTIG && vec16) {
            const std::string VT = std::string(T) == "float" ? "tzh_f32x4" : "tzh_f64x2";
            b += "        { const " + VT + " raw = *(const " + VT + " *)(" + ptr + " + off" + J + "(p, " + flat + "));\n";
            for (int e = 0; e < W; e++) b += "          " + LJ + "[" + std::to_string(e) + "] = raw[" + std::to_string(e) + "];\n";
            b += "        }\n";
        } else if (mode == VEC_CONTIG) {
            b += "        { const long long o = off" + J + "(p, " + flat + ");\n";
            for (int e = 0; e < W; e++)
                b += "          " + LJ + "[" + std::to_string(e) + "] = " + ptr + "[o + " + std::to_string(e) + "];\n";
            b += "        }\n";
        } else if (mode == VEC_SPLAT) {
            b += "        { const " + std::string(T) + " x = " + ptr + "[off" + J + "(p, " + flat + ")];\n";
            for (int e = 0; e < W; e++) b += "          " + LJ + "[" + std::to_string(e) + "] = x;\n";
            b += "        }\n";
        } else {
            for (int e = 0; e < W; e++)
                b += "        " + LJ + "[" + std::to_string(e) + "] = " + ptr + "[off" + J + "(p, " + flat + " + " +
                     std::to_string(e) + ")];\n";
        }
    }
    return b;
}

// The stack program run symbolically (slot -> expression name) on the
// loaded leaves: r<sfx>[0..W).
std::string compute(const EwProgram &p, const char *T, int W, const std::string &sfx) {
    std::string b;
    for (int e = 0; e < W; e++) {
        const std::string E = std::to_string(e);
        std::string slot[kMaxDepth + 1];
        for (int i = 0; i < p.n_nodes; i++) {
            const EwNode &nd = p.nodes[i];
            const std::string v = "v" + std::to_string(i) + "_" + E + sfx;
            const std::string I = std::to_string(i);
            switch (nd.kind) {
            case EK_LEAF:
                slot[nd.slot] = "L" + std::to_string(nd.arg) + sfx + "[" + E + "]";
                break;
            case EK_CONST:
                b += "        const " + std::string(T) + " " + v + " = (" + T + ")p.nodes[" + I + "].cval;\n";
                slot[nd.slot] = v;
                break;
            case EK_UNARY:
                b += "        const " + std::string(T) + " " + v + " = unary_op<" + T + ">(" + std::to_string(nd.op) +
                     ", " + slot[nd.slot] + ");\n";
                slot[nd.slot] = v;
                break;
            default:
                b += "        const " + std::string(T) + " " + v + " = binary_op<" + T + ">(" + std::to_string(nd.op) +
                     ", " + slot[nd.slot] + ", " + slot[nd.slot + 1] + ");\n";
                slot[nd.slot] = v;
                break;
            }
        }
        b += "        r" + sfx + "[" + E + "] = " + slot[0] + ";\n";
    }
    return b;
}

// Store of r<sfx>[0..W) at out + flat (16-byte nontemporal when whole).
std::string store(const char *T, int W, bool vec16, bool f64, const std::string &sfx, const std::string &flat) {
    std::string b;
    if (vec16) {
        const std::string VT = f64 ? "tzh_f64x2" : "tzh_f32x4";
        b += "        { " + VT + " o;\n";
        for (int e = 0; e < W; e++) b += "          o[" + std::to_string(e) + "] = r" + sfx + "[" + std::to_string(e) + "];\n";
        b += "          __builtin_nontemporal_store(o, (" + VT + " *)(out + " + flat + ")); }\n";
    } else {
        for (int e = 0; e < W; e++)
            b += "        out[" + flat + " + " + std::to_string(e) + "] = r" + sfx + "[" + std::to_string(e) + "];\n";
    }
    return b;
}

// Grid-stride kernel over numel / V vectors of V outputs.  Each thread
// takes kUnroll vectors (one grid stride apart) per trip: all their leaf
// loads are issued before any arithmetic, which doubles the bytes in flight
// per thread.  Leftover vectors run one per trip; the numel % V tail
// elements run one per thread of block 0.
constexpr int kUnroll = 2;

std::string chain_source(const EwProgram &p, bool f64, int V) {
    const char *T = f64 ? "double" : "float";
    const bool vec16 = V * (f64 ? 8 : 4) == 16;
    std::string s = prelude();
    for (int j = 0; j < p.n_leaves; j++) s += offset_fn(p, j);
    const std::string VS = std::to_string(V);
    s += "extern \"C\" __global__ void __launch_bounds__(256) tzh_chain(const EwProgram p, " + std::string(T) +
         " *__restrict__ out) {\n";
    s += "    const long long nvec = p.numel / " + VS + ";\n";
    s += "    const long long stride = (long long)gridDim.x * blockDim.x;\n";
    s += "    long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x;\n";
    s += "    for (; v + " + std::to_string(kUnroll - 1) + " * stride < nvec; v += " + std::to_string(kUnroll) +
         " * stride) {\n";
    for (int u = 0; u < kUnroll; u++) {
        const std::string U = "_" + std::to_string(u);
        s += "        const long long flat" + U + " = (v + " + std::to_string(u) + " * stride) * " + VS + ";\n";
        s += loads(p, T, V, vec16, U, "flat" + U);
    }
    for (int u = 0; u < kUnroll; u++) {
        const std::string U = "_" + std::to_string(u);
        s += "        " + std::string(T) + " r" + U + "[" + VS + "];\n";
        s += compute(p, T, V, U);
        s += store(T, V, vec16, f64, U, "flat" + U);
    }
    s += "    }\n";
    s += "    for (; v < nvec; v += stride) {\n";
    s += "        const long long flat = v * " + VS + ";\n";
    s += loads(p, T, V, vec16, "", "flat");
    s += "        " + std::string(T) + " r[" + VS + "];\n";
    s += compute(p, T, V, "");
    s += store(T, V, vec16, f64, "", "flat");
    s += "    }\n";
    // tail (numel % V elements): one element per thread of block 0
    s += "    if (blockIdx.x == 0) {\n";
    s += "        const long long flat = nvec * " + VS + " + threadIdx.x;\n";
    s += "        if (flat < p.numel) {\n";
    s += loads(p, T, 1, false, "", "flat");
    s += "        " + std::string(T) + " r[1];\n";
    s += compute(p, T, 1, "");
    s += "        out[flat] = r[0];\n";
    s += "        }\n    }\n}\n";
    return s;
}

// Reduction kernel (reduce_rows or reduce_cols of ew_shared.inc) whose
// operand is the chain: Src::load reads every leaf of kU vectors before any
// arithmetic.
std::string reduce_source(const EwProgram &p, bool cols, bool f64, int V) {
    constexpr int U = 4;
    const std::string T = f64 ? "double" : "float", VS = std::to_string(V), US = std::to_string(U);
    const bool vec16 = V * (f64 ? 8 : 4) == 16;
    std::string s = prelude();
    for (int j = 0; j < p.n_leaves; j++) s += offset_fn(p, j);
    s += "struct Src {\n    static constexpr int kU = " + US + ";\n    const EwProgram &p;\n";
    s += "    __device__ __forceinline__ Batch<" + T + ", " + VS + ", kU> load(const long long (&flat)[kU]) const {\n";
    s += "        Batch<" + T + ", " + VS + ", kU> r;\n";
    for (int u = 0; u < U; u++) s += loads(p, T.c_str(), V, vec16, "_" + std::to_string(u), "flat[" + std::to_string(u) + "]");
    for (int u = 0; u < U; u++) {
        const std::string S = "_" + std::to_string(u);
        s += "        " + T + " r" + S + "[" + VS + "];\n" + compute(p, T.c_str(), V, S);
        for (int e = 0; e < V; e++) {
            const std::string E = std::to_string(e);
            s += "        r.v[" + std::to_string(u) + "].v[" + E + "] = r" + S + "[" + E + "];\n";
        }
    }
    s += "        return r;\n    }\n";
    s += "    __device__ __forceinline__ " + T + " load1(long long flat) const {\n";
    s += loads(p, T.c_str(), 1, false, "", "flat");
    s += "        " + T + " r[1];\n" + compute(p, T.c_str(), 1, "") + "        return r[0];\n    }\n};\n";
    s += "extern \"C\" __global__ void __launch_bounds__(256) tzh_reduce(const EwProgram p, const RedArgs a, " + T +
         " *__restrict__ out) {\n    __shared__ " + T + " smem[" + (cols ? "256 * " + VS : std::string("4")) + "];\n" +
         "    reduce_" + (cols ? "cols" : "rows") + "<" + T + ", " + VS + ">(Src{p}, a, out, smem);\n}\n";
    return s;
}

enum Form : char { kChainForm, kRowsForm, kColsForm };

std::string source_of(const EwProgram &p, Form form, bool f64, int V) {
    return form == kChainForm ? chain_source(p, f64, V) : reduce_source(p, form == kColsForm, f64, V);
}

// What the generated text depends on, in a few hundred bytes: kernels are
// looked up by it, so that a call whose kernel exists builds no text (writing
// and hashing the text took 10 us of a 24 us call).
std::string key_of(int device, const EwProgram &p, Form form, bool f64, int V) {
    std::string k;
    k.reserve(16 + 8 * (size_t)p.n_nodes + 16 * (size_t)p.n_leaves);
    auto put = [&](long long v, int bytes) {
        for (int i = 0; i < bytes; i++) k.push_back((char)((unsigned long long)v >> (8 * i)));
    };
    put(device, 4);
    put(form, 1);
    put(f64, 1);
    put(V, 1);
    put(p.small, 1);
    put(p.ndim, 1);
    put(p.n_nodes, 1);
    put(p.n_leaves, 1);
    for (int i = 0; i < p.n_nodes; i++) {
        const EwNode &nd = p.nodes[i];
        put(nd.kind, 1);
        put(nd.op, 2);
        put(nd.slot, 1);
        put(nd.arg, 1);
    }
    for (int j = 0; j < p.n_leaves; j++) {
        const EwLeaf &lf = p.leaves[j];
        put(lf.general, 1);
        put(lf.vec, 1);
        put(lf.div != 1, 1);
        put(lf.mod <= (long long)0xffffffff, 1);
        int strided = 0;
        for (int d = 0; d < p.ndim; d++) strided |= (lf.strides[d] != 0) << d;
        put(strided, 1);
    }
    return k;
}

// Whether a reduction's kernel should run generated: it is there, or the
// program comes for the second time and may be compiled now.  A compile takes
// about 175 ms, the interpreter a few times the generated kernel's time (0.03
// against 0.02 ms for 64 rows of 384), so a program that evaluates many
// reductions once each compiles none; nor is a module loaded into a stream
// capture.  Both give the same bits.  An
// unseen program leaves an empty entry in the cache.
template <typename Cache, typename There>
bool wants_generated(tzh_ctx *ctx, Cache &cache, const std::string &key, There there) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    const bool capturing = hipStreamIsCapturing(ctx->stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone;
    if (capturing) (void)hipGetLastError();
    auto it = cache.find(key);
    if (it == cache.end()) {
        cache.emplace(key, typename Cache::mapped_type{});
        return false;
    }
    return !capturing || there(it->second);
}

#ifdef TZH_EMULATION
// CPU emulation build (tests/cpu_emu; test infrastructure only): the same
// generated text is compiled as C++ against the emulated runtime header,
// with AddressSanitizer, into a shared object linked to the emulation
// library, and its kernel is run on the emulator's fibers.  The compiler
// and header directory are fixed when the emulation library is built.
using EmuLaunch = void (*)(unsigned grid, const void *p, const void *a, void *out);

std::mutex g_mu;
std::unordered_map<std::string, EmuLaunch> g_cache;  // by key_of
std::string g_dir;

int emu_compile(const std::string &src, bool f64, bool reduce, EmuLaunch *out) {
    if (g_dir.empty()) {
        char tmpl[] = "/tmp/tzh_emu_jit_XXXXXX";
        if (!mkdtemp(tmpl)) return tzh_fail(TZH_ERR_DEVICE, "emulated chain kernel: mkdtemp failed");
        g_dir = tmpl;
    }
    Dl_info info{};
    if (!dladdr((const void *)&jit_chain_launch, &info) || !info.dli_fname)
        return tzh_fail(TZH_ERR_DEVICE, "emulated chain kernel: cannot locate the emulation library");
    static int compiled = 0;  // (under g_mu)
    const std::string stem = g_dir + "/k" + std::to_string(compiled++);
    const char *T = f64 ? "double" : "float";
    std::string text = "#include \"hip/hip_runtime.h\"\n" + src;
    const std::string kernel = reduce ? "tzh_reduce" : "tzh_chain";
    text += "extern \"C\" void tzh_chain_emu_launch(unsigned grid, const void *p, const void *a, void *out) {\n"
            "    emu::launch_kernel(\"" + kernel + " (generated)\", " + kernel + ", dim3(grid), dim3(256),\n"
            "                       *(const EwProgram *)p, " + (reduce ? "*(const RedArgs *)a, " : "") + "(" +
            std::string(T) + " *)out);\n}\n";
    FILE *f = std::fopen((stem + ".cpp").c_str(), "w");
    if (!f) return tzh_fail(TZH_ERR_DEVICE, "emulated chain kernel: cannot write %s.cpp", stem.c_str());
    std::fwrite(text.data(), 1, text.size(), f);
    std::fclose(f);
    const std::string cmd = std::string(TZH_EMU_CXX) + " -x c++ -std=c++17 -O1 -g -fPIC -shared -fsanitize=address" +
                            " -ffp-contract=off -Wno-unused-result -I" + TZH_EMU_INC + " " + stem + ".cpp -x none " +
                            info.dli_fname + " -o " + stem + ".so > " + stem + ".log 2>&1";
    if (std::system(cmd.c_str()) != 0)
        return tzh_fail(TZH_ERR_DEVICE, "emulated chain kernel: compile failed (see %s.log)", stem.c_str());
    void *h = dlopen((stem + ".so").c_str(), RTLD_NOW | RTLD_LOCAL);
    if (!h) return tzh_fail(TZH_ERR_DEVICE, "emulated chain kernel: %s", dlerror());
    *out = (EmuLaunch)dlsym(h, "tzh_chain_emu_launch");
    if (!*out) return tzh_fail(TZH_ERR_DEVICE, "emulated chain kernel: no launcher");
    return TZH_OK;
}

}  // namespace

namespace {

int emu_launch(Form form, const EwProgram &p, const RedArgs *a, bool f64, int V, int grid, void *out) {
    EmuLaunch fn = nullptr;
    {
        const std::string key = key_of(0, p, form, f64, V);
        std::lock_guard<std::mutex> lock(g_mu);
        auto it = g_cache.find(key);
        if (it == g_cache.end() || !it->second) {
            TZH_TRY(emu_compile(source_of(p, form, f64, V), f64, a != nullptr, &fn));
            g_cache[key] = fn;
        } else {
            fn = it->second;
        }
    }
    fn((unsigned)grid, &p, a, out);
    return TZH_OK;
}

}  // namespace

int jit_chain_launch(tzh_ctx *, const EwProgram &p, bool f64, int V, int grid, void *out) {
    return emu_launch(kChainForm, p, nullptr, f64, V, grid, out);
}

bool jit_reduce_wanted(tzh_ctx *ctx, const EwProgram &p, const RedArgs &a, bool f64, int V) {
    const std::string key = key_of(0, p, a.inner > 1 ? kColsForm : kRowsForm, f64, V);
    std::lock_guard<std::mutex> lock(g_mu);
    return wants_generated(ctx, g_cache, key, [](EmuLaunch fn) { return fn != nullptr; });
}

int jit_reduce_launch(tzh_ctx *, const EwProgram &p, const RedArgs &a, bool f64, int V, int grid, void *out) {
    return emu_launch(a.inner > 1 ? kColsForm : kRowsForm, p, &a, f64, V, grid, out);
}

#else
struct Compiled {
    hipModule_t module;
    hipFunction_t fn;
};

std::mutex g_mu;
std::unordered_map<std::string, Compiled> g_cache;  // by key_of

int compile(int device, const std::string &src, const char *kernel, Compiled *out) {
    hipDeviceProp_t prop;
    TZH_HIP(hipGetDeviceProperties(&prop, device));
    std::string arch = prop.gcnArchName;
    arch = arch.substr(0, arch.find(':'));
    hiprtcProgram prog;
    if (hiprtcCreateProgram(&prog, src.c_str(), "tzh_chain.hip", 0, nullptr, nullptr) != HIPRTC_SUCCESS)
        return tzh_fail(TZH_ERR_DEVICE, "hiprtcCreateProgram failed");
    const std::string arch_opt = "--offload-arch=" + arch;
    // same floating-point contract as the library build: no contraction, no
    // packed f32 instructions
    const char *opts[] = {arch_opt.c_str(), "-O3", "-std=c++17", "-ffp-contract=off",
                          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"};
    const hiprtcResult rc = hiprtcCompileProgram(prog, (int)(sizeof opts / sizeof opts[0]), opts);
    if (rc != HIPRTC_SUCCESS) {
        size_t n = 0;
        hiprtcGetProgramLogSize(prog, &n);
        std::string log(n + 1, '\0');
        hiprtcGetProgramLog(prog, &log[0]);
        hiprtcDestroyProgram(&prog);
        return tzh_fail(TZH_ERR_DEVICE, "chain kernel compilation failed (%s): %.1500s", hiprtcGetErrorString(rc),
                        log.c_str());
    }
    size_t n = 0;
    hiprtcGetCodeSize(prog, &n);
    std::vector<char> code(n);
    hiprtcGetCode(prog, code.data());
    hiprtcDestroyProgram(&prog);
    TZH_HIP(hipModuleLoadData(&out->module, code.data()));
    TZH_HIP(hipModuleGetFunction(&out->fn, out->module, kernel));
    return TZH_OK;
}

// The kernel of a program in one form, compiled at its first use on the device.
int lookup(tzh_ctx *ctx, const EwProgram &p, Form form, bool f64, int V, hipFunction_t *fn) {
    const std::string key = key_of(ctx->device, p, form, f64, V);
    std::lock_guard<std::mutex> lock(g_mu);
    auto it = g_cache.find(key);
    if (it == g_cache.end() || !it->second.fn) {
        Compiled k{};
        TZH_TRY(compile(ctx->device, source_of(p, form, f64, V), form == kChainForm ? "tzh_chain" : "tzh_reduce", &k));
        it = g_cache.insert_or_assign(key, k).first;
    }
    *fn = it->second.fn;
    return TZH_OK;
}

}  // namespace

int jit_chain_launch(tzh_ctx *ctx, const EwProgram &p, bool f64, int V, int grid, void *out) {
    hipFunction_t fn;
    TZH_TRY(lookup(ctx, p, kChainForm, f64, V, &fn));
    EwProgram arg = p;
    void *args[] = {&arg, &out};
    TZH_HIP(hipModuleLaunchKernel(fn, (unsigned)grid, 1, 1, 256, 1, 1, 0, ctx->stream, args, nullptr));
    return TZH_OK;
}

bool jit_reduce_wanted(tzh_ctx *ctx, const EwProgram &p, const RedArgs &a, bool f64, int V) {
    const std::string key = key_of(ctx->device, p, a.inner > 1 ? kColsForm : kRowsForm, f64, V);
    std::lock_guard<std::mutex> lock(g_mu);
    return wants_generated(ctx, g_cache, key, [](const Compiled &k) { return k.fn != nullptr; });
}

int jit_reduce_launch(tzh_ctx *ctx, const EwProgram &p, const RedArgs &a, bool f64, int V, int grid, void *out) {
    hipFunction_t fn;
    TZH_TRY(lookup(ctx, p, a.inner > 1 ? kColsForm : kRowsForm, f64, V, &fn));
    EwProgram arg = p;
    RedArgs red = a;
    void *args[] = {&arg, &red, &out};
    TZH_HIP(hipModuleLaunchKernel(fn, (unsigned)grid, 1, 1, 256, 1, 1, 0, ctx->stream, args, nullptr));
    return TZH_OK;
}

#endif

}  // namespace tzh_ew
