// User score / mask mods: the forward, dQ and dK/dV kernels compiled at run
// time (hipRTC) with a policy struct generated from the user's callables, so
// an arbitrary mask_mod / score_mod runs inside the same hand-scheduled tile
// loops as the built-in epilogues.  Host code, included by capi.hip inside its
// anonymous namespace; the exported C ABI functions are at the end of capi.hip.
//
// The policy source defines `struct UserMod` with the members of
// fa::BuiltinMod (kargs.h): kMask / kScore and the mask / score functions,
// reading tensors through Problem::mod_buf.  The kernel headers are embedded
// in the library at build time (rtc_sources.inc, generated by build.py from
// the files under csrc/), so compiling needs nothing but libhiprtc.
//
// A compiled set is a "code blob": a small header (magic, ABI version, the
// hash of the embedded kernel headers, the kernel argument sizes, flags, the
// lowered kernel names) followed by the code object; fa_mods_compile returns
// it (no GPU needed), fa_mods_load turns it into loaded kernels on the
// current GPU.  A blob from another build of the kernel headers (one a
// caller stored, or an old disk-cache entry) would be launched with this
// build's argument layout, so fa_mods_load refuses it (FA_ERR_VERSION)
// before touching the GPU.
#pragma once
// (capi.hip includes <hip/hiprtc.h>, <cstring>, <cstdlib>, <string>, <vector>)
#include "rtc_sources.inc"

// (struct fa_mods, the loaded kernels, is defined in capi.hip at global scope)

constexpr uint32_t kBlobMagic = 0x46414d44;  // "FAMD"
constexpr int kBlobNames = 3;               // fwd, dq, dkdv
constexpr int kNameBytes = 160;

struct BlobHeader {
  uint32_t magic;
  uint32_t abi_version;     // FA_ABI_VERSION of the compiling library
  uint64_t rtc_hash;        // kRtcHash: the kernel headers the code was built from
  uint32_t fwd_args_bytes;  // sizeof(FwdArgs), sizeof(BwdArgs) of that build
  uint32_t bwd_args_bytes;
  int32_t dtype, D, flags;
  char names[kBlobNames][kNameBytes];
  uint64_t code_bytes;
};

// Kernel instantiations for a policy: the bf16 tile kernels (128-query
// forward / dQ tiles of 64 keys, 128-key dK/dV tiles of 64 queries) or the
// float32 split kernels (32-row tiles).  dK/dV in float32 at D = 128 runs the
// general kernel: the split one fills all 512 registers by itself, and with a
// policy's registers spilled on top the compiler (LLVM 22) crashed on two of
// eight policies tried, in the pass that rewrites MFMA copies after spilling.
// (Built-in masks: 680 us with the general kernel, 428 with the split one at
// B2 H16 S2048 causal.)  `general` (FA_MODS_GENERAL): all three, for policies
// that are too much for the split forward or dQ.
std::vector<std::string> mod_kernels(int dtype, int D, bool mods, bool general) {
  const std::string d = std::to_string(D), m = mods ? "true" : "false";
  if (dtype == FA_DTYPE_BF16)
    return {"fa::fwd_bf16_kernel<" + d + ", 64, 4, " + m + ", UserMod>",
            "fa::dq_bf16_kernel<" + d + ", 64, 4, " + m + ", UserMod>",
            "fa::dkdv_bf16_kernel<" + d + ", 64, 4, " + m + ", UserMod>"};
  if (general)
    return {"fa::fwd_kernel<float, " + d + ", 32, 4, " + m + ", UserMod>", "fa::dq_kernel<float, " + d + ", 32, 4, " + m + ", UserMod>",
            "fa::dkdv_kernel<float, " + d + ", 32, 4, " + m + ", UserMod>"};
  return {"fa::fwd_f32_kernel<" + d + ", 4, " + m + ", UserMod>", "fa::dq_f32_kernel<" + d + ", 4, " + m + ", UserMod>",
          D == 128 ? "fa::dkdv_kernel<float, 128, 32, 4, " + m + ", UserMod>"
                   : "fa::dkdv_f32_kernel<" + d + ", 4, " + m + ", UserMod>"};
}

void copy_log(const std::string& text, char* log, size_t log_bytes) {
  if (!log || !log_bytes) return;
  const size_t n = text.size() < log_bytes - 1 ? text.size() : log_bytes - 1;
  memcpy(log, text.data(), n);
  log[n] = '\0';
}

int compile_mods(const char* policy, int dtype, int D, int flags, std::vector<char>* blob, char* log,
                 size_t log_bytes) {
  if (!policy || !blob) return FA_ERR_NULL;
  if (dtype != FA_DTYPE_BF16 && dtype != FA_DTYPE_F32) return FA_ERR_DTYPE;
  if (D != 32 && D != 64 && D != 128) return FA_ERR_UNSUPPORTED;
  const bool general = (flags & FA_MODS_GENERAL) != 0;
  if (general && dtype != FA_DTYPE_F32) return FA_ERR_UNSUPPORTED;
  flags &= ~FA_MODS_GENERAL;  // (the blob's launches are the same)
  if (flags & ~(FA_MODS_MASK | FA_MODS_SCORE | FA_MODS_BUILTIN_SCORE)) return FA_ERR_UNSUPPORTED;
  // the built-in ALiBi / soft-cap epilogue runs only without a user score
  if ((flags & FA_MODS_SCORE) && (flags & FA_MODS_BUILTIN_SCORE)) return FA_ERR_UNSUPPORTED;
  // the kernels' score path runs when the user score or the built-in
  // ALiBi / soft-cap is present
  const bool mods = (flags & (FA_MODS_SCORE | FA_MODS_BUILTIN_SCORE)) != 0;
  const std::vector<std::string> kernels = mod_kernels(dtype, D, mods, general);
  std::string src = dtype == FA_DTYPE_BF16 ? "#include \"fwd_bf16.h\"\n#include \"bwd_bf16.h\"\n"
                                           : "#include \"f32_split.h\"\n";
  src += "\n";
  src += policy;
  src += "\n";
  // the policy must be the one the flags describe: the launches set up the
  // mask walk and the score epilogue from the flags
  src += std::string("static_assert(UserMod::kMask == ") + ((flags & FA_MODS_MASK) ? "true" : "false") +
         ", \"UserMod::kMask disagrees with FA_MODS_MASK\");\n";
  src += std::string("static_assert(UserMod::kScore == ") + ((flags & FA_MODS_SCORE) ? "true" : "false") +
         ", \"UserMod::kScore disagrees with FA_MODS_SCORE\");\n";
  const char* args[kBlobNames] = {"fa::FwdArgs", "fa::BwdArgs", "fa::BwdArgs"};
  for (int i = 0; i < kBlobNames; ++i) src += "template __global__ void " + kernels[i] + "(" + args[i] + ");\n";

  hiprtcProgram prog;
  if (hiprtcCreateProgram(&prog, src.c_str(), "user_mods.hip", kRtcHeaders, kRtcHeaderSources, kRtcHeaderNames) !=
      HIPRTC_SUCCESS)
    return FA_ERR_COMPILE;
  std::vector<std::string> exprs;
  for (const auto& k : kernels) exprs.push_back("&" + k);
  for (const auto& e : exprs) hiprtcAddNameExpression(prog, e.c_str());
  const char* opts[] = {"--offload-arch=gfx950", "-O3", "-std=c++17",
                        // the build's own flags (build.py): no packed-fp32 VALU, MFMA
                        // accumulators in VGPRs, fully unrolled tile schedules
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                        "-mllvm", "-amdgpu-mfma-vgpr-form=1", "-mllvm", "-pragma-unroll-threshold=200000"};
  const hiprtcResult cr = hiprtcCompileProgram(prog, (int)(sizeof(opts) / sizeof(opts[0])), opts);
  size_t log_size = 0;
  hiprtcGetProgramLogSize(prog, &log_size);
  std::string text(log_size, '\0');
  if (log_size) hiprtcGetProgramLog(prog, &text[0]);
  copy_log(text, log, log_bytes);
  if (cr != HIPRTC_SUCCESS) {
    hiprtcDestroyProgram(&prog);
    return FA_ERR_COMPILE;
  }
  BlobHeader h;
  memset(&h, 0, sizeof(h));
  h.magic = kBlobMagic;
  h.abi_version = FA_ABI_VERSION;
  h.rtc_hash = kRtcHash;
  h.fwd_args_bytes = (uint32_t)sizeof(FwdArgs);
  h.bwd_args_bytes = (uint32_t)sizeof(BwdArgs);
  h.dtype = dtype;
  h.D = D;
  h.flags = flags;
  for (int i = 0; i < kBlobNames; ++i) {
    const char* lowered = nullptr;
    if (hiprtcGetLoweredName(prog, exprs[i].c_str(), &lowered) != HIPRTC_SUCCESS || !lowered ||
        strlen(lowered) >= (size_t)kNameBytes) {
      hiprtcDestroyProgram(&prog);
      return FA_ERR_COMPILE;
    }
    strcpy(h.names[i], lowered);
  }
  size_t code_bytes = 0;
  hiprtcGetCodeSize(prog, &code_bytes);
  h.code_bytes = code_bytes;
  blob->assign(sizeof(h) + code_bytes, 0);
  memcpy(blob->data(), &h, sizeof(h));
  hiprtcGetCode(prog, blob->data() + sizeof(h));
  hiprtcDestroyProgram(&prog);
  return FA_OK;
}

int load_mods(const void* blob, size_t bytes, fa_mods** out) {
  if (!blob || !out) return FA_ERR_NULL;
  BlobHeader h;
  if (bytes < sizeof(h)) return FA_ERR_SHAPE;
  memcpy(&h, blob, sizeof(h));
  if (h.magic != kBlobMagic) return FA_ERR_SHAPE;
  if (h.abi_version != FA_ABI_VERSION || h.rtc_hash != kRtcHash || h.fwd_args_bytes != sizeof(FwdArgs) ||
      h.bwd_args_bytes != sizeof(BwdArgs))
    return FA_ERR_VERSION;
  if (sizeof(h) + h.code_bytes != bytes) return FA_ERR_SHAPE;
  if ((h.dtype != FA_DTYPE_BF16 && h.dtype != FA_DTYPE_F32) || (h.D != 32 && h.D != 64 && h.D != 128))
    return FA_ERR_SHAPE;
  for (int i = 0; i < kBlobNames; ++i)
    if (memchr(h.names[i], 0, kNameBytes) == nullptr) return FA_ERR_SHAPE;
  fa_mods* m = new fa_mods;
  m->dtype = h.dtype;
  m->D = h.D;
  m->flags = h.flags;
  if (hipGetDevice(&m->device) != hipSuccess ||
      hipModuleLoadData(&m->module, static_cast<const char*>(blob) + sizeof(h)) != hipSuccess) {
    delete m;
    return FA_ERR_LAUNCH;
  }
  hipFunction_t* fns[kBlobNames] = {&m->fwd, &m->dq, &m->dkdv};
  for (int i = 0; i < kBlobNames; ++i) {
    if (hipModuleGetFunction(fns[i], m->module, h.names[i]) != hipSuccess) {
      (void)hipModuleUnload(m->module);  // the lookup's error is the one reported
      delete m;
      return FA_ERR_LAUNCH;
    }
  }
  *out = m;
  return FA_OK;
}

template <typename Args>
int launch_module(hipFunction_t f, unsigned grid, unsigned block, const Args& a, hipStream_t s) {
  Args copy = a;
  void* params[] = {&copy};
  return hipModuleLaunchKernel(f, grid, 1, 1, block, 1, 1, 0, s, params, nullptr) == hipSuccess ? FA_OK
                                                                                              : FA_ERR_LAUNCH;
}

// Problem for a call with user mods: the fa_params checks of fa_fwd / fa_bwd,
// plus the mods' tensors and (with a user mask) partial-tile masking on
// dense walks.
int mods_problem(const fa_mods* m, const fa_params* p, const void* const* bufs, int nbufs, Problem* pr,
                 Tiles* t) {
  if (!m || !p) return FA_ERR_NULL;
  (void)device_scratch();
  if (p->dtype != m->dtype || p->D != m->D) return FA_ERR_DTYPE;
  if (nbufs < 0 || nbufs > 8 || (nbufs > 0 && !bufs)) return FA_ERR_SHAPE;
  fa_params q = *p;
  q.block_m = q.block_n = q.block_kv = q.block_q = q.lds_stages = 0;  // the compiled tiles
  int rc = default_tiles(&q, t);
  if (rc) return rc;
  t->bq = m->dtype == FA_DTYPE_BF16 ? 64 : 32;  // (mod_kernels)
  rc = build_problem(&q, *t, pr);
  if (rc) return rc;
  // the bf16 tile kernels take masks as key intervals (window, contiguous
  // documents); document labels travel inside a user mask instead
  if (m->dtype == FA_DTYPE_BF16 && !interval_masks(*pr)) return FA_ERR_UNSUPPORTED;
  // ALiBi / soft-cap in the params run only in a blob built for them
  // (FA_MODS_BUILTIN_SCORE); any other blob would silently drop them
  if (has_mods(*pr) && !(m->flags & FA_MODS_BUILTIN_SCORE)) return FA_ERR_UNSUPPORTED;
  for (int i = 0; i < 8; ++i) pr->mod_buf[i] = i < nbufs ? bufs[i] : nullptr;
  if (m->flags & FA_MODS_MASK) pr->has_mask = 1;
  return FA_OK;
}
