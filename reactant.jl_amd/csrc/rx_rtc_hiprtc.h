// One compilation with the hiprtc that this program or library is linked to (rx_rtc.cpp and rx_rtc_worker.cpp).
#pragma once
#include <hip/hiprtc.h>
#include <limits.h>
#include <link.h>

#include <cstdlib>
#include <cstring>

#include <cstdint>
#include <string>
#include <vector>

#include "rx_embedded.inc"

#ifndef RX_ROCM_LIB
#define RX_ROCM_LIB "/opt/rocm/lib"
#endif

namespace rx {

static std::string real_dir(const char* path) {
  char buf[PATH_MAX];
  const std::string p = realpath(path, buf) ? buf : path;
  const size_t s = p.rfind('/');
  return s == std::string::npos ? std::string(".") : p.substr(0, s);
}

// Has a hiprtc or a comgr from elsewhere than RX_ROCM_LIB been loaded into this process?
static bool foreign_compiler_loaded() {
  static const std::string own = real_dir(RX_ROCM_LIB "/libhiprtc.so");
  bool foreign = false;
  dl_iterate_phdr(
      [](struct dl_phdr_info* i, size_t, void* f) {
        const char* base = i->dlpi_name ? strrchr(i->dlpi_name, '/') : nullptr;
        if (base && (!strncmp(base, "/libhiprtc.so", 13) || !strncmp(base, "/libamd_comgr.so", 16)) && real_dir(i->dlpi_name) != own) *(bool*)f = true;
        return 0;
      },
      &foreign);
  return foreign;
}

constexpr int kWorkerResult = 3;   // the descriptor that the worker writes its answer to
// What follows the answer, a code object (status 0) or an error text (1).
struct WorkerEnd { uint64_t magic, status, length; };
constexpr uint64_t kWorkerMagic = 0x5258525443454e44;

// 0 and the code object, or non-zero and the error text.
static int hiprtc_compile(const std::string& source, const std::string& arch, std::string* out) {
  hiprtcProgram prog;
  const char* hdr_src[] = {kRxPreambleSrc, kRxGemmKernelsSrc};
  const char* hdr_name[] = {"rx_preamble.h", "rx_gemm_kernels.h"};
  hiprtcResult r = hiprtcCreateProgram(&prog, source.c_str(), "rx_module.hip", 2, hdr_src, hdr_name);
  if (r != HIPRTC_SUCCESS) {
    *out = std::string("hiprtcCreateProgram: ") + hiprtcGetErrorString(r);
    return 1;
  }
  std::string archopt = "--offload-arch=" + arch;
  std::vector<const char*> opts = {archopt.c_str(), "-O3", "-std=c++17", "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang",
                                   "-packed-fp32-ops", "-Wno-unused-value"};
  r = hiprtcCompileProgram(prog, (int)opts.size(), opts.data());
  size_t n = 0;
  if (r != HIPRTC_SUCCESS) {
    hiprtcGetProgramLogSize(prog, &n);
    std::string log(n, '\0');
    if (n) hiprtcGetProgramLog(prog, &log[0]);
    *out = std::string("kernel compilation failed (") + hiprtcGetErrorString(r) + "):\n" + log;
    hiprtcDestroyProgram(&prog);
    return 1;
  }
  hiprtcGetCodeSize(prog, &n);
  out->assign(n, '\0');
  hiprtcGetCode(prog, &(*out)[0]);
  hiprtcDestroyProgram(&prog);
  return 0;
}

}  // namespace rx
