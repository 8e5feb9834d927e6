// One compilation with the hiprtc that this program or library is linked to (rx_rtc.cpp and rx_rtc_worker.cpp).
#pragma once
#include <hip/hiprtc.h>

#include <cstdint>
#include <string>
#include <vector>

#include "rx_embedded.inc"

namespace rx {

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
