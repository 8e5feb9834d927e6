// Kernel text -> code object, with the compiler of the ROCm that the library was built with.
//
// hiprtc and the compiler behind it (comgr) are found by soname, so a process that has already loaded another
// ROCm's copies (PyTorch ships its own) would compile the kernels with those.  What that costs is not small: the
// waits of the MFMA skeletons are placed by hand, and a compiler that does not see that a direct-to-LDS load and an
// LDS read touch different stages adds a full `s_waitcnt vmcnt(0)` in front of the reads (44 instead of 7 in the bf16
// 256 x 256 kernel) and spills (46 registers in the fp8 one).  MLP of 412 GFLOP in a process with PyTorch's ROCm 7.0
// libraries: 0.872 ms compiled in the process, 0.33 ms compiled by ROCm 7.2; fp8 8192^3 layer 1.73 against 0.47 ms.
// Where another copy is loaded, the text goes to a child process (rx_rtc_worker.cpp, a program without any other
// library) instead; where none is, hiprtc is called here, which saves the child's start (about 0.1 s).
#include "rx_rtc.h"

#include <fcntl.h>
#include <spawn.h>
#include <sys/mman.h>
#include <sys/stat.h>
#include <sys/wait.h>
#include <unistd.h>

#include <dlfcn.h>

#include <algorithm>
#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "rx_ir.h"
#include "rx_rtc_hiprtc.h"

extern char** environ;

namespace rx {
namespace {

// The worker's environment: without another ROCm's libraries (LD_LIBRARY_PATH, which goes before the path that hiprtc looks for
// comgr on; entries of LD_PRELOAD that are one of ROCm's), and without what makes a profiler's library start the GPU.
std::vector<std::string> worker_environment() {
  std::vector<std::string> env;
  auto starts = [](const std::string& s, const char* p) { return s.compare(0, strlen(p), p) == 0; };
  for (char** e = environ; *e; ++e) {
    const std::string v = *e;
    if (starts(v, "LD_LIBRARY_PATH=") || starts(v, "ROCP_") || starts(v, "ROCPROF") || starts(v, "ROCTRACER_") || starts(v, "HSA_TOOLS_")) continue;
    if (!starts(v, "LD_PRELOAD=")) { env.push_back(v); continue; }
    std::string kept;
    for (size_t at = strlen("LD_PRELOAD="); at < v.size();) {
      const size_t end = std::min(v.find_first_of(": ", at), v.size());
      const std::string lib = v.substr(at, end - at), base = lib.substr(lib.rfind('/') + 1);
      bool rocm = lib.empty();
      for (const char* p : {"libamd_comgr", "libhiprtc", "libamdhip64", "libhsa-runtime64", "librocprof", "libroctracer", "libroctx"}) rocm = rocm || starts(base, p);
      if (!rocm) kept += (kept.empty() ? "" : ":") + lib;
      at = end + 1;
    }
    if (!kept.empty()) env.push_back("LD_PRELOAD=" + kept);
  }
  return env;
}

// The worker lies beside this library.
const std::string& worker_path() {
  static const std::string path = [] {
    Dl_info i;
    if (!dladdr((const void*)&rtc_compile, &i) || !i.dli_fname) return std::string();
    return real_dir(i.dli_fname) + "/rx_rtc_worker.so";
  }();
  return path;
}

struct Fd {
  int fd = -1;
  ~Fd() { if (fd >= 0) close(fd); }
};

// An anonymous file, above the descriptors that the worker's process uses.
int anonymous_file(const char* name) {
  const int fd = memfd_create(name, MFD_CLOEXEC);
  if (fd < 0) return -1;
  const int up = fcntl(fd, F_DUPFD_CLOEXEC, kWorkerResult + 1);
  close(fd);
  return up;
}

// Source and result pass through anonymous files, so neither side waits for the other while it writes.  The result has a
// descriptor of its own: a library that is preloaded into every process may write to standard output.
// True: *code / *error is the worker's answer.  False: it could not be started or did not finish.  That is read off the result's
// last bytes, not the exit status, which a process that ignores SIGCHLD or waits for any child does not get to see.
bool worker_compile(const std::string& source, const std::string& arch, std::string* code, std::string* error) {
  Fd in, out;
  in.fd = anonymous_file("rx_source");
  out.fd = anonymous_file("rx_code");
  if (in.fd < 0 || out.fd < 0) return false;
  for (size_t at = 0; at < source.size();) {
    const ssize_t n = write(in.fd, source.data() + at, source.size() - at);
    if (n < 0 && errno == EINTR) continue;
    if (n <= 0) return false;
    at += (size_t)n;
  }
  if (lseek(in.fd, 0, SEEK_SET) < 0) return false;
  posix_spawn_file_actions_t fa;
  if (posix_spawn_file_actions_init(&fa) != 0) return false;
  posix_spawn_file_actions_adddup2(&fa, in.fd, 0);
  posix_spawn_file_actions_adddup2(&fa, out.fd, kWorkerResult);
  posix_spawn_file_actions_addopen(&fa, 1, "/dev/null", O_WRONLY, 0);
  posix_spawn_file_actions_addclosefrom_np(&fa, kWorkerResult + 1);
  const char* argv[] = {worker_path().c_str(), arch.c_str(), nullptr};
  pid_t pid = -1;
  std::vector<std::string> env = worker_environment();
  std::vector<char*> envp;
  for (std::string& v : env) envp.push_back(&v[0]);
  envp.push_back(nullptr);
  const int rc = posix_spawn(&pid, argv[0], &fa, nullptr, const_cast<char**>(argv), envp.data());
  posix_spawn_file_actions_destroy(&fa);
  if (rc != 0) return false;
  // fails with ECHILD once the worker has ended if its status went elsewhere
  while (waitpid(pid, nullptr, 0) < 0)
    if (errno != EINTR) break;
  struct stat st;
  if (fstat(out.fd, &st) != 0 || st.st_size < (off_t)sizeof(WorkerEnd)) return false;
  std::string got((size_t)st.st_size, '\0');
  for (size_t at = 0; at < got.size();) {
    const ssize_t n = pread(out.fd, &got[at], got.size() - at, (off_t)at);
    if (n < 0 && errno == EINTR) continue;
    if (n <= 0) return false;
    at += (size_t)n;
  }
  WorkerEnd end;
  got.copy((char*)&end, sizeof(end), got.size() - sizeof(end));
  got.resize(got.size() - sizeof(end));
  if (end.magic != kWorkerMagic || end.length != got.size() || end.status > 1) return false;
  (end.status == 0 ? *code : *error) = std::move(got);
  return true;
}

}  // namespace

std::string rtc_compile(const std::string& source, const std::string& arch) {
  std::string code, error;
  bool done = false;
  if (foreign_compiler_loaded()) {
    done = worker_compile(source, arch, &code, &error);
    if (!done) {
      static std::once_flag told;
      std::call_once(told, [] {
        fprintf(stderr, "reactant_mi355x: %s could not be run; kernels are compiled by the hiprtc that this process has loaded, "
                        "which may make them slower\n", worker_path().c_str());
      });
    }
  }
  if (!done && hiprtc_compile(source, arch, &code) != 0) { error.swap(code); }
  if (!error.empty()) {
    if (getenv("RX_DUMP_FAILED_SOURCE")) {
      FILE* f = fopen(getenv("RX_DUMP_FAILED_SOURCE"), "w");
      if (f) { fputs(source.c_str(), f); fclose(f); }
    }
    throw Error(error);
  }
  if (const char* e = getenv("RX_DUMP_CODE_OBJECT")) {
    FILE* f = fopen(e, "wb");
    if (f) { fwrite(code.data(), 1, code.size(), f); fclose(f); }
  }
  return code;
}

}  // namespace rx
