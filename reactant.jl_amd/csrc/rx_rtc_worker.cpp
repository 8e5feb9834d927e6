// Compiles one kernel text in a process of its own: source on standard input, architecture as the argument, the code
// object or the error text and a WorkerEnd on descriptor kWorkerResult.  Started by rx_rtc.cpp; touches no GPU.
// Ends without an answer where another ROCm's compiler was loaded into it all the same.
#include <unistd.h>

#include <cerrno>

#include "rx_rtc_hiprtc.h"

int main(int argc, char** argv) {
  if (argc != 2) return 2;
  std::string source, out;
  char buf[1 << 16];
  for (;;) {
    const ssize_t n = read(0, buf, sizeof(buf));
    if (n < 0 && errno == EINTR) continue;
    if (n < 0) return 2;
    if (n == 0) break;
    source.append(buf, (size_t)n);
  }
  const int rc = rx::hiprtc_compile(source, argv[1], &out) == 0 ? 0 : 1;
  if (rx::foreign_compiler_loaded()) return 2;
  const rx::WorkerEnd end = {rx::kWorkerMagic, (uint64_t)rc, out.size()};
  out.append((const char*)&end, sizeof(end));
  for (size_t at = 0; at < out.size();) {
    const ssize_t n = write(rx::kWorkerResult, out.data() + at, out.size() - at);
    if (n < 0 && errno == EINTR) continue;
    if (n <= 0) return 2;
    at += (size_t)n;
  }
  return rc;
}
