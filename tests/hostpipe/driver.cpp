// HostPipe on the stand-in runtime: prints, for the case named on the command
// line, the return code, whether the bytes arrived, how many copies the link
// made and how many of them used the caller's own memory.
#include "../../m2c_amd/csrc/m2c_hostcopy.h"
#include <cstdio>
#include <string>

using m2c::HostPipe;

int main(int argc, char** argv) {
  const std::string what = argv[1];
  const bool up = std::string(argv[2]) == "up";
  const size_t n = (size_t)std::atol(argv[3]);
  FakeHip& f = fake();
  std::vector<char> host(n), dev(n);
  for (size_t i = 0; i < n; i++) (up ? host : dev)[i] = (char)(i * 2654435761u >> 13);
  f.unregistered_is_error = what == "older-runtime";
  f.no_pinned = what == "no-pinned-memory";
  if (what == "pinned") f.pin(host.data(), n);
  if (what == "pinned-tail") f.pin(host.data() + n / 2, n - n / 2);
  if (what == "pinned-head") f.pin(host.data(), n / 2);
  if (what == "link-fails") f.fail_copy = 5;
  HostPipe pipe;
  for (int pass = 0; pass < 2; pass++) {  // the second uses the ring again
    f.log.clear();
    if (pass) std::memset((up ? dev : host).data(), 0, n);
    const hipError_t e = up ? pipe.to_device(0, dev.data(), host.data(), n, 0)
                            : pipe.to_host(0, host.data(), dev.data(), n, 0);
    size_t own = 0;
    for (auto& c : f.log) {
      const char* p = static_cast<const char*>(up ? c.src : c.dst);
      own += p >= host.data() && p < host.data() + n;
    }
    std::printf("%d %d %zu %zu\n", (int)e, (int)(host == dev), f.log.size(), own);
  }
  return 0;
}
