// HostPipe on the stand-in runtime: prints, for the case named on the command
// line, the return code, whether the bytes arrived, how many copies the link
// made and how many of them used the caller's own memory.  "solvers <up|down>
// <bytes> <threads>": that many threads with a pipe each, three copies of each,
// one thread after another (up) or all at once (down); prints the bytes that
// arrived wrong, the rings allocated, those held before and after the pipes go.
#include "../../m2c_amd/csrc/m2c_hostcopy.h"
#include <cstdio>
#include <string>

using m2c::HostPipe;

static int solvers(bool in_turn, size_t n, int count) {
  std::vector<HostPipe> pipes(count);
  std::atomic<int> bad{0};
  auto work = [&](int q) {
    pipes[q].attach(0);
    std::vector<char> a(n), b(n);
    for (int pass = 0; pass < 3; pass++) {
      std::memset(a.data(), 16 * q + pass + 1, n);
      const hipError_t e = pass % 2 ? pipes[q].to_device(b.data(), a.data(), n, 0) : pipes[q].to_host(b.data(), a.data(), n, 0);
      if (e != hipSuccess || a != b) bad++;
    }
  };
  std::vector<std::thread> t;
  for (int q = 0; q < count; q++) {
    t.emplace_back(work, q);
    if (in_turn) t[q].join();
  }
  if (!in_turn)
    for (auto& x : t) x.join();
  const size_t held = fake().pinned.size();
  pipes = std::vector<HostPipe>();
  std::printf("%d %zu %zu %zu\n", bad.load(), fake().allocated, held, fake().pinned.size());
  return 0;
}

int main(int argc, char** argv) {
  const std::string what = argv[1];
  if (what == "solvers") return solvers(std::string(argv[2]) == "up", (size_t)std::atol(argv[3]), std::atoi(argv[4]));
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
  pipe.attach(0);
  for (int pass = 0; pass < 2; pass++) {  // the second uses the ring again
    f.log.clear();
    if (pass) std::memset((up ? dev : host).data(), 0, n);
    const hipError_t e = up ? pipe.to_device(dev.data(), host.data(), n, 0)
                            : pipe.to_host(host.data(), dev.data(), n, 0);
    size_t own = 0;
    for (auto& c : f.log) {
      const char* p = static_cast<const char*>(up ? c.src : c.dst);
      own += p >= host.data() && p < host.data() + n;
    }
    std::printf("%d %d %zu %zu\n", (int)e, (int)(host == dev), f.log.size(), own);
  }
  return 0;
}
