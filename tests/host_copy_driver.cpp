// Transfers through host_copy.hip on the CPU (tests/fake_hip), one per argument:
//   h<bytes> to the host, d<bytes> to the device, p<bytes> to a pinned host buffer,
//   f<n> from now on at most n pinned slots, g give the stage back.
// Prints per transfer: whether the bytes are right, chunks moved by the kernel, plain
// copies, pinned slots held, calls for pinned memory.
#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

#include "host_copy.hpp"

int main(int argc, char **argv) {
  chan::HostStage s;
  unsigned seed = 1;
  for (int i = 1; i < argc; i++) {
    const char what = argv[i][0];
    const size_t n = std::strtoull(argv[i] + 1, nullptr, 10);
    if (what == 'f') {
      fake::pin_limit = (int)n;
      continue;
    }
    if (what == 'g') {
      s.free();
      std::printf("held %d %d\n", fake::pinned.load(), fake::events.load());
      continue;
    }
    std::vector<unsigned> a(n / 4), b(n / 4 + 1, 7u);
    for (auto &v : a) v = seed = seed * 1664525u + 1013904223u;
    const int l0 = fake::launches, p0 = fake::plain, c0 = fake::pin_calls, w0 = fake::waits;
    fake::pinned_host = what == 'p' ? b.data() : nullptr;
    const hipError_t e = what == 'd' ? chan::copy_to_device(s, b.data(), a.data(), n, nullptr)
                                     : chan::copy_to_host(s, b.data(), a.data(), n, nullptr);
    const bool ok = e == hipSuccess && std::memcmp(a.data(), b.data(), n) == 0 && b[n / 4] == 7u &&
                    (what == 'd' || fake::waits > w0);
    std::printf("%d %d %d %d %d\n", ok, fake::launches - l0, fake::plain - p0, fake::pinned.load(), fake::pin_calls - c0);
  }
  s.free();
  return fake::pinned || fake::events ? 3 : 0;
}
