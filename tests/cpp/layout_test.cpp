// Host checks of sizes and index arithmetic that kernels rely on.
#include <cstdint>
#include <cstdio>
#include <string>

#include "pst_internal.hpp"

namespace {
int g_bad = 0;
void check(bool ok, const char* what, unsigned long long n, int line) {
  if (ok) return;
  g_bad++;
  std::printf("FAILED line %d (n = %llu): %s\n", line, n, what);
}
#define CHECK(x, n) check((x), #x, static_cast<unsigned long long>(n), __LINE__)

// Level index construction reads both slot arrays and every level 16 bytes at
// a time: each starts 256-byte aligned, and nothing overlaps.
void level_slots() {
  for (size_t n : {size_t{1}, size_t{2}, size_t{3}, size_t{63}, size_t{64}, size_t{65}, size_t{4099}, size_t{8000003},
                   size_t{1} << 26, (size_t{1} << 31) - 1}) {
    const pst::LevelSlots s = pst::level_slots(n);
    CHECK(s.second * 4 % 256 == 0, n);
    CHECK(s.second >= n, n);
    CHECK(s.bytes >= (s.second + n) * 4, n);
    CHECK(pst::level_stride(n) * 4 % 256 == 0 && pst::level_stride(n) >= n, n);
  }
}
}  // namespace

int main(int argc, char** argv) {
  const std::string only = argc > 1 ? argv[1] : "";
  if (only.empty() || only == "level_slots") level_slots();
  std::printf(g_bad ? "%d checks failed\n" : "LAYOUT OK\n", g_bad);
  return g_bad != 0;
}
