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

// The entries that a range minimum reads, over all lanes: exactly the range,
// each value once, also next to 2^32, at most two wave reads per end and step.
void stretch() {
  const uint32_t top = 0xfffffffeu;
  auto one = [&](uint32_t lo, uint32_t hi) {
    unsigned long long covered = 0;
    bool inside = true;
    uint32_t most = 0;
    for (uint32_t lane = 0; lane < 64; lane++) {
      uint32_t few = 0;
      pst::stretch_minima(lo, hi, lane, [&](uint32_t step, uint32_t i) {
        const unsigned long long w = 1ull << (6 * step);
        inside &= i * w >= lo && i * w + w <= hi;
        covered += w;
        if (step < 3) few++;
      });
      most = few > most ? few : most;
    }
    CHECK(inside, lo);
    CHECK(covered == (hi > lo ? hi - lo : 0), lo);
    CHECK(most <= 6, lo);
  };
  for (uint32_t n : {1u, 63u, 64u, 65u, 128u, 4095u, 4096u, 4097u, 300007u, 0x10000000u, 0xffffff80u, 0xffffffbfu,
                     0xffffffc0u, 0xffffffc1u, 0xfffffff0u, top}) {
    one(0, n);
    for (uint32_t d : {0u, 1u, 2u, 62u, 63u, 64u, 65u, 127u, 128u, 4000u, 4096u, 5000u, 270000u})
      for (uint32_t w : {1u, 2u, 63u, 64u, 65u, 127u, 128u, 200u, 4097u, 262145u})
        if (d + w <= n) {
          one(n - d - w, n - d);  // ranges that end at or near the array's end
          one(d, d + w);
        }
  }
  for (uint32_t n : {1u, 64u, 65u, 0xffffffc0u, 0xffffffc1u, top}) {
    CHECK(pst::blocks_of(n) == (n + 63ull) / 64, n);
    CHECK(pst::blocks_of(static_cast<size_t>(n)) == (n + 63ull) / 64, n);
  }
  // hole lists: a level's segments hold at most one hole per level above it
  for (unsigned long long n : {1ull, 2048ull, 2049ull, 1ull << 26, 1ull << 31, 0xfffffffeull}) {
    CHECK(pst::finish_level(n + 1) <= pst::kMaxHoles, n);
    CHECK(pst::level_size(n + 1, pst::finish_level(n + 1), 0) <= 2048, n);
  }
}

// A round's list over its waves: every item once, shares within one of each
// other, and no more grabs than allowed where the list could be dealt evenly.
void deal() {
  for (uint32_t waves : {1u, 3u, 256u, 8192u})
    for (uint32_t most : {1u, 4u, 64u})
      for (uint32_t grabs : {0u, 1u, 100u, 8192u})
        for (unsigned long long per : {0ull, 1ull, 2ull, 3ull, 17ull, 63ull, 64ull, 200ull})
          for (unsigned long long more : {0ull, 1ull, waves / 2ull, waves - 1ull}) {
            const unsigned long long count = per * waves + (more < waves ? more : 0);
            unsigned long long at = 0, low = ~0ull, high = 0, dyn = 0;
            uint32_t unit = 0;
            bool ok = true;
            for (uint32_t w = 0; w < waves; w++) {
              const pst::Deal d = pst::deal_items(count, waves, w, most, grabs);
              ok &= (w == 0 || (d.dyn == dyn && d.unit == unit)) && d.base == at && d.cnt <= most;
              dyn = d.dyn;
              unit = d.unit;
              at += d.cnt;
              low = d.cnt < low ? d.cnt : low;
              high = d.cnt > high ? d.cnt : high;
            }
            CHECK(ok, count);
            CHECK(at == dyn && dyn <= count, count);
            CHECK(high - low <= 1, count);
            const unsigned long long left = count - dyn;
            CHECK(left == 0 || unit > 0, count);
            CHECK(left == 0 || per >= most || (left + unit - 1) / unit <= grabs, count);
          }
}

// Which lists of a round count as short: forests and budgets set by the caller
// as ever, the default schedule of group walks on a deep tree four times that.
void few() {
  pst::SearchArgs a{};
  a.n = 1 << 24;
  CHECK(pst::few_items(a, 8, 8192) == 4 * 8192, 0);
  CHECK(pst::few_items(a, 1, 8192) == 8192, 0);
  a.budget_small = 6;
  CHECK(pst::few_items(a, 8, 8192) == 8192, 0);
  a.budget_small = 0;
  a.rounds = 4;
  CHECK(pst::few_items(a, 8, 8192) == 8192, 0);
  a.rounds = 2;
  CHECK(pst::few_items(a, 8, 8192) == 4 * 8192, 0);
  a.rounds = 0;
  a.slots_per_tree = 1023;
  CHECK(pst::few_items(a, 8, 8192) == 8192, 0);
}
}  // namespace

int main(int argc, char** argv) {
  const std::string only = argc > 1 ? argv[1] : "";
  if (only.empty() || only == "level_slots") level_slots();
  if (only.empty() || only == "stretch") stretch();
  if (only.empty() || only == "deal") deal();
  if (only.empty() || only == "few") few();
  std::printf(g_bad ? "%d checks failed\n" : "LAYOUT OK\n", g_bad);
  return g_bad != 0;
}
