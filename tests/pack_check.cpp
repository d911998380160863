// Host-side check of what a packed residue's heads and words have to be to be believed (pack.h), built by
// tests/test_pack_check.py. Heads and words are made as k_pack makes them; then every single bit of
// what is read back is flipped in turn, and a head or a run of words goes missing. Prints "OK" or the first failures.
#include "pack.h"

#include <cstdio>
#include <random>
#include <vector>

namespace {
int bad = 0;
void expect(bool ok, const char* what) {
  if (!ok && ++bad <= 10) { std::printf("%s\n", what); }
}
struct Read {
  PackHead h[2];
  std::vector<uint32_t> w;
};
// Random words and the head for them; negative: the digits are worth 2^E - 1 less.
Read packed(uint32_t E, std::mt19937_64& gen, bool negative, uint32_t groups) {
  Read r{};
  r.w.resize((E - 1) / 32 + 1);
  uint64_t sum = 0;
  for (auto& x : r.w) { x = uint32_t(gen()); }
  r.w.back() &= (1u << E % 32) - 1;
  for (uint32_t x : r.w) { sum += x; }
  constexpr uint64_t M = 0xffffffffu;
  const uint64_t less = negative ? M - ((uint64_t(1) << E % 32) - 1) % M : 0;
  r.h[0] = {sum, (sum + less) % M + M * (gen() % 1000), PACK_NONZERO | (negative ? PACK_NEGATIVE : 0u), groups, 0};  // summed over groups, not reduced
  r.h[1] = r.h[0];
  return r;
}
}  // namespace

int main() {
  std::mt19937_64 gen(5);
  for (uint32_t E : {1000003u, 4000037u, 65537u, 2097169u, 1048607u}) {
    for (bool negative : {false, true}) {
      const uint32_t groups = 200;
      const Read good = packed(E, gen, negative, groups);
      const uint32_t n = uint32_t(good.w.size());
      expect(packVerdict(good.h, groups) == PackRead::Words, "good head refused");
      expect(packedWordsMatch(good.w.data(), n, good.h[0], E), "good words refused");
      for (size_t bit = 0; bit < 8 * sizeof(good.h); ++bit) {
        Read r = good;
        reinterpret_cast<uint8_t*>(r.h)[bit / 8] ^= uint8_t(1u << bit % 8);
        expect(packVerdict(r.h, groups) == PackRead::Again, "one wrong bit in a head believed");
      }
      for (int i = 0; i < 2; ++i) {
        Read r = good;
        r.h[i] = {};
        expect(packVerdict(r.h, groups) == PackRead::Again, "one empty head believed");
      }
      for (int i = 0; i < 2000; ++i) {
        Read r = good;
        r.w[gen() % n] ^= 1u << gen() % 32;
        expect(!packedWordsMatch(r.w.data(), n, r.h[0], E), "one wrong bit in a word believed");
      }
      // words that were packed wrongly: their own sum agrees, the digits' value does not
      for (int i = 0; i < 2000; ++i) {
        Read r = good;
        r.w[gen() % (n - 1)] ^= 1u << gen() % 32;
        uint64_t sum = 0;
        for (uint32_t x : r.w) { sum += x; }
        r.h[0].sum = r.h[1].sum = sum;
        expect(packVerdict(r.h, groups) == PackRead::Words && !packedWordsMatch(r.w.data(), n, r.h[0], E),
               "wrongly packed word believed");
      }
    }
  }
  PackHead h[2] = {};
  expect(packVerdict(h, 200) == PackRead::Again, "a head that nobody wrote taken for a zero residue");
  h[0].groups = h[1].groups = 200;
  expect(packVerdict(h, 200) == PackRead::Zero, "zero");
  h[0].digits = h[1].digits = 3 * uint64_t(0xffffffffu);
  expect(packVerdict(h, 200) == PackRead::Zero, "zero by digits that cancel");
  h[0].digits = h[1].digits = 5;
  expect(packVerdict(h, 200) == PackRead::Again, "zero although the digits are worth something");
  h[0].digits = h[1].digits = 0;
  h[0].sum = h[1].sum = 1;
  expect(packVerdict(h, 200) == PackRead::Again, "zero although words were stored");
  h[0].flags = h[1].flags = PACK_NONZERO | PACK_UNDECIDED;
  expect(packVerdict(h, 200) == PackRead::Host, "undecided");
  h[0].flags = h[1].flags = PACK_NONZERO | PACK_UNDECIDED | PACK_TIMED_OUT;
  expect(packVerdict(h, 200) == PackRead::TimedOut, "timed out");
  expect(packVerdict(h, 199) == PackRead::Again, "another launch's groups");
  if (!bad) { std::printf("OK\n"); }
  return bad != 0;
}
