#include "TrigBufCache.h"

#include "Trig.h"
#include "coltab.h"

#include <map>
#include <mutex>
#include <tuple>
#include <vector>

namespace {
double2 d2(std::pair<double, double> p) { return double2{p.first, p.second}; }

// The entries of ColTab<H, C0, C1, C2> (coltab.h).
std::vector<double2> colTabOf(u32 H) {
  const ColRadices r = colRadices(H);
  if (!r.c0) { return {}; }
  const u32 KS = (r.c1 - 1) | 1, ROOTS = 256;
  std::vector<double2> t(colTabLds(H) + 6 * ROOTS, double2{0, 0});
  auto product = [&](u32 at, u32 rows, u32 n) {  // w_n^(p*k), p < rows, 1 <= k < C1
    for (u32 p = 0; p < rows; ++p) {
      for (u32 k = 1; k < u32(r.c1); ++k) { t[at + p * KS + k - 1] = d2(root1(n, p * k)); }
    }
  };
  product(0, r.c0, r.c0 * r.c1);
  if (r.c2 != r.c0) { product(r.c0 * KS, r.c2, r.c2 * r.c1); }
  const u32 m[6] = {1, 2, 3, 4, 8, 12};
  for (u32 i = 0; i < 6; ++i) {
    for (u32 k = 0; k < ROOTS; ++k) { t[colTabLds(H) + i * ROOTS + k] = d2(root1(H, m[i] * k)); }
  }
  return t;
}
}  // namespace

std::shared_ptr<const TrigTables> TrigBufCache::get(u32 W, u32 H, bool oneRegion, owl_queue q) {
  static std::mutex mtx;
  static std::map<std::tuple<u32, u32, bool>, std::weak_ptr<const TrigTables>> cache;
  std::lock_guard<std::mutex> lock(mtx);
  auto key = std::make_tuple(W, H, oneRegion);
  if (auto it = cache.find(key); it != cache.end()) {
    if (auto sp = it->second.lock()) { return sp; }
  }
  const u32 ND = W * H;
  const u32 nHi = (H + 63) / 64;
  std::vector<double2> row(W), col(H), midA(size_t(W) * 64), midB(size_t(W) * nHi), pair(W), mid(size_t(W) * 16);
  for (u32 m = 0; m < W; ++m) { row[m] = d2(root1(W, m)); }
  for (u32 m = 0; m < H; ++m) { col[m] = d2(root1(H, m)); }
  for (u32 a = 0; a < W; ++a) {
    pair[a] = d2(root1(ND, a));
    for (u32 lo = 0; lo < 64; ++lo) { midA[size_t(a) * 64 + lo] = d2(root1(ND, u64(a) * lo)); }
    for (u32 hi = 0; hi < nHi; ++hi) { midB[size_t(a) * nHi + hi] = d2(root1(ND, u64(a) * 64 * hi % ND)); }
  }
  auto t = std::make_shared<TrigTables>();
  t->row = Buffer<double2>(q, row);
  t->col = Buffer<double2>(q, col);
  t->midA = Buffer<double2>(q, midA);
  t->midB = Buffer<double2>(q, midB);
  t->pair = Buffer<double2>(q, pair);
  const u32 c0 = oneRegion ? 16 : colRadices(H).c0;
  if (c0) {
    for (u32 a = 0; a < W; ++a) {
      for (u32 k = 0; k < 16; ++k) { mid[size_t(a) * 16 + k] = d2(root1(ND, u64(a) * k * (H / c0) % ND)); }
    }
    (oneRegion ? t->midS : t->midM) = Buffer<double2>(q, mid);
    if (!oneRegion) { t->colTab = Buffer<double2>(q, colTabOf(H)); }
  }
  cache[key] = t;
  return t;
}
