#include "TrigBufCache.h"

#include "Trig.h"
#include "coltab.h"

#include <map>
#include <mutex>
#include <tuple>
#include <vector>

namespace {
double2 d2(std::pair<double, double> p) { return double2{p.first, p.second}; }

// The entries of ColTab<H, C0, C1, C2> (coltab.h), from the H-th roots.
std::vector<double2> colTabOf(u32 H, const std::vector<double2>& roots) {
  const ColRadices r = colRadices(H);
  if (!r.c0) { return {}; }
  const u32 KS = (r.c1 - 1) | 1, ROOTS = 256;
  std::vector<double2> t(colTabLds(H) + 15 * ROOTS, double2{0, 0});
  auto product = [&](u32 at, u32 rows, u32 n) {  // w_n^(p*k), p < rows, 1 <= k < C1
    for (u32 p = 0; p < rows; ++p) {
      for (u32 k = 1; k < u32(r.c1); ++k) { t[at + p * KS + k - 1] = roots[p * k * (H / n)]; }
    }
  };
  product(0, r.c0, r.c0 * r.c1);
  if (r.c2 != r.c0) { product(r.c0 * KS, r.c2, r.c2 * r.c1); }
  for (u32 m = 0; m < 15; ++m) {
    for (u32 k = 0; k < ROOTS; ++k) { t[colTabLds(H) + m * ROOTS + k] = roots[(m + 1) * k % H]; }
  }
  return t;
}
}  // namespace

std::shared_ptr<const TrigTables> TrigBufCache::get(u32 W, u32 H, ColKind kind, owl_queue q) {
  static std::mutex mtx;
  static std::map<std::tuple<u32, u32, ColKind>, std::weak_ptr<const TrigTables>> cache;
  std::lock_guard<std::mutex> lock(mtx);
  auto key = std::make_tuple(W, H, kind);
  if (auto it = cache.find(key); it != cache.end()) {
    if (auto sp = it->second.lock()) { return sp; }
  }
  const u32 ND = W * H;
  auto t = std::make_shared<TrigTables>();
  // n entries exp(-2 pi i f(i) / L)
  auto table = [&](u32 n, u32 L, auto f) {
    std::vector<double2> v(n);
    for (u32 i = 0; i < n; ++i) { v[i] = d2(root1(L, f(i))); }
    return Buffer<double2>(q, v);
  };
  t->row = table(W, W, [](u32 m) { return u64(m); });
  std::vector<double2> colRoots(H);
  for (u32 m = 0; m < H; ++m) { colRoots[m] = d2(root1(H, m)); }
  t->col = Buffer<double2>(q, colRoots);
  t->pair = table(W, ND, [](u32 a) { return u64(a); });
  if (kind != ColKind::Mirrored) {
    const u32 nHi = (H + 63) / 64;
    t->midA = table(W * 64, ND, [](u32 i) { return u64(i / 64) * (i % 64); });
    t->midB = table(W * nHi, ND, [=](u32 i) { return u64(i / nHi) * 64 * (i % nHi); });
    if (kind == ColKind::OneRegion) {
      t->midS = table(W * 16, ND, [=](u32 i) { return u64(i / 16) * (i % 16) * (H / 16); });
    }
  } else {
    const u32 NB0 = H / colRadices(H).c0, rows = W / 2 + 1, nHi = (NB0 + 63) / 64;
    t->midM = table(W * 16, ND, [=](u32 i) { return u64(i / 16) * (i % 16) * NB0; });
    t->colTab = Buffer<double2>(q, colTabOf(H, colRoots));
    // midBase: products of two factors with their low parts, rounded once, on the device: per row 64 low factors
    // exp(-2 pi i a*lo / ND) and nHi high ones, each with its low part after it
    const u32 per = 2 * (64 + nHi);
    std::vector<double2> f(size_t(rows) * per);
    for (u32 a = 0; a < rows; ++a) {
      for (u32 i = 0; i < 64 + nHi; ++i) {
        const u64 k = i < 64 ? u64(a) * i : u64(a) * 64 * (i - 64);
        const RootParts r = root1Parts(ND, k);
        f[size_t(a) * per + 2 * i] = d2(r.high);
        f[size_t(a) * per + 2 * i + 1] = d2(r.low);
      }
    }
    Buffer<double2> factors(q, f);
    t->midBase = Buffer<double2>(size_t(rows) * NB0);
    owl_kernel k = nullptr;
    owlCheck(owl_hip_kernel_get("midBase", &k), "kernel");
    double2* out = t->midBase.get();
    const double2* in = factors.get();
    u32 nb0 = NB0, n = rows * NB0, nh = nHi;
    void* args[] = {&out, &in, &nb0, &nh, &n};
    owlCheck(owl_hip_launch(q, k, (n + 255) / 256, 1, 256, 0, args), "midBase");
    owlCheck(owl_hip_finish(q), "midBase");
  }
  cache[key] = t;
  return t;
}
