// Layout of the mirrored column pass's twiddle table (JobDesc::colTab), built by the host in the order
// in which the pass reads it, so that every read of it is coalesced.
#pragma once

// H = C0*C1*C2, forward radices C0, C1, C2, inverse C2, C1, C0. The first LDS entries are copied to LDS:
// product tables with rows of odd stride KS,
//   A: w_(C0*C1)^(p*k), p < C0, 1 <= k < C1, at p*KS + k - 1 (forward stage 1)
//   B: w_(C2*C1)^(p*k), p < C2 (inverse stage 1); A itself when C2 = C0
// then 15 rows of ROOTS entries, w_H^(m*t) for m = 1 ... 15 and t < ROOTS, which thread t reads.
template<int H, int C0, int C1, int C2> struct ColTab {
  static constexpr int KS = (C1 - 1) | 1;
  static constexpr int A = 0;
  static constexpr int B = C0 == C2 ? A : C0 * KS;
  static constexpr int LDS = (C0 == C2 ? C0 : C0 + C2) * KS;
  static constexpr int ROOTS = 256;
};

// The radices of the mirrored pass at height H (0 where there is none).
struct ColRadices {
  int c0, c1, c2;
};
constexpr ColRadices colRadices(int H) {
  switch (H) {
    case 512: return {8, 8, 8};
    case 768: return {8, 12, 8};
    case 1024: return {8, 16, 8};
    case 1152: return {9, 16, 8};
    case 1280: return {10, 16, 8};
    case 1408: return {11, 16, 8};
    case 1536: return {12, 16, 8};
    case 1664: return {13, 16, 8};
    case 1792: return {14, 16, 8};
    case 1920: return {12, 16, 10};
    case 2048: return {16, 16, 8};
    case 2304: return {12, 16, 12};
  }
  if (H >= 2560 && H <= 4096 && H % 256 == 0) { return {16, 16, H / 256}; }
  return {0, 0, 0};
}
// ColTab's LDS for that height (0 where there is no mirrored pass).
constexpr unsigned colTabLds(int H) {
  const ColRadices r = colRadices(H);
  return r.c0 ? unsigned((r.c0 == r.c2 ? r.c0 : r.c0 + r.c2) * ((r.c1 - 1) | 1)) : 0u;
}
// Elements (doubles, or complex where an exchange is not split) of one column's region in the mirrored pass: the
// longest of its exchanges' layouts, rounded up to 16 mod 32 doubles or 8 mod 16 complex elements: the other
// column's region then uses the other half of the LDS banks.
constexpr int colRegionX(int H, bool split) {
  const ColRadices r = colRadices(H);
  if (!r.c0) { return 0; }
  const int a = H / r.c0 * (r.c0 | 1), b = H / r.c2 * (r.c2 | 1), c = H + r.c0 * r.c2;
  const int m = a > b ? (a > c ? a : c) : (b > c ? b : c);
  return split ? (m + 15) / 32 * 32 + 16 : (m + 7) / 16 * 16 + 8;
}
// Its LDS in 16-byte slots: two regions and the product tables.
constexpr unsigned colSlotsX(int H, bool split) { return (split ? 1 : 2) * colRegionX(H, split) + colTabLds(H); }
// Its threads: two columns of butterflies of the stage with the most, whole waves.
constexpr int colThreadsX(int H) {
  const ColRadices r = colRadices(H);
  if (!r.c0) { return 0; }
  const int c = r.c0 < r.c1 ? (r.c0 < r.c2 ? r.c0 : r.c2) : (r.c1 < r.c2 ? r.c1 : r.c2);
  return (2 * (H / c) + 63) / 64 * 64;
}

// Row pass with 16 elements per thread (k_rowm): line strides of its exchanges in elements, and its LDS. Split
// exchanges move doubles (real, then imaginary parts), the others complex elements.
struct RowLayout {
  int l1, l3, l4;  // exchanges 1, 3 and 4 (exchange 2: W)
  int tab;         // 16-byte slots before the product table of 16 rows of ks entries
  int ks, slots;   // slots: all of it, the 64 bytes of round-off values at the end included
};
constexpr int leastMod(int n, int r, int m) { return n + ((r - n) % m + m) % m; }  // least value >= n that is r mod m
constexpr RowLayout rowLayout(int W, int R, int F0, int F1, bool split) {
  RowLayout g{};
  const int u = split ? 16 : 8;  // elements per LDS write cycle; a read serves twice as many
  g.l1 = leastMod(W + W / 16, u / R, u);
  g.l3 = W + W / 16;
  g.l4 = leastMod(W + 16 * F0, 2 * u / R, 2 * u);
  const int l = g.l1 > g.l4 ? (g.l1 > g.l3 ? g.l1 : g.l3) : (g.l4 > g.l3 ? g.l4 : g.l3);
  g.ks = (F1 - 1) | 1;
  g.tab = split ? (R * l + 1) / 2 : R * l;
  g.slots = g.tab + 16 * g.ks + 4;
  return g;
}
