// Layout of the mirrored column pass's twiddle table (JobDesc::colTab), built by the host in the order
// in which the pass reads it, so that every read of it is coalesced.
#pragma once

// H = C0*C1*C2, forward radices C0, C1, C2, inverse C2, C1, C0. The first LDS entries are copied to LDS:
// product tables with rows of odd stride KS,
//   A: w_(C0*C1)^(p*k), p < C0, 1 <= k < C1, at p*KS + k - 1 (forward stage 1)
//   B: w_(C2*C1)^(p*k), p < C2 (inverse stage 1); A itself when C2 = C0
// then six rows of ROOTS entries, w_H^(m*t) for m = 1, 2, 3, 4, 8, 12 and t < ROOTS, which thread t reads.
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
