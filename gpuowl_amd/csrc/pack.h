// What the host makes of a residue packed or unpacked on the device (k_pack, k_unpack): nothing that was read from the
// device is believed unless something else says the same.
#pragma once

#include <cstdint>
#include <cstring>

// The kernels write it twice, from different lanes to different addresses, and both are read.
struct PackHead {
  uint64_t sum;     // of the packed words, as they were stored
  uint64_t digits;  // of the digits' values mod 2^32 - 1, by groups that read the digits on their own
  uint32_t flags;   // PACK_*
  uint32_t groups;  // that have reported
  uint64_t pad;
};
enum {
  PACK_NONZERO = 1,    // a digit is not zero
  PACK_UNDECIDED = 2,  // a carry or a digit is the host's to decide
  PACK_TIMED_OUT = 4,  // JobDesc::flags[2]
  PACK_NEGATIVE = 8,   // the digits' value is negative
};

enum class PackRead {
  Again,     // not what the kernel wrote
  TimedOut,  // a carry hand-off timed out
  Zero,
  Host,      // the host converts the digits itself
  Words,     // as packed, if packedWordsMatch
};

// Whether both heads are what a launch of so many groups leaves.
inline bool packHeadsAgree(const PackHead (&h)[2], uint32_t groups) {
  return memcmp(&h[0], &h[1], sizeof(PackHead)) == 0 && h[0].groups == groups;
}

inline PackRead packVerdict(const PackHead (&h)[2], uint32_t groups) {
  const PackHead& a = h[0];
  if (!packHeadsAgree(h, groups)) { return PackRead::Again; }
  if (a.flags & PACK_TIMED_OUT) { return PackRead::TimedOut; }
  if (!(a.flags & PACK_NONZERO)) { return a.sum || a.digits % 0xffffffffu ? PackRead::Again : PackRead::Zero; }
  return a.flags & PACK_UNDECIDED ? PackRead::Host : PackRead::Words;
}

// Whether the n words that reached the host are those the kernel stored (by their sum) and have the digits' value, to
// which 2^E - 1 has come where it is negative. Mod 2^32 - 1 a word counts as it is.
inline bool packedWordsMatch(const uint32_t* w, uint32_t n, const PackHead& h, uint32_t E) {
  constexpr uint64_t M = 0xffffffffu;
  uint64_t sum = 0;
  for (uint32_t i = 0; i < n; ++i) { sum += w[i]; }
  const uint64_t wrap = h.flags & PACK_NEGATIVE ? (uint64_t(1) << E % 32) - 1 : 0;
  return sum == h.sum && sum % M == (h.digits + wrap) % M;
}
