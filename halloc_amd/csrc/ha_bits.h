// ha_bits.h -- pure bit arithmetic of the wave-run layout, shared by device
// and host code (the host side is unit-tested with g++ against brute force).
#pragma once

#include <cstdint>

#if defined(__HIPCC__) || defined(__HIP__)
#define HA_HD __host__ __device__
#else
#define HA_HD
#endif

namespace ha {

using u32 = uint32_t;
using u64 = uint64_t;

// bit i of x moves to bit f*i (x holds at most 64/f meaningful bits).  Each
// 32-bit half is spread by itself: the shift-or-mask steps are one
// instruction each in 32 bits, and two or more in 64.
HA_HD inline u32 spread_half(u32 x, u32 f) {
  switch (f) {
    case 2:
      x = (x | x << 8) & 0x00FF00FFu;
      x = (x | x << 4) & 0x0F0F0F0Fu;
      x = (x | x << 2) & 0x33333333u;
      return (x | x << 1) & 0x55555555u;
    case 4:
      x = (x | x << 12) & 0x000F000Fu;
      x = (x | x << 6) & 0x03030303u;
      return (x | x << 3) & 0x11111111u;
    case 8:
      x = (x | x << 14) & 0x00030003u;
      return (x | x << 7) & 0x01010101u;
    case 16:
      return (x | x << 15) & 0x00010001u;
    default:  // 32
      return x;
  }
}
HA_HD inline u64 spread_bits(u64 x, u32 f) {
  if (f == 1) return x;
  if (f > 32) return 0;
  const u32 h = 32 / f, m = h >= 32 ? ~0u : (1u << h) - 1;
  return (u64)spread_half((u32)(x >> h) & m, f) << 32 | spread_half((u32)x & m, f);
}

// A run of 64 k-chunk slots starts at chunk s (slot of lane l = s + l*k,
// unwrapped); k is a power of two (1, 2, 4 or 8), so the divisions by k are
// shifts.  s must be a multiple of k (mod 2^32): for other starts the unions
// below are wrong, so a caller that derives s from block positions checks it.  For lane `me` and the lanes in bitmap B, return the unwrapped
// index of the word holding me's slot, the union of B-lanes' fields inside that
// word, and the lowest B-lane in that word (64 if none).
//   bit array:    64 chunks per word, field = k one-bits
//   nibble array: 16 chunks per word, field = 4-bit value `val` (15 or a power
//                 of two) at the slot start
// With j = the slot's place in its word, the word holds the lanes me - j on:
// B shifted there, cut to the word's slots, is the word's lanes slot by slot,
// and spreading them gives the union already in place.
HA_HD inline u64 word_lanes(u64 B, int d) { return d >= 0 ? B >> (d & 63) : B << (-d & 63); }
HA_HD inline void run_word_bits(u64 B, u32 me, u32 s, u32 k, u32& word, u64& uni, u32& issuer) {
  const u32 c = s + me * k;
  word = c >> 6;
  const u32 ks = (u32)__builtin_ctz(k);
  const int d = (int)me - (int)((c & 63u) >> ks);  // lane of the word's first slot
  const u64 x = word_lanes(B, d);
  if (k == 1) {
    uni = x;
    issuer = x ? (u32)(d + (int)__builtin_ctzll(x)) : 64u;
  } else {
    const u32 y = k == 2 ? (u32)x : (u32)x & ((1u << (64u >> ks)) - 1);
    const u64 t = spread_bits(y, k);
    uni = (t << k) - t;  // every slot's first bit widened to k ones
    issuer = y ? (u32)(d + (int)__builtin_ctz(y)) : 64u;
  }
}
HA_HD inline void run_word_nibs(u64 B, u32 me, u32 s, u32 k, u64 val, u32& word, u64& uni,
                                              u32& issuer) {
  const u32 c = s + me * k;
  word = c >> 4;
  const u32 ks = (u32)__builtin_ctz(k);
  const int d = (int)me - (int)((c & 15u) >> ks);
  const u32 y = (u32)word_lanes(B, d) & ((1u << (16u >> ks)) - 1);
  const u64 t = spread_bits(y, 4 * k);
  uni = val == 15 ? (t << 4) - t : t << (u32)__builtin_ctzll(val);
  issuer = y ? (u32)(d + (int)__builtin_ctz(y)) : 64u;
}

// ----------------------------------------------------------- unit fields
// The large-block region keeps one bit per 4 KiB unit in 64-bit words; a block
// of k = 2^c units (k <= 64) is a k-bit field aligned to k inside one word.

// k one-bits (k in 1..64)
HA_HD inline u64 low_mask(u32 k) { return k >= 64 ? ~0ull : ((1ull << k) - 1); }
// one bit at every multiple of k: the start bits of the aligned k-bit fields
HA_HD inline u64 field_starts(u32 k) { return k >= 64 ? 1ull : ~0ull / low_mask(k); }
// start bits of the aligned k-bit fields of v that are entirely zero
HA_HD inline u64 free_fields(u64 v, u32 k) {
  u64 f = ~v;
  for (u32 s = 1; s < k; s <<= 1) f &= f >> s;
  return f & field_starts(k);
}
// start bits of the aligned k-bit fields of v that hold at least one one-bit
HA_HD inline u64 used_fields(u64 v, u32 k) {
  u64 f = v;
  for (u32 s = 1; s < k; s <<= 1) f |= f >> s;
  return f & field_starts(k);
}
// every start bit of b (aligned to k) widened to its k-bit field
HA_HD inline u64 widen_fields(u64 b, u32 k) { return b * low_mask(k); }
// position of the r-th lowest one-bit of x (r < popcount(x))
HA_HD inline u32 select_bit(u64 x, u32 r) {
  u32 pos = 0;
  for (u32 w = 32; w; w >>= 1) {
    const u32 c = (u32)__builtin_popcountll(x & low_mask(w));
    if (r >= c) {
      r -= c;
      x >>= w;
      pos += w;
    }
  }
  return pos;
}
// the n lowest one-bits of x
HA_HD inline u64 lowest_bits(u64 x, u32 n) {
  if (n == 0) return 0;
  if (n >= (u32)__builtin_popcountll(x)) return x;
  return x & low_mask(select_bit(x, n - 1) + 1);
}
// The first word a group of large requests of class c looks at: its ticket
// spread over the nw words by a multiplicative (Fibonacci) hash.
HA_HD inline u32 large_start(u32 ticket, u32 c, u32 nw) {
  const u32 h = (ticket * 0x9E3779B1u) ^ (c * 0x85EBCA77u);
  return (u32)(((u64)h * nw) >> 32);
}

// The largest block (in units) the large region's bit words lb[0..nw) can
// hand out now, over classes 0..ncl-1: a free aligned field inside a word
// for up to 64 units, an aligned run of zero words above.
inline u64 large_max_units(const u64* lb, u32 nw, u32 ncl) {
  u64 best = 0;
  for (u32 c = 0; c < ncl; ++c) {
    bool found = false;
    if (c <= 6) {
      for (u32 w = 0; w < nw && !found; ++w) found = free_fields(lb[w], 1u << c) != 0;
    } else {
      const u32 m = 1u << (c - 6);
      for (u32 g = 0; g + 1 <= nw / m && !found; ++g) {
        bool z = true;
        for (u32 j = 0; j < m && z; ++j) z = lb[(u64)g * m + j] == 0;
        found = z;
      }
    }
    if (!found) break;  // no class above fits either
    best = 1ull << c;
  }
  return best;
}

// x mod n without a division, for x < 2^32 and 1 <= n, given m = mod_magic(n)
// = floor(2^32 / n) (0 for n = 1): q = floor(x * m / 2^32) is floor(x / n) or
// one less, since x * m / 2^32 lies in (x / n - 1, x / n]; one correction step
// finishes
HA_HD inline u32 mod_magic(u32 n) { return n < 2 ? 0u : (u32)(0x100000000ull / n); }
HA_HD inline u32 mod_by(u32 x, u32 n, u32 m) {
  const u32 q = (u32)(((u64)x * m) >> 32);
  u32 r = x - q * n;
  r = r >= n ? r - n : r;
  return n < 2 ? 0u : r;
}

}  // namespace ha
