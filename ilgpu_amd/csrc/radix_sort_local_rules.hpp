// The sizes and the arithmetic of the local sort (radix_sort_local.hpp) that need no GPU: plain
// C++, for the kernels, the host code that launches them, and a program that checks them on
// the CPU.
#pragma once

#include <stdint.h>

#include <cmath>

#ifdef __HIPCC__
#define ILGPU_HIP_RULE __host__ __device__
#else
#define ILGPU_HIP_RULE
#endif

namespace ilgpu_hip {

struct LocalBlock {
  static constexpr int kBlock = 256;
  static constexpr int kWaves = kBlock / 64;
  static constexpr int kStageBytes = 36 * 1024;  // four blocks share a compute unit's LDS
  static constexpr int kBinsLog2 = 15;
  static constexpr int kBins = 1 << kBinsLog2;
  // A thread scans 32 words, four bins each; rows of 36 spread a wave's
  // 16-byte accesses over all banks.
  static constexpr int kRowWords = kBins / 4 / kBlock;
  static constexpr int kRowStride = kRowWords + 4;
  static constexpr int kList = 1984;  // bins of two keys or more that a window lists (some 1070 in a full one of random keys)
};
static_assert(LocalBlock::kBlock * LocalBlock::kRowStride * 4 == LocalBlock::kStageBytes, "the counts fill the stage");
// Pairs keep the place a key came from next to it.
constexpr int local_items(int key_bytes, int value_bytes) {
  return LocalBlock::kStageBytes / (key_bytes + (value_bytes > 0 ? 2 : 0)) / LocalBlock::kBlock & ~1;
}
constexpr int local_window(int key_bytes, int value_bytes) {
  return local_items(key_bytes, value_bytes) * LocalBlock::kBlock;
}
constexpr bool local_sorts(int key_bytes, int value_bytes) { return key_bytes >= 4 && value_bytes <= 8; }

// Blocks of the local sort: a compute unit holds four.
inline int64_t local_blocks(int64_t n, int64_t cus) {
  const int64_t of_keys = (n + 1023) / 1024;
  return of_keys < cus * 4 ? of_keys : cus * 4;
}
// Windows and runs that a block may have to put off, at most all of them.  Two windows in a row hold more than one
// full window between them, unless the second ends the block's part.
ILGPU_HIP_RULE constexpr uint32_t local_deferred(uint32_t part, uint32_t window) { return 2 * (part / window) + 6; }
// What the lists of all blocks take, two words an entry.  They lie in the status words of the passes, some 0.11
// bytes per key and more against 0.05; where they would not fit the local sort is not offered.
inline int64_t local_deferred_bytes(int64_t n, int64_t blocks, uint32_t window) {
  return blocks * (int64_t)local_deferred((uint32_t)((n + blocks - 1) / blocks), window) * 8;
}

// ---- draws ---------------------------------------------------------------------
// Whether the local sort can do what passes over the topmost digits leave is asked of m draws,
// one from every m-th part of the input, before anything is counted (radix_sort_impl.hpp:
// sort_draw_kernel, choose_local_digits).
constexpr int kLocalMinDrawBits = 12, kLocalMaxDrawBits = 16;
constexpr int kLocalChunkBits = 14;   // draws that the block that looks at them holds at a time
constexpr int kLocalPartBits = 13;    // draws of one part of the values
constexpr int kLocalPrefixBits = 15;  // draws whose prefixes are counted
constexpr int local_draw_bits(int64_t n) {
  return n <= 1ll << 21 ? kLocalMinDrawBits : (n <= 1ll << 23 ? 13 : (n <= 1ll << 25 ? 14 : kLocalMaxDrawBits));
}
// Parts of the values, and those whose draws are asked whether they meet: as many as the block has time for while
// others count the keys, some 37 us each with 2^16 draws.  (All four of 2^27 + 1 u32 keys 1063 -> 1129 us, both
// of 10^7 150 -> 162, one of 2^28 takes a column of six copies of every value one time in nine.)
constexpr int local_parts(int draw_bits) { return draw_bits > kLocalPartBits ? 1 << (draw_bits - kLocalPartBits) : 1; }
constexpr int local_parts_asked(int64_t n, int draw_bits) {
  const int64_t parts = n >> 26 < 1 ? 1 : n >> 26;
  return parts < local_parts(draw_bits) ? (int)parts : local_parts(draw_bits);
}
// A random place in part s of 2^bits.
ILGPU_HIP_RULE inline uint64_t local_draw_place(uint64_t s, int bits, uint64_t n) {
  uint64_t z = (s + 1ull) * 0x9E3779B97F4A7C15ull;  // splitmix64
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  const uint64_t at = (s << 32 | (uint32_t)z) << (32 - bits);
  return (uint64_t)(((unsigned __int128)at * n) >> 64);
}
// Where it is kept: every chunk holds draws from all over the input.  (Not all the questions look at all
// chunks.  With the parts in a row, columns filled in front and padded behind passed: 2^28 u32 keys of which the
// second half was the same, a second on one compute unit instead of 2.3 ms.)
ILGPU_HIP_RULE constexpr uint32_t local_draw_slot(uint32_t s, int bits) {
  return bits <= kLocalChunkBits ? s : (s & ((1u << (bits - kLocalChunkBits)) - 1u)) << kLocalChunkBits |
                                           s >> (bits - kLocalChunkBits);
}

// What the draws may show.
struct LocalLimits {
  uint32_t draw_bits;  // log2 of the number of draws
  uint32_t bin_bits;   // of a draw, from the topmost bit that differs on
  uint32_t parts;      // of the values, that are asked
  uint32_t max_equal;  // draws of these that meet an earlier one in these bits
  uint32_t max_pairs;  // pairs of draws that share a 16-bit prefix (0: one digit makes runs that may fit a window,
                       // which its counts tell)
  uint32_t max_draws;  // of one prefix
  uint32_t max_run;    // keys of a run of one digit (0: two digits)
};
inline LocalLimits local_limits(int64_t keys, int key_bytes, int value_bytes) {
  const int64_t window = local_window(key_bytes, value_bytes);
  LocalLimits limits{};
  limits.draw_bits = (uint32_t)local_draw_bits(keys);
  const double draws = (double)(1ll << limits.draw_bits), n = (double)keys;
  while (limits.bin_bits < 31 && keys >> limits.bin_bits != 0) ++limits.bin_bits;  // log2(n) + 1
  const int parts = local_parts((int)limits.draw_bits);
  limits.parts = (uint32_t)local_parts_asked(keys, (int)limits.draw_bits);
  const bool one_digit = keys <= window * 256 * 15 / 16;
  const double most_equal = (key_bytes == 4 && !one_digit ? 0.9 : 1.25) * draws * draws / n;
  limits.max_equal = ((uint32_t)most_equal + 6u) * limits.parts / (uint32_t)parts;
  if (one_digit) {
    limits.max_run = (uint32_t)window;
  } else {
    // Runs of 0.6 windows, as the mean over the keys.  (With 0.95, with a copy in front, us, every digit / the local sort: 2^29
    // u32 keys 4556 / 3968, but two copies of every value, which 2^16 draws hardly show at that length, 4560 / 8571; 450 * 2^20
    // 4011 / 3531 and 4008 / 7755; u32 pairs of 300 * 2^20 5043 / 4076, two copies of 260 * 2^20 4367 / 4419.  Those were
    // windows whose list ran over going the slow way.)
    const double looked_at = std::fmin(draws, (double)(1ll << kLocalPrefixBits));
    limits.max_pairs = (uint32_t)(looked_at * looked_at * 0.5 * (0.6 * (double)window / n)) + 1u;
    const double of_window = looked_at * (double)window / n;
    const double most = of_window + 5.0 * std::sqrt(of_window) + 6.0;
    limits.max_draws = most < 100.0 ? (uint32_t)most : 100u;
  }
  return limits;
}

// Two digits are refused by their exact counts where the draws may have missed a long run, which is one
// block's: one of L keys adds L to the count of its lower digit, and other keys spread over that digit
// evenly where their runs are short.  `most_upper` and `most_lower`: keys of the most frequent upper and lower digit.
// A block takes 3 ns for a key of 4 bytes and 11 for one of 8, once a run is longer than a window; n / 4096
// keys are half of what the local sort gains.  Whatever the keys are, no run is longer than n / 256 and that.
// The 256 runs of an upper digit are longer than a window if it has 256 windows.
ILGPU_HIP_RULE constexpr bool local_counts_allow(uint32_t n, uint32_t most_upper, uint32_t most_lower,
                                                 uint32_t window) {
  return most_upper <= (uint64_t)window * 256 && most_lower <= n / 256 + (window > n / 4096 ? window : n / 4096);
}

// ---- bins -------------------------------------------------------------------
// bin = ((key - low) >> shift) * scale >> 16: the shift leaves 18 bits, the scale spreads
// what they hold over all the bins.  Keys of the window, up to low + span, have bins below kBins; others
// may have any 16-bit number.
struct LocalScale {
  int shift;
  uint32_t scale;
};
template <typename K>
ILGPU_HIP_RULE inline LocalScale local_scale(K span) {
  const int span_bits = sizeof(K) == 8 ? 64 - __builtin_clzll((uint64_t)span | 1ull)
                                       : 32 - __builtin_clz((uint32_t)span | 1u);
  LocalScale s;
  s.shift = span_bits > 18 ? span_bits - 18 : 0;
  s.scale = 0x7FFFFFFFu / ((uint32_t)(span >> s.shift) + 1u);
  if (s.scale > 1u << 16) s.scale = 1u << 16;
  return s;
}

// A bin's code: the byte offset of its word in the stage, and in the lowest two bits which of the word's
// four counts it is.  16 bits: two bins at once as a vector of them.
template <typename Bins>
ILGPU_HIP_RULE constexpr Bins local_bin_codes(Bins bins) {
  return (Bins)((Bins)((Bins)(bins >> (uint16_t)7) * (uint16_t)16) + bins);
}
static_assert((LocalBlock::kRowStride - LocalBlock::kRowWords) * 4 == 16 && LocalBlock::kRowWords * 4 == 1 << 7,
              "a row of 2^7 bins is followed by 16 bytes of nothing");
static_assert(local_bin_codes<uint32_t>(LocalBlock::kBins - 1) / 4 * 4 + 4 <= (uint32_t)LocalBlock::kStageBytes,
              "every bin's word lies in the stage");
// Two keys' codes, without that of the first (0) or the second (1): where a thread holds no key of the window, the
// first bin stands for it (the number it has may lie outside of the stage).
ILGPU_HIP_RULE constexpr uint32_t local_codes_without(uint32_t codes, int which) {
  return codes & (which == 0 ? 0xFFFF0000u : 0x0000FFFFu);
}

}  // namespace ilgpu_hip
