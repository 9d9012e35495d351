// The sizes and the arithmetic of the local sort (radix_sort_local.hpp) that need no GPU: plain
// C++, for the kernels, the host code that launches them, and a program that checks them on
// the CPU.
#pragma once

#include <stdint.h>

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
  static constexpr int kList = 1984;  // bins of two keys or more that a window may have (some 1070 in a full one)
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
