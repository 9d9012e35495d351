// The sizes and the arithmetic of the local sort as plain functions, for tests/test_local_sort_rules.py.
#include "../../ilgpu_amd/csrc/radix_sort_local_rules.hpp"

using namespace ilgpu_hip;

extern "C" {

int32_t rule_window(int32_t key_bytes, int32_t value_bytes) { return local_window(key_bytes, value_bytes); }
int32_t rule_stage_bytes() { return LocalBlock::kStageBytes; }

int64_t rule_blocks(int64_t n, int64_t cus) { return local_blocks(n, cus); }
uint32_t rule_deferred(uint32_t part, uint32_t window) { return local_deferred(part, window); }
int64_t rule_deferred_bytes(int64_t n, int64_t blocks, uint32_t window) {
  return local_deferred_bytes(n, blocks, window);
}

// The draws of n keys: their places in the input and where they are kept; the number of them.
int32_t rule_draws(int64_t n, uint64_t* places, uint32_t* slots) {
  const int bits = local_draw_bits(n);
  for (uint32_t s = 0; s < 1u << bits; ++s) {
    places[s] = local_draw_place(s, bits, (uint64_t)n);
    slots[s] = local_draw_slot(s, bits);
  }
  return 1 << bits;
}
int32_t rule_chunk_draws() { return 1 << kLocalChunkBits; }
int32_t rule_prefix_draws() { return 1 << kLocalPrefixBits; }
int32_t rule_parts(int32_t draw_bits) { return local_parts(draw_bits); }
void rule_limits(int64_t n, int32_t key_bytes, int32_t value_bytes, uint32_t* out) {
  const LocalLimits limits = local_limits(n, key_bytes, value_bytes);
  const uint32_t all[] = {limits.draw_bits, limits.bin_bits,  limits.parts,  limits.max_equal,
                          limits.max_pairs, limits.max_draws, limits.max_run};
  for (int i = 0; i < 7; ++i) out[i] = all[i];
}

int32_t rule_counts_allow(uint32_t n, uint32_t most_upper, uint32_t most_lower, uint32_t window) {
  return local_counts_allow(n, most_upper, most_lower, window);
}

// The codes of two keys' bins in a window whose keys are up to `span` behind its lowest, as the kernel
// packs them; has_key: bit 0 the first, bit 1 the second key is one of the window.
uint32_t rule_codes(int32_t key_bytes, uint64_t span, uint64_t first, uint64_t second, int32_t has_key) {
  const LocalScale s = key_bytes == 8 ? local_scale<uint64_t>(span) : local_scale<uint32_t>((uint32_t)span);
  uint32_t codes = 0;
  for (int which = 0; which < 2; ++which) {
    const uint64_t key = which == 0 ? first : second;
    const uint32_t shifted = key_bytes == 8 ? (uint32_t)(key >> s.shift) : (uint32_t)key >> s.shift;
    const uint32_t scaled = (shifted & 0xFFFFFFu) * s.scale;  // 24 bits times 17
    codes |= (uint32_t)local_bin_codes<uint16_t>((uint16_t)(scaled >> 16)) << (16 * which);
  }
  for (int which = 0; which < 2; ++which)
    if (!(has_key >> which & 1)) codes = local_codes_without(codes, which);
  return codes;
}

}  // extern "C"
