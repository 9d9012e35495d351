// Radix sort of keys and key/value pairs: onesweep LSD sort, 8-bit digits.
//
// Stands in for the RadixSort / RadixSortPairs delegates of
// RadixSortExtensions.cs:1017-1337.  The reference runs NumBits/2 passes of
// {memset, local 4-way split, counter scan, scatter} (:1276-1334) and packs
// pairs into an array of structs first (:1057-1072).  Here a sort of k-byte
// keys is
//
//   zero      clears the global digit histograms, tile tickets and look-back
//             status words (one launch), and draws keys where the local sort is
//             offered;
//   histogram one read of the keys builds the 256-bin histogram of every digit
//             position in LDS (replicated counters) and adds it to global; from
//             8-byte keys it also draws a sample of upper halves, and one block
//             of it looks at the draws for the local sort;
//   plan      one block turns the histograms into exclusive digit offsets,
//             marks passes whose digit is the same for every key (they are
//             skipped), is left to the local sort since passes over the one or two
//             topmost digits make short runs, or to the ties since the upper halves
//             drawn rarely meet, and records which buffer each pass reads;
//   pass x k  onesweep: a block takes a tile by ticket, ranks its keys (one
//             returning LDS add per key on per-wave digit counters; the LDS
//             serves the lanes of an instruction in lane order, so equal digits
//             keep memory order: every pass is stable), publishes
//             its 256 digit counts, resolves the counts of all earlier tiles by
//             decoupled look-back, stages the tile in digit order through LDS
//             and writes each digit's run to its final place;
//   finish    copies the result back if an odd number of passes ran; after
//             passes over the topmost digits it sorts the runs of keys that agree
//             in them, a window of whole runs at a time in LDS (local_sort_kernel,
//             radix_sort_local.hpp); after passes over the upper half of 8-byte keys it
//             orders the runs of keys that share one (ties_kernel).
//
// Keys and values stay in separate arrays (structure of arrays); a value
// travels with its key through the same tile-local permutation.
//
// Key order: digit(k) = ((k ^ xor_mask ^ f(k)) >> shift) & 0xFF, where
// xor_mask folds the sign-bit flip of signed/float types and the complement
// of Descending* (RadixSortOperations.tt:77-93, 122-123) and f(k) is the
// per-key term of the float transforms.  Float keys are converted once, by the
// first pass that runs, and converted back by the last one.
//
// Algorithmic HBM traffic for n keys of k bytes, values of v bytes and P
// executed passes: n * (k * (2P + 1) + v * 2P) bytes, n * k where ties are left, and
// 2 n (k + v) where the local sort follows.
//
// This header holds the kernels and their launch code as templates; one
// translation unit per key size (radix_sort_k1/2/4/8.hip) instantiates them, so
// that the key sizes compile side by side, and radix_sort.hip holds what does
// not depend on the key size.  (A kernel has to be defined in the translation
// unit that launches it, hence a header and not a library of kernels.)
#pragma once

#include <hip/hip_fp16.h>

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "kernels.hpp"
#include "radix_sort_local_rules.hpp"

namespace ilgpu_hip {

// Process-wide sort parameters (ilgpu_hip_sort_set_parameter), defined in
// radix_sort.hip.
extern std::atomic<uint32_t> g_sort_spin_limit;
extern std::atomic<int32_t> g_sort_large_min_tiles_per_cu;  // negative: the defaults
extern std::atomic<int32_t> g_sort_small_kernel;            // 0: one-tile inputs take the passes too
extern std::atomic<int32_t> g_sort_short_tile_max_tiles;    // negative: the default

namespace {

constexpr int kRadix = 256;
constexpr int kMaxPasses = 8;
// Launch shape of the onesweep pass.  The block size fixes the number of
// per-wave sub-tiles (and with it the LDS footprint of the ranking counters);
// items per thread fix the tile size.
#ifndef ILGPU_HIP_SORT_BLOCK
#define ILGPU_HIP_SORT_BLOCK 512
#endif
#ifndef ILGPU_HIP_SORT_ITEMS
#define ILGPU_HIP_SORT_ITEMS 36
#endif
#ifndef ILGPU_HIP_SORT_ITEMS8
#define ILGPU_HIP_SORT_ITEMS8 18
#endif
#ifndef ILGPU_HIP_SORT_PAIR_ITEMS2
#define ILGPU_HIP_SORT_PAIR_ITEMS2 16
#endif
#ifndef ILGPU_HIP_SORT_PAIR_ITEMS4
#define ILGPU_HIP_SORT_PAIR_ITEMS4 10
#endif
#ifndef ILGPU_HIP_SORT_PAIR_ITEMS3
#define ILGPU_HIP_SORT_PAIR_ITEMS3 14
#endif
#ifndef ILGPU_HIP_SORT_LOOKBACK
#define ILGPU_HIP_SORT_LOOKBACK 4
#endif
// Rows whose LDS operations are in flight together while ranking, and staged
// keys a thread reads per batch of the write-out.
#ifndef ILGPU_HIP_SORT_RANK_GROUP
#define ILGPU_HIP_SORT_RANK_GROUP 6
#endif
#ifndef ILGPU_HIP_SORT_PAIR_RANK_GROUP
#define ILGPU_HIP_SORT_PAIR_RANK_GROUP 2
#endif
#ifndef ILGPU_HIP_SORT_PAIR_WRITE_GROUP
#define ILGPU_HIP_SORT_PAIR_WRITE_GROUP 4
#endif
// Tiles are handed out in chunks of consecutive tiles, one chunk at a time to
// each of kTicketGroups groups of blocks (block b is in group b % 8: blocks are
// dispatched round-robin over the eight XCDs, so a group is the blocks of one
// XCD).  Neighbouring tiles write neighbouring runs; when they run on one XCD
// the partially written lines between their runs merge in that XCD's L2.
#ifndef ILGPU_HIP_SORT_MAX_CHUNK_SHIFT
#define ILGPU_HIP_SORT_MAX_CHUNK_SHIFT 3
#endif
constexpr int kTicketGroups = 8;
constexpr int kTicketStride = 32;          // words: one 128-byte line per group
constexpr int kMaxChunkShift = ILGPU_HIP_SORT_MAX_CHUNK_SHIFT;
// Polls of an empty status word before a look-back stops waiting for the tile
// and counts its digit itself.
constexpr uint32_t kDefaultSpinLimit = 4096;
#ifndef ILGPU_HIP_SORT_WRITE_GROUP
#define ILGPU_HIP_SORT_WRITE_GROUP 12
#endif
// Two block sizes.  Large inputs take 1024-thread blocks, one per compute unit:
// twice the tile, so every digit's run is twice as long (it is run length that
// the scattered writes pay for, pairs above all, whose tiles are short), and
// half as many tiles to chain.  Smaller inputs take 512-thread blocks, two per
// compute unit, which fill the GPU with fewer keys.
constexpr int kSortBlock = ILGPU_HIP_SORT_BLOCK;      // small inputs, and the self-test
constexpr int kSortBlockLarge = 1024;
// The large block is used from this many of its tiles per compute unit on.
// Keys without values take the pipelined pass there, measured against the
// 512-thread classic pass on u32 keys (ms per sort): 2^24.6 keys (2.7 tiles
// per CU) 0.291 / 0.277, 2^25 (3.6) 0.328 / 0.347, 2^25.6 (5.3) 0.461 / 0.480,
// 2^26 (7.1) 0.572 / 0.617, 2^27 1.040 / 1.136.  The classic 1024-thread pass
// (ILGPU_HIP_SORT_PIPELINED=0) pays from ten tiles per CU on; pairs of u64 keys
// and u32 values gain 4 to 8 % from 2^23 pairs on.
#ifndef ILGPU_HIP_SORT_PIPELINED
#define ILGPU_HIP_SORT_PIPELINED 1
#endif
constexpr int kLargeMinTilesPerCuKeys = ILGPU_HIP_SORT_PIPELINED ? 3 : 10;
constexpr int kLargeMinTilesPerCuPairs = 2;
// Lanes that rank together (a sub-tile row): one wave.
constexpr int kSubLanes = kWaveSize;
constexpr int kLookback = ILGPU_HIP_SORT_LOOKBACK;
#ifndef ILGPU_HIP_SORT_HIST_BLOCK
#define ILGPU_HIP_SORT_HIST_BLOCK 512
#endif
#ifndef ILGPU_HIP_SORT_HIST_BLOCKS_PER_CU
#define ILGPU_HIP_SORT_HIST_BLOCKS_PER_CU 2
#endif
#ifndef ILGPU_HIP_SORT_HIST_RUNS
#define ILGPU_HIP_SORT_HIST_RUNS 1
#endif
#ifndef ILGPU_HIP_SORT_HIST_NT
#define ILGPU_HIP_SORT_HIST_NT 1
#endif
#ifndef ILGPU_HIP_SORT_HIST_UNROLL
#define ILGPU_HIP_SORT_HIST_UNROLL 2
#endif
constexpr int kHistUnroll = ILGPU_HIP_SORT_HIST_UNROLL;
constexpr int kHistBlock = ILGPU_HIP_SORT_HIST_BLOCK;
#ifndef ILGPU_HIP_SORT_HIST_LDS_WORDS
#define ILGPU_HIP_SORT_HIST_LDS_WORDS 16384
#endif
constexpr int kHistLdsWords = ILGPU_HIP_SORT_HIST_LDS_WORDS;
// Look-back status word of a (tile, digit): 0 = nothing published yet;
// top bits 11 = the tile's own count in the low 30 bits (a count is at most a
// tile); anything else = inclusive count over all tiles up to this one, plus
// one.  An inclusive count is at most n <= 2^31 - 1, so count + 1 <= 2^31
// never has both top bits set and is never 0.
constexpr uint32_t kStatusAggregate = 3u << 30;
constexpr uint32_t kStatusCountMask = (1u << 30) - 1u;
__device__ __forceinline__ uint32_t status_aggregate(uint32_t count) {
  return kStatusAggregate | count;
}
__device__ __forceinline__ uint32_t status_prefix(uint32_t inclusive) { return inclusive + 1u; }
__device__ __forceinline__ bool status_is_aggregate(uint32_t w) {
  return (w & kStatusAggregate) == kStatusAggregate;
}
// Value of a non-empty word and whether it ends the look-back.
__device__ __forceinline__ uint32_t status_value(uint32_t w) {
  return status_is_aggregate(w) ? w & kStatusCountMask : w - 1u;
}
// Where all tiles of a pass run at once (a grid of as many blocks as there are tiles) nothing is published
// but counts: a tile's own, as above, and by the last tile of kLookGroup tiles, in place of its own, theirs
// together, with the top bits 10.
constexpr int kLookGroup = 16;
constexpr uint32_t kStatusGroup = 2u << 30;
__device__ __forceinline__ uint32_t status_group(uint32_t count) { return kStatusGroup | count; }
__device__ __forceinline__ bool status_is_group(uint32_t w) { return (w & kStatusAggregate) == kStatusGroup; }
constexpr int64_t kMaxSortLength = 0x7fffffffll;  // like the reference: int.MaxValue

template <int KEY_BYTES> struct KeyOf;
template <> struct KeyOf<1> { using type = uint8_t; };
template <> struct KeyOf<2> { using type = uint16_t; };
template <> struct KeyOf<4> { using type = uint32_t; };
template <> struct KeyOf<8> { using type = uint64_t; };

struct alignas(16) Bytes16 { uint32_t x, y, z, w; };
template <int VALUE_BYTES> struct ValueOf { using type = uint8_t; };
template <> struct ValueOf<2> { using type = uint16_t; };
template <> struct ValueOf<4> { using type = uint32_t; };
template <> struct ValueOf<8> { using type = uint64_t; };
template <> struct ValueOf<16> { using type = Bytes16; };

// The value a sequencer gives element i (Sequencers.tt:25-37, Sequencer.cs:36-75):
// mode 1 = the integer sequencers and IndexSequencer, (T)i with T as wide as the
// value; mode 2 = HalfSequencer, FloatSequencer and DoubleSequencer, (T)i in
// floating point (long to float rounds to nearest even, Half goes through
// float as the C# conversion does).
template <int VALUE_BYTES>
__device__ __forceinline__ typename ValueOf<VALUE_BYTES>::type index_value(int64_t i, int mode) {
  using Val = typename ValueOf<VALUE_BYTES>::type;
  if constexpr (VALUE_BYTES == 1) {
    return (Val)(uint8_t)i;
  } else if constexpr (VALUE_BYTES == 2) {
    if (mode == 2) return (Val)__half_as_ushort(__float2half((float)i));
    return (Val)(uint16_t)i;
  } else if constexpr (VALUE_BYTES == 4) {
    if (mode == 2) return (Val)__float_as_uint((float)i);
    return (Val)(uint32_t)i;
  } else if constexpr (VALUE_BYTES == 8) {
    if (mode == 2) return (Val)(uint64_t)__double_as_longlong((double)i);
    return (Val)(uint64_t)i;
  } else {
    return Val{};  // 16-byte values are never generated (refused by the entry point)
  }
}

// Keys per thread and tile.  Long tiles pay: the runs they scatter are longer
// (fewer partial cache lines) and there are fewer tiles to chain.  Keys-only
// sorts take 36 keys of up to 4 bytes or 18 of 8 bytes per thread: the most
// that the 160 KiB of LDS of a compute unit stage for sixteen waves.  Values
// live in registers next to the keys, which caps pairs lower, by the registers
// one pair takes: at two (key and value of up to 4 bytes each) 16 items with
// 4-byte values and 20 with shorter ones, 14 at three, 10 at four, 8 with
// 16-byte values.  (Measured per pass on 2^27 pairs with 1024-thread blocks:
// u32 + u32 at 16 / 18 / 20 / 24 items 0.470 / 0.486 / 0.486 / 0.972 ms; u64 +
// u32 at 10 / 12 / 14 / 16 / 18 items 0.714 / 0.681 / 0.667 / 0.702 / 0.691;
// u64 + u64 at 10 / 12 / 14 items 0.902 / 0.919 / 0.947; u32 + u8 at 16 / 18 /
// 20 items 0.597 / 0.594 / 0.579.)
constexpr int items_per_thread(int key_bytes, int value_bytes) {
  if (value_bytes == 0) return key_bytes == 8 ? ILGPU_HIP_SORT_ITEMS8 : ILGPU_HIP_SORT_ITEMS;
  if (value_bytes == 16) return 8;
  const int registers = (key_bytes == 8 ? 2 : 1) + (value_bytes == 8 ? 2 : 1);
  if (registers == 2) return value_bytes <= 2 ? 20 : ILGPU_HIP_SORT_PAIR_ITEMS2;
  return registers == 3 ? ILGPU_HIP_SORT_PAIR_ITEMS3 : ILGPU_HIP_SORT_PAIR_ITEMS4;
}
// 4-byte floating-point keys without values, whose order takes registers of its own, in full tiles of 512 threads: with 36
// keys 33 registers spill, with 32 a third fewer, and none where all tiles run at once.  (Normal keys with a copy in front, us,
// 36 / 32: 8 * 10^6 165 / 135, 9.6 * 10^6 187 / 181, 14 * 10^6 229 / 224, 20 000 003 305 / 279, 25 * 10^6 348 / 330; 28 and 24 keys for
// 20 000 003: 303 and 310.  Integer keys lose by it: whole numbers below 10^6, 14 * 10^6 176 / 182, 9.6 * 10^6 140 / 145.)
constexpr int kFloatItems = 32;
constexpr int tile_keys(int key_bytes, int value_bytes, int block) {
  return block * items_per_thread(key_bytes, value_bytes);
}
// Short tiles.  A sort of a few hundred tiles leaves compute units idle, and
// each of its passes lasts as long as one tile takes from its first load to its
// last store.  Keys without values that fit kShortTileMaxTiles tiles of a
// shorter class (a third, a half or two thirds of the usual keys per thread)
// take the shortest class that does: every tile resident at once, in one
// round, more compute units at work and fewer rows to rank and to write per
// block.
#ifndef ILGPU_HIP_SORT_SHORT_TILE_MAX_TILES
#define ILGPU_HIP_SORT_SHORT_TILE_MAX_TILES 512
#endif
constexpr int kShortTileMaxTiles = ILGPU_HIP_SORT_SHORT_TILE_MAX_TILES;
constexpr int kShortTileClasses = 3;
constexpr int short_items_per_thread(int key_bytes, int short_class) {
  const int full = items_per_thread(key_bytes, 0);
  const int items = short_class == 0 ? full / 3 : (short_class == 1 ? full / 2 : full * 2 / 3);
  return items < 2 ? 2 : items & ~1;
}

// How raw key bits map to unsigned bits that sort in the requested order.
// ordered(k) = k ^ xor_mask ^ (lsr(~k, bits-1) & reference_term) ^ (asr(k, bits-1) & total_term):
// branch-free for every mode.  reference_term is 1 for the float order of the
// reference (RadixSortOperations.tt:81-89 as written: the complement mask is a
// LOGICAL shift of ~bits, i.e. 1 for non-negative values and 0 otherwise);
// total_term is all bits below the sign for IEEE totalOrder (negative values
// have them flipped); both are 0 for integer keys.
struct KeyXform {
  uint64_t xor_mask;
  uint64_t reference_term;
  uint64_t total_term;
};

template <typename K>
__device__ __forceinline__ K key_term(K k, const KeyXform& xf) {
  constexpr int kBits = sizeof(K) * 8;
  using S = typename std::make_signed<K>::type;
  return (K)(((K)((K)(~k) >> (kBits - 1)) & (K)xf.reference_term) ^
             ((K)((S)k >> (kBits - 1)) & (K)xf.total_term));
}

template <typename K>
__device__ __forceinline__ K ordered_bits(K k, const KeyXform& xf) {
  return (K)(k ^ (K)xf.xor_mask ^ key_term(k, xf));
}

template <typename K>
__device__ __forceinline__ uint32_t digit_of(K k, const KeyXform& xf, int shift) {
  return (uint32_t)(ordered_bits(k, xf) >> shift) & (kRadix - 1);
}

// Inverse of ordered_bits.  The per-key term depends on the key's sign bit
// only and never changes it, so u = o ^ xor_mask has the sign bit of the key
// and the same term taken from u gives the key back.
template <typename K>
__device__ __forceinline__ K raw_bits(K o, const KeyXform& xf) {
  const K u = (K)(o ^ (K)xf.xor_mask);
  return (K)(u ^ key_term(u, xf));
}

constexpr uint32_t kNoHotDigit = 0xFFFFFFFFu;
constexpr int kMaxHot = 4;
// Device-resident description of the passes, written by plan_kernel.
struct SortPlan {
  uint32_t skip[kMaxPasses];        // digit identical for all keys, or left to the ties
  uint32_t src_is_alt[kMaxPasses];  // pass reads the alternate buffer
  // Up to kMaxHot digits that each hold an eighth of the keys or more, most
  // frequent first; unused entries are kNoHotDigit.
  uint32_t hot[kMaxPasses][kMaxHot];
  uint32_t first_executed;          // index of the first pass that runs
  uint32_t last_executed;           // index of the last pass that runs
  uint32_t executed;                // number of passes that run
  uint32_t final_in_alt;            // result sits in the alternate buffer
  uint32_t ties_left;               // the lower digits are left to ties_kernel
  uint32_t local_from;              // the digits below this one are left to local_sort_kernel
};
static_assert(sizeof(SortPlan) <= 256, "the temp view holds 256 bytes for the plan");

// Passes that take turns with two status arrays: each clears the words of the next one that runs, which the pass before it is
// done with, and only the first array is cleared beforehand.  Tiles shorter than what the temp view is sized for find room that
// way (tiles that all run at once, floating-point ones), and 2^27 u64 keys clear 9 MB in place of 75 (us, an array for every pass / turns:
// 2005 / 1994, with index values 2708 / 2699).  Long 4-byte keys, of which two of four passes run, take as long either way
// (2^26 to 2^28 u32 keys within 0.5 %, which is what two builds of the same code differ by); full tiles of 512 threads lose half a
// percent (14 * 10^6 u32 keys 175 / 176) and have an array for every pass.
constexpr bool sort_status_turns(int key_bytes, int block, bool at_once, bool float_tile) {
  return key_bytes > 1 && (block > ILGPU_HIP_SORT_BLOCK || at_once || float_tile);
}
// Clears the words of the pass that runs after this one, if there is one.
__device__ __forceinline__ void clear_next_status(uint32_t* status, int64_t region_words, const SortPlan* plan, int pass,
                                                  int threads) {
  if (plan->last_executed == (uint32_t)pass) return;
  uint4* words = reinterpret_cast<uint4*>(status + (plan->src_is_alt[pass] != 0 ? 0 : region_words));
  for (int64_t i = (int64_t)blockIdx.x * threads + threadIdx.x; i < region_words / 4; i += (int64_t)gridDim.x * threads)
    words[i] = make_uint4(0u, 0u, 0u, 0u);
}

// 8-byte keys whose upper halves rarely meet are sorted by that half alone, four
// passes instead of eight; what is left is to order the few neighbours whose
// upper halves are the same (ties_kernel), which reads the keys once.  Whether
// they rarely meet no digit histogram tells, so the histogram kernel also draws m
// keys, one from every m-th part of the input (positions that differ), and counts
// the upper halves that are drawn twice or more, those that are drawn three times or more,
// and the pairs of draws that share one, c (c - 1) / 2 where one is drawn c times.
// A run of L keys gives some L (L - 1) / 2 * m^2 / n^2 of them.
// The short way is taken
//   up to m^2 / n upper halves that are drawn twice or more: as many pairs as there are
//   keys (uniform keys have n^2 / 2^33 pairs);
//   up to kTieGroups upper halves that are drawn three times or more: short inputs,
//   of which a key in 64 is drawn, would pass with some thousand runs of a few dozen
//   keys, and where those lie side by side a few waves would order all of them;
//   up to 3 m^2 / n pairs, which is what a run of sqrt(6 n) keys gives: the longest that
//   ties_kernel orders in about the time of the passes that are saved (3500 of
//   2^21 keys, 28 000 of 2^27).
// (The draws that met an earlier one, counted once each, bound neither: one run of
// 16 000 keys, a thousand of 32.)
// (Whole sorts of u64 keys with a copy in front, us, all eight digits / the count of
// draws that met an earlier one / this.  2^21 keys: uniform 173 / 120 / 115; one cluster of
// 1000 keys 174 / 305 / 127, of 3000 173 / 811 / 153, of 16 000, refused, 174 / 5126 / 176; 2^24:
// uniform 622 / 393 / 390, one cluster of 4000 620 / 1356 / 435; 2^27: uniform 4231 / 2740 / 2722,
// one cluster of 16 000 4261 / 4243 / 3010, every upper half taken from as many as there are
// keys 4268 / 4263 / 3540.)
// From kTieMinKeys keys on: below that a pass takes so little time that the
// sampling, the ties kernel and four passes that return at once cost the same.
// Where the draws say no the sampling is lost: Zipf values below 2^15 as int64, two passes,
// 2^21 keys 79.8 / 83.4 / 81.7, 2^22 95.5 / 97.7 / 98.2, 2^24 239 / 235 / 240; values
// below 10^6, three passes, 2^21 97.9 / 99.8 / 98.2.
constexpr int kTiePasses = 4;                // passes over the upper half
constexpr uint32_t kTieGroups = 8;
// Draws: one key of 256 within these limits (2^18 draws of 2^27 keys cost 0.7 % more where they
// say no).
constexpr int kTieMinSampleBits = 15, kTieMaxSampleBits = 16;
constexpr int kTieSlotsPerDrawLog2 = 2;
// Slots that a draw tries before it goes uncounted: in its block's table, and in the
// grid's, where the second try lies behind the first vectors (one in 60 upper halves
// finds both taken).
constexpr int kTieBlockProbes = 8;
#ifndef ILGPU_HIP_SORT_TIE_MIN_LOG2
#define ILGPU_HIP_SORT_TIE_MIN_LOG2 21
#endif
constexpr int64_t kTieMinKeys = 1ll << ILGPU_HIP_SORT_TIE_MIN_LOG2;
static_assert(kTieMinKeys >= 1ll << (kTieMinSampleBits + kTieSlotsPerDrawLog2) &&
                  kTieSlotsPerDrawLog2 <= 8,
              "the table lies in the alternate keys");
struct TieSampling {
  // Upper halves met, in open addressing: upper half << 32 | times drawn, 0 where
  // nothing is.  nullptr: no sampling.
  unsigned long long* table;
  uint32_t* counts;         // kTicketGroups times {pairs, doubles, groups}, kTicketStride words apart
  uint32_t sample_bits;     // log2 of the number of draws
  uint32_t max_doubles, max_pairs;
};

// Whether the local sort (local_sort_kernel) can do what passes over the topmost digits leave is asked
// of m draws, one from every m-th part of the input, before anything is counted:
// sort_draw_kernel draws them and one block of the histogram kernel looks at them.
//   Keys may not crowd: sixteen of them in one of the local sort's bins, of which there are some
//   four for every key, send a window the slow way.  Of draws that agree down to a bin (in
//   log2(n) + 1 bits from the topmost one that differs) there are some m^2 / 4n if
//   the keys spread evenly and k m^2 / 2n if each bin in use holds k of them; up to 1.25 m^2 / n
//   are taken (k = 2.5; from k = 5 on a window in nine has such a bin).  Of 4-byte keys after two digits
//   0.9 m^2 / n: there, bins that have to be put into order cost as much as is saved from k = 1 on (with a copy in front, us,
//   every digit / the local sort, k = 1, 2, 3: 2^26 keys 656 / 665 / 775 / 840, pairs 1112 / 1083 / 1253 / 1383).
//   Two digits make runs that fit a window if few draws share a 16-bit prefix: a run of L keys
//   is drawn L m / n times and gives half the square of that in pairs of draws.
//   (Whether one digit does, its counts tell exactly.)
//   A frequent value among others, which sends one window the slow way, is not asked for: a short sort waits for that
//   window, so u32 keys lose there, but pairs and 8-byte keys gain all the same (with a copy in front, us, every digit / the
//   local sort: 300 000 keys, a hundredth of them one value, u32 57 / 66, pairs 65 / 66, u64 103 / 87; 30 000, 20 copies of one, 47 / 54,
//   59 / 54, 76 / 66; 2 000 000, 20 values 20 times each, u32 92 / 107).
// (2^26 u32 keys, every value some 30 times, with a copy in front, us: every digit sorted 750, the local
// sort 1236.)
struct LocalSampling {
  const void* draws;        // keys in their ordered form.  nullptr: not asked
  uint32_t* from;           // out: the lowest digit of the prefix whose runs are short (0: they are not),
                            // and in the next word whether the keys spread
  LocalLimits limits;
};
// Where the draws lie in the alternate keys: behind the table of TieSampling.
constexpr int64_t kLocalDrawsOffset = 8ll << (kTieMaxSampleBits + kTieSlotsPerDrawLog2);

// Clears words[0..count) and more[0..more_count) and takes the draws of LocalSampling.
template <typename K, bool FLOAT_KEYS>
__global__ __launch_bounds__(256) void sort_draw_kernel(
    uint32_t* words, int64_t count, uint32_t* more, int64_t more_count, const K* __restrict__ keys,
    int64_t n, KeyXform xf, K* draws, uint32_t draw_bits) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  const int64_t first = (int64_t)blockIdx.x * 256 + threadIdx.x;
  for (int64_t s = first; s < 1ll << draw_bits; s += stride) {
    const K k = keys[local_draw_place((uint64_t)s, (int)draw_bits, (uint64_t)n)];
    const K o = FLOAT_KEYS ? ordered_bits(k, xf) : (K)(k ^ (K)xf.xor_mask);
    draws[local_draw_slot((uint32_t)s, (int)draw_bits)] = o;
  }
  for (int64_t i = first; i < count; i += stride) words[i] = 0u;
  for (int64_t i = first; i < more_count; i += stride) more[i] = 0u;
}

// By one block of the histogram kernel, with its LDS: what the draws say, into local.from[0..1].
// (The draws are held in registers where one chunk is all of them: short inputs wait for this block.)
template <typename K>
__device__ __forceinline__ void choose_local_digits(const LocalSampling& local, uint32_t* s_table) {
  constexpr int kTableBits = 14;  // words
  static_assert(kHistLdsWords >= 1 << kTableBits, "a byte for every 16-bit prefix");
  constexpr int kPerVector = 16 / (int)sizeof(K);
  constexpr int kVectors = (1 << kLocalChunkBits) / kPerVector / kHistBlock;  // of a thread and a chunk of draws
  using V = typename Vec16<K>::type;
  const int t = threadIdx.x;
  __shared__ unsigned long long s_diff;
  __shared__ uint32_t s_equal, s_pairs, s_draws;
  auto clear_table = [&]() {
    for (int i = t; i < (1 << kTableBits) / 4; i += kHistBlock)
      reinterpret_cast<uint4*>(s_table)[i] = make_uint4(0u, 0u, 0u, 0u);
  };
  const V* draws = static_cast<const V*>(local.draws);
  const LocalLimits& limits = local.limits;
  const int vectors = (1 << limits.draw_bits) / kPerVector;
  const int chunks = (int)limits.draw_bits > kLocalChunkBits ? 1 << (limits.draw_bits - kLocalChunkBits) : 1;
  V d[kVectors];
  auto load = [&](int chunk) {
#pragma unroll
    for (int v = 0; v < kVectors; ++v) {
      const int i = (chunk * kVectors + v) * kHistBlock + t;
      d[v] = draws[i < vectors ? i : 0];
    }
  };
  auto in_use = [&](int chunk, int v) { return (chunk * kVectors + v) * kHistBlock + t < vectors; };
  load(0);
  const K first = static_cast<const K*>(local.draws)[0];
  clear_table();
  if (t == 0) {
    s_diff = 0ull;
    s_equal = s_pairs = s_draws = 0u;
  }
  K diff = 0;
#pragma unroll
  for (int v = 0; v < kVectors; ++v)
#pragma unroll
    for (int u = 0; u < kPerVector; ++u) diff |= (K)(d[v][u] ^ first);
#pragma unroll
  for (int s = 1; s < kWaveSize; s <<= 1) diff |= shfl(diff, (t & (kWaveSize - 1)) ^ s);
  __syncthreads();
  if ((t & (kWaveSize - 1)) == 0) atomicOr(&s_diff, (unsigned long long)diff);
  __syncthreads();
  // The topmost bit that differs in a chunk, and its digit.  (One that fewer than some thousandth of the keys have may be
  // missed: their runs are shorter than is thought, and no others longer.)
  const int top_bit = s_diff != 0ull ? 63 - __builtin_clzll(s_diff) : 0;
  const int top = top_bit / 8;
  if (top < 3) return;  // two digits at least have to be below the passes' for the way to pay
  // 32 bits from the topmost one that differs on.
  auto upper = [&](K k) -> uint32_t {
    return top_bit >= 31 ? (uint32_t)(k >> (top_bit - 31)) : (uint32_t)k << (31 - top_bit);
  };

  // Draws that meet an earlier one, in a table of open addressing: of many draws those of one part
  // of the values at a time, which half fill it, and of some parts.  (Single frequent values are mostly in another part: those the draws of one
  // prefix tell.)
  static_assert(kTableBits == kLocalPartBits + 1, "draws of a part half fill the table");
  constexpr uint32_t kSlots = 1u << kTableBits;
  const uint32_t part_mask = (uint32_t)local_parts((int)limits.draw_bits) - 1u;
  uint32_t equal = 0;
  for (int turn = 0; turn < chunks * (int)limits.parts; ++turn) {
    const int chunk = turn & (chunks - 1);
    const uint32_t part = (uint32_t)(turn / chunks);
    if (chunks > 1) load(chunk);
    if (chunk == 0 && part != 0u) {
      __syncthreads();
      clear_table();
      __syncthreads();
    }
#pragma unroll
    for (int v = 0; v < kVectors; ++v) {
      if (!in_use(chunk, v)) continue;
      uint32_t value[kPerVector], slot[kPerVector], old[kPerVector];
#pragma unroll
      for (int u = 0; u < kPerVector; ++u) {
        value[u] = upper(d[v][u]) >> (32 - limits.bin_bits);  // at most 31 bits
        uint32_t hash = value[u] * 0x9E3779B1u;
        hash = (hash ^ hash >> 16) * 0x85EBCA6Bu;
        slot[u] = hash >> (32 - kTableBits);
        old[u] = 0u;
        if ((hash & part_mask) == part) old[u] = atomicCAS(&s_table[slot[u]], 0u, value[u] + 1u);
      }
#pragma unroll
      for (int u = 0; u < kPerVector; ++u) {
        for (int probe = 0; probe < 8 && old[u] != 0u && old[u] != value[u] + 1u; ++probe) {
          slot[u] = (slot[u] + 1u) & (kSlots - 1u);
          old[u] = atomicCAS(&s_table[slot[u]], 0u, value[u] + 1u);
        }
        equal += old[u] == value[u] + 1u;
      }
    }
  }
#pragma unroll
  for (int s = 1; s < kWaveSize; s <<= 1) equal += shfl(equal, (t & (kWaveSize - 1)) ^ s);
  if ((t & (kWaveSize - 1)) == 0) atomicAdd(&s_equal, equal);
  __syncthreads();
  if (s_equal > limits.max_equal) return;
  if (t == 0) local.from[1] = 1u;
  if (limits.max_pairs == 0u) return;  // one digit is enough

  // Draws of every prefix, a byte each (of 2^15 draws from all over the input at most: with 2^16 the histogram of 2^26
  // keys waited 16 us for this block).
  clear_table();
  __syncthreads();
  uint32_t pairs = 0, most = 0;
  for (int chunk = 0; chunk < chunks && chunk < 1 << (kLocalPrefixBits - kLocalChunkBits); ++chunk) {
    if (chunks > 1) load(chunk);
#pragma unroll
    for (int v = 0; v < kVectors; ++v) {
      // (Far too many of one prefix: enough.  A count that runs over says the same.)
      if (!in_use(chunk, v) || most >= 128u) continue;
      uint32_t old[kPerVector];
#pragma unroll
      for (int u = 0; u < kPerVector; ++u) {
        const uint32_t prefix = (uint32_t)(d[v][u] >> (8 * (top - 1))) & 0xFFFFu;
        const uint32_t at = (prefix & 3u) * 8u;
        old[u] = (atomicAdd(&s_table[prefix >> 2], 1u << at) >> at) & 0xFFu;
      }
#pragma unroll
      for (int u = 0; u < kPerVector; ++u) {
        pairs += old[u];
        most = most < old[u] ? old[u] : most;
      }
    }
  }
#pragma unroll
  for (int s = 1; s < kWaveSize; s <<= 1) {
    pairs += shfl(pairs, (t & (kWaveSize - 1)) ^ s);
    const uint32_t other = shfl(most, (t & (kWaveSize - 1)) ^ s);
    most = most < other ? other : most;
  }
  if ((t & (kWaveSize - 1)) == 0) {
    atomicAdd(&s_pairs, pairs);
    atomicMax(&s_draws, most + 1u);
  }
  __syncthreads();
  if (t == 0 && s_pairs <= limits.max_pairs && s_draws <= limits.max_draws) local.from[0] = (uint32_t)(top - 1);
}

// The first active lane's key, as a wave-uniform value.
__device__ __forceinline__ uint64_t readfirstlane_key(uint64_t k) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)k);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(k >> 32));
  return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint32_t readfirstlane_key(uint32_t k) {
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)k);
}
__device__ __forceinline__ uint32_t readfirstlane_key(uint16_t k) {
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)k);
}
__device__ __forceinline__ uint32_t readfirstlane_key(uint8_t k) {
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)k);
}

// ---- histogram of all digit positions ------------------------------------
template <typename K, bool FLOAT_KEYS>
__global__ __launch_bounds__(kHistBlock) void sort_histogram_kernel(
    const K* __restrict__ keys, int64_t n, KeyXform xf, int passes,
    int replica_shift, uint32_t* __restrict__ global_hist, TieSampling ties, LocalSampling local) {
  using V = typename Vec16<K>::type;
  constexpr int VN = Vec16<K>::N;
  extern __shared__ __align__(8) uint32_t s_hist[];  // [passes][256][replicas]
  // Blocks that count, and this one among them: where draws are looked at the last block of the
  // grid does that.
  const uint32_t counting = gridDim.x - (sizeof(K) >= 4 && local.draws != nullptr ? 1u : 0u);
  if constexpr (sizeof(K) >= 4) {
    if (blockIdx.x == counting) {
      choose_local_digits<K>(local, s_hist);
      return;
    }
  }
  const int words = (passes * kRadix) << replica_shift;
  // This thread's draw of the tie sampling.  Draws meet within their block first, in
  // LDS: where many keys share an upper half, all draws of the grid would queue
  // at one slot of the table (2^17 draws: 1.5 ms).  The thread that enters an upper
  // half into the block's table takes it to the grid's, with its count; the answer is
  // looked at when the keys have been counted.
  __shared__ uint32_t s_pairs, s_doubles, s_groups;
  uint32_t upper = 0, drawn = 0, slot = 0;  // drawn: times in this block, 0 for all but one thread
  unsigned long long met = 0;
  // The first blocks draw, a key per thread: the others, one of which is next to each of them
  // on its compute unit in long inputs, have more of the LDS meanwhile (2^24 keys with 128 draws
  // per block 41 us, with 512 in a quarter of the blocks 37.6).
  const bool sampling = sizeof(K) == 8 && ties.table != nullptr &&
                        blockIdx.x * (uint32_t)kHistBlock < (1u << ties.sample_bits);
  if constexpr (sizeof(K) == 8) {
    if (sampling) {
      constexpr int kBlockSlotBits = 10;
      constexpr uint32_t kBlockSlots = 1u << kBlockSlotBits;
      static_assert(kBlockSlots >= 2 * kHistBlock && kBlockSlots * 2 <= kMaxPasses * kRadix,
                    "room for every draw in the counters of the histogram");
      auto* block_table = reinterpret_cast<unsigned long long*>(s_hist);
      for (uint32_t i = threadIdx.x; i < kBlockSlots; i += kHistBlock) block_table[i] = 0ull;
      if (threadIdx.x == 0) s_pairs = s_doubles = s_groups = 0u;
      static_assert(1 << kTieMinSampleBits >= kHistBlock, "a block's threads all draw");
      const uint32_t s = blockIdx.x * (uint32_t)kHistBlock + threadIdx.x;
      {
        uint64_t z = ((uint64_t)s + 1ull) * 0x9E3779B97F4A7C15ull;  // splitmix64
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        // A random place in part s of the input.
        const uint64_t at = ((uint64_t)s << 32 | (uint32_t)z) << (32 - ties.sample_bits);
        upper = (uint32_t)(keys[__umul64hi(at, (uint64_t)n)] >> 32);
      }
      __syncthreads();
      // (The lanes that agree with the first one go together: keys that all share an upper half
      // would queue at one word 512 deep, 2 us.)
      const uint64_t same = __ballot(upper == (uint32_t)__builtin_amdgcn_readfirstlane((int)upper));
      const int lane = threadIdx.x & (kWaveSize - 1);
      drawn = lane == 0 ? (uint32_t)__popcll(same) : (same >> lane & 1ull ? 0u : 1u);
      if (drawn != 0) {
        slot = (upper * 0x85EBCA6Bu) >> (32 - kBlockSlotBits);
        int probe = 0;
        for (; probe < kTieBlockProbes; ++probe) {
          const unsigned long long old =
              atomicCAS(&block_table[slot], 0ull, (unsigned long long)upper << 32 | drawn);
          if (old == 0ull) break;
          if ((uint32_t)(old >> 32) == upper) {
            atomicAdd(&block_table[slot], (unsigned long long)drawn);
            drawn = 0;
            break;
          }
          slot = (slot + 1) & (kBlockSlots - 1);
        }
        if (probe == kTieBlockProbes) slot = kBlockSlots;
      }
      __syncthreads();
      if (drawn != 0 && slot < kBlockSlots) drawn = (uint32_t)block_table[slot];
      // (No sum counts more than one too many at a time, so that none overflows.)
      const uint32_t pairs = min(drawn * (drawn - 1) / 2, ties.max_pairs + 1);
      if (drawn > 1) atomicAdd(&s_pairs, pairs);
      if (drawn > 1 && pairs > ties.max_pairs) drawn = 0;  // enough said
      slot = (upper * 0x9E3779B1u) >> (32 - kTieSlotsPerDrawLog2 - ties.sample_bits);
      if (drawn != 0) met = atomicCAS(&ties.table[slot], 0ull, (unsigned long long)upper << 32 | drawn);
    }
  }
  for (int i = threadIdx.x; i < words; i += kHistBlock) s_hist[i] = 0u;
  __syncthreads();

  const uint32_t replica = threadIdx.x & ((1u << replica_shift) - 1u);
  auto count = [&](K k) {
    K o = (K)(k ^ (K)xf.xor_mask);
    if constexpr (FLOAT_KEYS) o ^= key_term(k, xf);
#pragma unroll
    for (int p = 0; p < (int)sizeof(K); ++p) {
      const uint32_t d = (uint32_t)(o >> (8 * p)) & (kRadix - 1);
      atomicAdd(&s_hist[((p * kRadix + d) << replica_shift) + replica], 1u);
    }
    // Key by key: with the digits of all keys of a vector extracted first and
    // their atomics issued in one burst the kernel measured 4 % slower.
    __builtin_amdgcn_sched_barrier(0);
  };

  // Non-temporal loads: 0.180 against 0.217 ms for 2^28 u32 keys.  The kernel
  // is bound by the rate of LDS instructions (a wave's atomic takes the LDS of
  // a compute unit about five cycles whatever its addresses) next to the key
  // stream, and the two overlap better when the keys do not allocate in L2.
  // Two vectors per round: one is 0.235 ms, four 0.208.
  auto load_keys = [](const V* p) -> V {
    return ILGPU_HIP_SORT_HIST_NT ? __builtin_nontemporal_load(p) : *p;
  };
  // Vectors whose keys are the same in every lane of a wave, wholly or in their
  // upper half (constant input; small values under large types), would meet
  // in one counter 256 keys deep.  They are counted as runs in registers, one
  // check per vector, and reach the counters when the value changes; only
  // with all 64 lanes at work, so that the run is the same in every lane.
  // (Sorts of 2^28 u32 keys: all equal 0.269 -> 0.197 ms, Zipf values below
  // 2^16 1.174 -> 1.120, uniform 2.056 -> 2.059.)
  constexpr int kHalfBits = 4 * (int)sizeof(K);
  K run_key = 0, run_half = 0;
  uint32_t run_key_count = 0, run_half_count = 0;
  auto flush_key_run = [&]() {
    if ((threadIdx.x & (kWaveSize - 1)) == 0 && run_key_count != 0u) {
      K o = (K)(run_key ^ (K)xf.xor_mask);
      if constexpr (FLOAT_KEYS) o ^= key_term(run_key, xf);
#pragma unroll
      for (int p = 0; p < (int)sizeof(K); ++p)
        atomicAdd(&s_hist[((p * kRadix + ((uint32_t)(o >> (8 * p)) & (kRadix - 1))) << replica_shift) + replica],
                  run_key_count);
    }
    run_key_count = 0u;
  };
  auto flush_half_run = [&]() {  // run_half: ordered bits above the lower half
    if constexpr (sizeof(K) >= 2) {  // a 1-byte key has no upper half of whole digits
      if ((threadIdx.x & (kWaveSize - 1)) == 0 && run_half_count != 0u) {
#pragma unroll
        for (int p = (int)sizeof(K) / 2; p < (int)sizeof(K); ++p)
          atomicAdd(&s_hist[((p * kRadix + ((uint32_t)(run_half >> (8 * p - kHalfBits)) & (kRadix - 1))) << replica_shift) + replica],
                    run_half_count);
      }
    }
    run_half_count = 0u;
  };
  // Whether a vector's keys agree in every lane of the (full) wave: wholly
  // (returns 2), in their upper half (1), or not (0).
  auto uniformity = [&](const V& v, K& first) -> int {
    K diff = 0;
#pragma unroll
    for (int k = 1; k < VN; ++k) diff |= (K)(v[k] ^ v[0]);
    first = (K)readfirstlane_key(v[0]);
    diff |= (K)(v[0] ^ first);
    if (__ballot(true) != ~0ull) return 0;
    if (__ballot(diff != 0) == 0ull) return 2;
    if (FLOAT_KEYS) return 0;  // the upper half of their ordered bits depends on the sign
    return __ballot((K)(diff >> kHalfBits) != 0) == 0ull ? 1 : 0;
  };
  auto count_vector = [&](auto checked, const V& v) {
    if constexpr (decltype(checked)::value) {
      K first;
      const int same = uniformity(v, first);
      if (same == 2) {
        if (first != run_key) { flush_key_run(); run_key = first; }
        run_key_count += (uint32_t)(kWaveSize * VN);
        return;
      }
      if (same == 1) {
        const K half = (K)((K)(first ^ (K)xf.xor_mask) >> kHalfBits);
        if (half != run_half) { flush_half_run(); run_half = half; }
        run_half_count += (uint32_t)(kWaveSize * VN);
#pragma unroll
        for (int k = 0; k < VN; ++k) {
          const K o = (K)(v[k] ^ (K)xf.xor_mask);
#pragma unroll
          for (int p = 0; p < (int)sizeof(K) / 2; ++p)
            atomicAdd(&s_hist[((p * kRadix + ((uint32_t)(o >> (8 * p)) & (kRadix - 1))) << replica_shift) + replica], 1u);
          __builtin_amdgcn_sched_barrier(0);
        }
        return;
      }
    }
#pragma unroll
    for (int k = 0; k < VN; ++k) count(v[k]);
  };
  const uintptr_t addr = reinterpret_cast<uintptr_t>(keys);
  int64_t head = (int64_t)(((16 - (addr & 15)) & 15) / sizeof(K));
  if (head > n) head = n;
  const V* body = reinterpret_cast<const V*>(keys + head);
  const int64_t nvec = (n - head) / VN;
  const int64_t tail_start = head + nvec * VN;
  const int64_t stride = (int64_t)counting * kHistBlock;
  // The first round's vectors are requested, and by the first of them a wave
  // decides whether it looks for runs at all: the check costs keys that vary
  // 1 to 2 % of a sort when every vector pays it.
  int64_t i = (int64_t)blockIdx.x * kHistBlock + threadIdx.x;
  V v0[kHistUnroll];
  const bool have_first = i + (kHistUnroll - 1) * stride < nvec;
  if (have_first) {
#pragma unroll
    for (int u = 0; u < kHistUnroll; ++u) v0[u] = load_keys(&body[i + u * stride]);
  }
  bool look_for_runs = false;
  if (ILGPU_HIP_SORT_HIST_RUNS && sizeof(K) >= 2 && have_first) {
    K first;
    look_for_runs = uniformity(v0[0], first) != 0;
  }
  auto count_body = [&](auto checked) {
    if (have_first) {
#pragma unroll
      for (int u = 0; u < kHistUnroll; ++u) count_vector(checked, v0[u]);
      i += kHistUnroll * stride;
    }
    if constexpr (sizeof(K) == 8) {  // the tie sampling's second slot
      if (met != 0ull && (uint32_t)(met >> 32) != upper) {
        slot ^= 1u;
        met = atomicCAS(&ties.table[slot], 0ull, (unsigned long long)upper << 32 | drawn);
      }
    }
    for (; i + (kHistUnroll - 1) * stride < nvec; i += kHistUnroll * stride) {
      V v[kHistUnroll];
#pragma unroll
      for (int u = 0; u < kHistUnroll; ++u) v[u] = load_keys(&body[i + u * stride]);
#pragma unroll
      for (int u = 0; u < kHistUnroll; ++u) count_vector(checked, v[u]);
    }
    for (; i < nvec; i += stride) {
      V a = load_keys(&body[i]);
      count_vector(checked, a);
    }
  };
  if (look_for_runs) count_body(std::true_type{});
  else count_body(std::false_type{});
  if (blockIdx.x == 0) {
    const int64_t extra = head + (n - tail_start);
    if ((int64_t)threadIdx.x < extra) {
      const int64_t idx = (int64_t)threadIdx.x < head
                              ? (int64_t)threadIdx.x
                              : tail_start + ((int64_t)threadIdx.x - head);
      count(keys[idx]);
    }
  }
  flush_key_run();
  flush_half_run();
  if constexpr (sizeof(K) == 8) {
    if (drawn != 0) {
      uint32_t before = 0;
      if (met != 0ull && (uint32_t)(met >> 32) == upper) {
        before = (uint32_t)atomicAdd(&ties.table[slot], (unsigned long long)drawn);
        atomicAdd(&s_pairs, min(drawn * before, ties.max_pairs + 1));
      }
      if (before < 2 && before + drawn >= 2) atomicAdd(&s_doubles, 1u);
      if (before < 3 && before + drawn >= 3) atomicAdd(&s_groups, 1u);
    }
    __syncthreads();
    // One add per block, to one of eight lines: 2^11 adds to one word, a wave each, took 20 us.
    if (sampling && threadIdx.x == 0 && s_pairs != 0) {
      uint32_t* counts = ties.counts + (blockIdx.x % kTicketGroups) * kTicketStride;
      atomicAdd(&counts[0], s_pairs);
      atomicAdd(&counts[1], s_doubles);
      atomicAdd(&counts[2], s_groups);
    }
  } else {
    __syncthreads();
  }

  const int replicas = 1 << replica_shift;
  for (int b = threadIdx.x; b < passes * kRadix; b += kHistBlock) {
    uint32_t c = 0;
    for (int r = 0; r < replicas; ++r)
      c += s_hist[(b << replica_shift) + ((r + b) & (replicas - 1))];
    if (c != 0) atomicAdd(&global_hist[b], c);
  }
}

// `join` over the lanes up to each one, for values that zero leaves as they are: six moves between lanes in place of trips to
// the LDS.
template <typename Join>
__device__ __forceinline__ uint32_t wave_inclusive(uint32_t v, Join join) {
  v = join(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false));  // row_shr:1
  v = join(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false));
  v = join(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false));
  v = join(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false));
  v = join(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));  // row_bcast:15
  v = join(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));  // row_bcast:31
  return v;
}
// Over all of them, in every lane: OR, the sum and the largest.
template <typename Join>
__device__ __forceinline__ uint32_t wave_join(uint32_t v, Join join) {
  return (uint32_t)__builtin_amdgcn_readlane((int)wave_inclusive(v, join), kWaveSize - 1);
}
__device__ __forceinline__ uint32_t wave_or(uint32_t v) {
  return wave_join(v, [](uint32_t a, uint32_t b) { return a | b; });
}
__device__ __forceinline__ int wave_sum(int v) {
  return (int)wave_join((uint32_t)v, [](uint32_t a, uint32_t b) { return a + b; });
}
__device__ __forceinline__ uint32_t wave_most(uint32_t v) {
  return wave_join(v, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
}

// ---- plan: exclusive digit offsets, skipped passes, buffer parity ---------
// One block; every 256 threads take a digit position, four at a time.  (One position after the other,
// a chain of barriers, took 4.5 us for 4-byte keys and 8.4 for 8-byte keys.)
constexpr int kPlanGroups = 4;
constexpr int kPlanBlock = kPlanGroups * kRadix;
__global__ __launch_bounds__(kPlanBlock) void plan_kernel(
    const uint32_t* __restrict__ global_hist, uint32_t* __restrict__ excl,
    SortPlan* __restrict__ plan, int passes, uint32_t n, TieSampling ties,
    const uint32_t* __restrict__ local_from, uint32_t local_max_run, uint32_t local_window_keys) {
  constexpr int kRounds = kMaxPasses / kPlanGroups;
  constexpr int kGroupWaves = kRadix / kWaveSize;
  constexpr int kFrequent = 8;  // digits with an eighth of the keys: no more than eight
  __shared__ uint32_t s_wave[kMaxPasses][kGroupWaves];
  __shared__ uint32_t s_most[kMaxPasses];  // keys of a position's most frequent digit
  __shared__ uint32_t s_frequent[kMaxPasses];
  __shared__ unsigned long long s_hot[kMaxPasses][kFrequent];  // count << 8 | digit
  const int d = threadIdx.x & (kRadix - 1);
  const int group = threadIdx.x / kRadix;
  const int lane = d & (kWaveSize - 1);
  const int wave = d / kWaveSize;
  uint32_t counts[kRounds], inclusive[kRounds];
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const int p = r * kPlanGroups + group;
    counts[r] = p < passes ? global_hist[p * kRadix + d] : 0u;
  }
  uint32_t pairs = 0, doubles = 0, groups = 0;
  if (ties.table != nullptr) {
    for (int g = 0; g < kTicketGroups; ++g) {
      pairs += ties.counts[g * kTicketStride];
      doubles += ties.counts[g * kTicketStride + 1];
      groups += ties.counts[g * kTicketStride + 2];
    }
  }
  const bool spread = local_from != nullptr && local_from[1] != 0u;
  const int two_digits = spread ? (int)local_from[0] : 0;
  if (threadIdx.x < kMaxPasses) s_most[threadIdx.x] = s_frequent[threadIdx.x] = 0u;
  if (threadIdx.x < kMaxPasses * kFrequent) s_hot[threadIdx.x / kFrequent][threadIdx.x % kFrequent] = 0ull;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const int p = r * kPlanGroups + group;
    inclusive[r] = 0u;
    if (r * kPlanGroups >= passes) break;
    const uint32_t c = counts[r];
    const uint32_t inc = wave_inclusive(c, [](uint32_t a, uint32_t b) { return a + b; });
    const uint32_t most = wave_most(c);
    inclusive[r] = inc;
    if (lane == kWaveSize - 1) s_wave[p][wave] = inc;
    if (lane == 0) atomicMax(&s_most[p], most);
    // A digit qualifies as dominant with an eighth of the keys (two lanes of a sub-tile row on
    // average).
    if (c != 0u && (uint64_t)c * kFrequent >= (uint64_t)n)
      s_hot[p][atomicAdd(&s_frequent[p], 1u)] = ((unsigned long long)c << 8) | (unsigned long long)d;
  }
  __syncthreads();
  uint32_t varies = 0;  // positions whose digit is not the same for every key
#pragma unroll
  for (int p = 0; p < kMaxPasses; ++p) varies |= p < passes && s_most[p] != n ? 1u << p : 0u;
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const int p = r * kPlanGroups + group;
    if (p >= passes) break;
    uint32_t off = 0;
#pragma unroll
    for (int w = 0; w < kGroupWaves; ++w) off += w < wave ? s_wave[p][w] : 0u;
    excl[p * kRadix + d] = off + inclusive[r] - counts[r];
    // The most frequent of the dominant digits, most frequent first.
    if (d < kFrequent) {
      const unsigned long long mine = s_hot[p][d];
      int before = 0;
#pragma unroll
      for (int h = 0; h < kFrequent; ++h)
        before += s_hot[p][h] > mine || (s_hot[p][h] == mine && h < d) ? 1 : 0;
      if (before < kMaxHot) plan->hot[p][before] = mine != 0ull ? (uint32_t)(mine & 0xFFull) : kNoHotDigit;
    }
  }
  if (threadIdx.x != 0) return;

  // The lower digits [0, left) are left to the local sort, if the draws say that the keys
  // spread and that saves two passes at least (a digit that all keys share needs none): below
  // the topmost digit that differs where none of its values has more keys than a window
  // (local_max_run != 0: the input may be short enough for that), or below two digits where the
  // draws found short runs and no count speaks for a long one.
  int left = 0, local = 0;
  if (spread && varies != 0u) {
    const int top = 31 - __builtin_clz(varies);
    if (local_max_run == 0) {
      if (two_digits != 0 && local_counts_allow(n, s_most[two_digits + 1], s_most[two_digits], local_window_keys))
        local = two_digits;
    } else if (s_most[top] <= local_max_run) local = top;
    if (__popc(varies & ((1u << local) - 1u)) < 2) local = 0;
    left = local;
  }
  // Or to the ties, if the draws rarely meet and that saves at least two passes.  An
  // even number of passes ends in the caller's buffer, where the ties are ordered: an
  // odd one takes a lower digit along.
  if (ties.table != nullptr && local == 0 && pairs <= ties.max_pairs && doubles <= ties.max_doubles &&
      groups <= kTieGroups) {
    left = kMaxPasses - kTiePasses;
    if (__popc(varies >> left) & 1)
      while (left > 0 && !(varies >> --left & 1u)) {}
    if (__popc(varies & ((1u << left) - 1u)) < 2) left = 0;
  }
  uint32_t parity = 0, executed = 0, first = (uint32_t)passes, last = (uint32_t)passes;
  for (int p = 0; p < passes; ++p) {
    const bool skipped = !(varies >> p & 1u) || p < left;
    plan->skip[p] = skipped ? 1u : 0u;
    plan->src_is_alt[p] = parity;
    if (!skipped) {
      if (executed == 0) first = (uint32_t)p;
      last = (uint32_t)p;
      parity ^= 1u;
      ++executed;
    }
  }
  plan->first_executed = first;
  plan->last_executed = last;
  plan->executed = executed;
  plan->final_in_alt = parity;
  plan->ties_left = left > 0 && local == 0 ? 1u : 0u;
  plan->local_from = (uint32_t)local;
}

// ---- onesweep pass ---------------------------------------------------------
// Ranking.  A block's tile is cut into sub-tiles, one per wave; lane l of wave
// w holds items w*64*kItems + j*64 + l, j = 0 .. kItems-1, so memory order
// inside a sub-tile is (row j, lane) and a row is one 256-byte load.  Every
// (wave, digit) pair owns one 32-bit LDS counter.  For row j every lane adds
// one to the counter of its digit with a returning LDS atomic; the value that
// comes back is the key's rank among the keys of that digit in the sub-tile.
//
// That the rank follows memory order rests on two properties of the LDS:
// instructions of one wave execute in issue order (rows chain through the
// counters without barriers), and the lanes of ONE atomic instruction that
// meet in one address are served in ascending lane order.  The second is a
// property of this hardware (gfx950), not of the programming model; it is
// checked on the device by ilgpu_hip_selftest_lds_atomic_order and, end to
// end, by every stability test of the pair sorts.  With it the pass is stable
// at one LDS operation per key and no cross-lane arithmetic.
template <int KEY_BYTES, int VALUE_BYTES, int BLOCK,
          int ITEMS = items_per_thread(KEY_BYTES, VALUE_BYTES)>
struct SortTile {
  static constexpr int kSubTiles = BLOCK / kSubLanes;
  static constexpr int kCounterWords = kSubTiles * kRadix;
  static constexpr int kCounterBytes = kCounterWords * 4;
  static constexpr int kItems = ITEMS;
  static constexpr int kTile = BLOCK * ITEMS;
  static constexpr int kSubTileKeys = kSubLanes * kItems;
  static constexpr int kKeyStageBytes = kTile * KEY_BYTES;
  // The values of a tile go through the same LDS bytes after the keys, all at
  // once when they fit (72 KiB per 512 threads: two such blocks or one of 1024
  // threads share a compute unit's LDS), else in rounds.
#ifndef ILGPU_HIP_SORT_VALUE_STAGE
#define ILGPU_HIP_SORT_VALUE_STAGE 1
#endif
  static constexpr int kValueStageLimit = ILGPU_HIP_SORT_VALUE_STAGE ? (BLOCK / 512) * 72 * 1024 : 0;
  static constexpr int kValueStageBytes =
      kTile * VALUE_BYTES <= kValueStageLimit ? kTile * VALUE_BYTES : 0;
  static constexpr int kKeyOrCounterBytes =
      kCounterBytes > kKeyStageBytes ? kCounterBytes : kKeyStageBytes;
  static constexpr int kStageBytes =
      kValueStageBytes > kKeyOrCounterBytes ? kValueStageBytes : kKeyOrCounterBytes;
};

// Cache policy of a pass's key loads and scattered stores.  Measured on 2^28
// u32 keys, ms per pass: plain / plain 0.477, non-temporal loads 0.486,
// non-temporal stores 0.658 (the scattered stores rely on L2 to merge the
// pieces of a line that different waves write).
#ifndef ILGPU_HIP_SORT_NT_LOAD
#define ILGPU_HIP_SORT_NT_LOAD 0
#endif
// Rows of a tile whose loads the pipelined pass issues before it starts to
// rank; the loads of the other rows follow one rank group at a time, so that
// a wave never has more than this many loads in flight (more than about 24
// stall a wave on an idle device).  Under load the effect is small: 2.045 ms
// per sort of 2^28 u32 keys with 24 against 2.053 with all 36 up front.
#ifndef ILGPU_HIP_SORT_LOAD_AHEAD
#define ILGPU_HIP_SORT_LOAD_AHEAD 24
#endif
#ifndef ILGPU_HIP_SORT_NT_STORE
#define ILGPU_HIP_SORT_NT_STORE 0
#endif
template <int KEY_BYTES, int ITEMS, bool FULL>
__device__ __forceinline__ void load_tile_keys(
    const typename KeyOf<KEY_BYTES>::type* __restrict__ src, int64_t tile_base,
    int valid, int first_local,
    typename KeyOf<KEY_BYTES>::type (&key)[ITEMS]) {
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const int local = first_local + j * kSubLanes;
    if (FULL || local < valid)
      key[j] = ILGPU_HIP_SORT_NT_LOAD ? __builtin_nontemporal_load(&src[tile_base + local])
                                      : src[tile_base + local];
    else key[j] = 0;
  }
}

// Waves per SIMD the pass kernel is compiled for: sixteen waves per CU, as two
// 512-thread blocks or one 1024-thread block.  That bounds a thread at 128
// registers (36 keys and 18 registers of packed ranks in a keys-only sort;
// fewer items when values ride along) and the blocks of a CU at 160 KiB of
// LDS together (a 36-key tile stages 72 KiB per 512 threads).
#ifndef ILGPU_HIP_SORT_WAVES_PER_EU
#define ILGPU_HIP_SORT_WAVES_PER_EU 4
#endif

// Where the code of the large kernels begins: at a fixed place, so that what is added to one kernel does not move the others.  A tile
// runs through 40 to 64 KiB of code, about what the instruction caches hold, and the same instructions take up to 1 % longer at
// another address.  This one is no better than any other by rule: it measured well, and what grows inside a kernel still moves its
// own loops.  (us, wherever the linker puts it / here, in one process: u32 2^25 314.5 / 310.5, 50 * 10^6 458.5 / 456.5, 2^26 below
// 10^6 636 / 631, 2^28 2063 / 2059; u64 2^24 to 2^27, pairs and floats within 0.3 % either way.)
#define ILGPU_HIP_SORT_CODE_ALIGNED __attribute__((aligned(4096)))

// Tile of a group's k-th draw: its chunks are g, g + 8, g + 16, ... of
// 2^chunk_shift consecutive tiles.
__device__ __forceinline__ int ticket_tile(uint32_t k, uint32_t g, uint32_t groups, int chunk_shift) {
  const uint32_t chunk = (k >> chunk_shift) * groups + g;
  return (int)((chunk << chunk_shift) + (k & ((1u << chunk_shift) - 1u)));
}

// Sorts one tile by the digit of `pass` and scatters it.
template <int KEY_BYTES, int VALUE_BYTES, bool FLOAT_KEYS, bool FULL, bool HOT, int BLOCK, int ITEMS, bool AT_ONCE>
__device__ __forceinline__ void sort_tile(
    typename KeyOf<KEY_BYTES>::type (&key)[ITEMS],
    const typename KeyOf<KEY_BYTES>::type* __restrict__ src_keys,
    typename KeyOf<KEY_BYTES>::type* __restrict__ dst_keys,
    const typename ValueOf<VALUE_BYTES>::type* __restrict__ src_vals,
    typename ValueOf<VALUE_BYTES>::type* __restrict__ dst_vals,
    int64_t tile_base, int valid, int tile, int pass, const KeyXform& xf,
    const uint32_t* __restrict__ excl, uint32_t* status, int make_index,
    unsigned char* s_stage, uint32_t* s_global_off, uint32_t* s_scan,
    const uint32_t (&hot)[kMaxHot], uint32_t spin_limit, bool in_raw, bool out_raw) {
  using K = typename KeyOf<KEY_BYTES>::type;
  using Val = typename ValueOf<VALUE_BYTES>::type;
  using TileCfg = SortTile<KEY_BYTES, VALUE_BYTES, BLOCK, ITEMS>;
  constexpr int kItems = TileCfg::kItems;
  constexpr int kSubTiles = TileCfg::kSubTiles;
  constexpr bool kPairs = VALUE_BYTES > 0;
  constexpr int kValuesPerRound =
      kPairs ? TileCfg::kStageBytes / (VALUE_BYTES > 0 ? VALUE_BYTES : 1) : 1;
  constexpr int kRounds =
      kPairs ? (TileCfg::kTile + kValuesPerRound - 1) / kValuesPerRound : 0;
  static_assert(kItems % 2 == 0 && TileCfg::kTile <= 65536,
                "ranks and tile positions are packed two to a register");
  static_assert(kItems * kSubLanes < 65536, "a sub-tile's digit count fits 16 bits");

  // Counter of (sub-tile, digit): keys of that digit in the rows ranked so far.
  uint32_t* s_counter = reinterpret_cast<uint32_t*>(s_stage);
  K* s_keys = reinterpret_cast<K*>(s_stage);
  Val* s_vals = reinterpret_cast<Val*>(s_stage);

  // The thread index is made opaque per tile (and again for the write-out):
  // otherwise every per-item index derived from it is hoisted out of the
  // tile loop and held in a register of its own, dozens of them.
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int lane = tid & (kWaveSize - 1);
  const int wave = tid / kWaveSize;
  const int sub = wave;                     // sub-tile index in the block
  const int first_local = sub * TileCfg::kSubTileKeys + lane;
  const int shift = pass * 8;


  // Float keys travel between the passes in their ordered form: the first
  // pass that runs converts them as it ranks them (in_raw), the last one
  // converts them back as it writes them (out_raw), and in between a digit is
  // a shift and a mask.  Other keys keep their bits; their order is one xor.
  // (A pass that finds them converted applies the identity: no mask, no term.)
  KeyXform xf_in = xf;
  if (!in_raw) xf_in = KeyXform{0, 0, 0};
  auto digit = [&](K k) -> uint32_t {
    if constexpr (FLOAT_KEYS) return (uint32_t)(k >> shift) & (kRadix - 1);
    else return (uint32_t)((K)(k ^ (K)xf.xor_mask) >> shift) & (kRadix - 1);
  };
  // Keys past the end of the input take digit 255; they come last in memory
  // order, so they rank behind every real key and are dropped on write-out.
  auto item_digit = [&](int j) -> uint32_t {
    return (FULL || first_local + j * kSubLanes < valid) ? digit(key[j])
                                                          : (uint32_t)(kRadix - 1);
  };

  Val val[kPairs ? kItems : 1];
  if constexpr (kPairs) {
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const int local = first_local + j * kSubLanes;
      if (FULL || local < valid) {
        if (make_index) {
          val[j] = index_value<VALUE_BYTES>(tile_base + local, make_index);
        } else {
          val[j] = src_vals[tile_base + local];
        }
      }
    }
  }

  // Rank inside the sub-tile, later position inside the tile: 16 bits each.
  uint32_t* my_counters = s_counter + sub * kRadix;
  uint32_t packed[kItems / 2];
  // HOT: some digits hold a large share of the keys each (known from the
  // global histogram).  Their keys would all meet in one counter, and LDS
  // serialises the atomics of a wave to one address; they are ranked by one
  // ballot per such digit instead and only the other keys go through the
  // counters.
  uint32_t hot_count[kMaxHot] = {};  // keys of each hot digit in this sub-tile so far
  // Rows are ranked in groups: the LDS operations of a group are issued back
  // to back and their results consumed together, so a wave waits for one LDS
  // round trip per group, not per row.
  // (Pairs hold their values in registers too and take smaller groups.)
  constexpr int kGroup = kPairs ? ILGPU_HIP_SORT_PAIR_RANK_GROUP : ILGPU_HIP_SORT_RANK_GROUP;
  static_assert(kGroup % 2 == 0, "ranks are packed in pairs");
#pragma unroll
  for (int j0 = 0; j0 < kItems; j0 += kGroup) {
    uint32_t fetched[kGroup];   // what the LDS returned for the row
    uint32_t offset[kGroup];    // added to it: lane index of a one-digit row
    bool broadcast[kGroup];     // wave-uniform: take lane 0's result
#pragma unroll
    for (int g = 0; g < kGroup; ++g) {
      const int j = j0 + g;
      if (j >= kItems) break;
      const uint32_t d = item_digit(j);
      fetched[g] = 0;
      offset[g] = 0;
      broadcast[g] = false;
      bool through_counter = true;
      if constexpr (HOT) {
#pragma unroll
        for (int h = 0; h < kMaxHot; ++h) {
          if (hot[h] == kNoHotDigit) continue;  // wave-uniform
          const bool is_hot = d == hot[h];
          const uint64_t hot_lanes = __ballot(is_hot);
          if (is_hot) {
            offset[g] = hot_count[h] + (uint32_t)mbcnt(hot_lanes);
            through_counter = false;
          }
          hot_count[h] += (uint32_t)__popcll(hot_lanes);
        }
      } else {
        // Keys that arrive in runs put one digit into whole rows of a
        // sub-tile; the 64 atomics of such a row would meet in one word and
        // serialise.  In a row that is all one digit only lane 0 adds (the
        // whole row at once) and the others take its result plus their lane
        // index.  Passes with dominant digits leave the check out: the
        // ballots above already took their frequent digits.
        const uint32_t row_digit = (uint32_t)__builtin_amdgcn_readfirstlane((int)d);
        broadcast[g] = __ballot(d == row_digit) == ~0ull;
        if (broadcast[g]) {
          offset[g] = (uint32_t)lane;
          through_counter = lane == 0;
        }
      }
      if (through_counter)
        fetched[g] = __hip_atomic_fetch_add(my_counters + d,
                                            broadcast[g] ? (uint32_t)kSubLanes : 1u,
                                            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
#pragma unroll
    for (int g = 0; g < kGroup; ++g) {
      const int j = j0 + g;
      if (j >= kItems) break;
      uint32_t rank = fetched[g];
      if constexpr (!HOT) {
        if (broadcast[g]) rank = (uint32_t)__builtin_amdgcn_readfirstlane((int)rank);
      }
      rank += offset[g];
      if (j % 2 == 0) packed[j / 2] = rank;
      else packed[j / 2] |= rank << 16;
    }
    // Pin the packed ranks here: left alone, the compiler sinks the rank
    // arithmetic of all rows to where the ranks are used and keeps two live
    // registers per key until then.
#pragma unroll
    for (int g = 0; g < kGroup; g += 2)
      if (j0 + g < kItems) asm volatile("" : "+v"(packed[(j0 + g) / 2]));
  }
  if constexpr (HOT) {
#pragma unroll
    for (int h = 0; h < kMaxHot; ++h)  // these counters are untouched so far: still zero
      if (hot[h] != kNoHotDigit && lane == 0) my_counters[hot[h]] = hot_count[h];
  }
  __syncthreads();

  // One thread per digit: totals over the sub-tiles, look-back over the tiles.
  uint32_t count = 0, inc = 0;
  uint32_t* tile_status = status + (int64_t)tile * kRadix;
  if (tid < kRadix) {
#pragma unroll
    for (int s = 0; s < kSubTiles; ++s) count += s_counter[s * kRadix + tid];
    __hip_atomic_store(&tile_status[tid],
                       tile == 0 && !AT_ONCE ? status_prefix(count) : status_aggregate(count),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    inc = count;
#pragma unroll
    for (int s = 1; s < kWaveSize; s <<= 1) {
      const uint32_t o = shfl_up(inc, s);
      if (lane >= s) inc += o;
    }
    if (lane == kWaveSize - 1) s_scan[wave] = inc;
  }
  __syncthreads();
  // Digit threads: run starts, and the first step of the look-back is put in
  // flight; it is consumed after the keys are staged, so its round trip
  // overlaps the position and staging work of the whole block.
  uint32_t digit_start = 0;
  uint32_t first_step[kLookback];
  if (tid < kRadix) {
    digit_start = inc - count;
    for (int w = 0; w < wave; ++w) digit_start += s_scan[w];
    // Tile-local position of the first key of every (sub-tile, digit) run.
    {
      uint32_t run = digit_start;
#pragma unroll
      for (int s = 0; s < kSubTiles; ++s) {
        const uint32_t t = s_counter[s * kRadix + tid];
        s_counter[s * kRadix + tid] = run;
        run += t;
      }
    }
    if constexpr (!AT_ONCE) {
#pragma unroll
      for (int u = 0; u < kLookback; ++u) {
        const int idx = tile - 1 - u < 0 ? 0 : tile - 1 - u;
        first_step[u] = __hip_atomic_load(&status[(int64_t)idx * kRadix + tid],
                                          __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  __syncthreads();

  // Tile-local position of every key; afterwards the counters are dead and
  // the same LDS bytes stage the keys in digit order.
#pragma unroll
  for (int j = 0; j < kItems; j += 2) {
    const uint32_t p0 = my_counters[item_digit(j)] + (packed[j / 2] & 0xFFFFu);
    const uint32_t p1 = my_counters[item_digit(j + 1)] + (packed[j / 2] >> 16);
    packed[j / 2] = p0 | (p1 << 16);
    if (j % 8 == 6) __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kItems; ++j)
    s_keys[j % 2 == 0 ? packed[j / 2] & 0xFFFFu : packed[j / 2] >> 16] = key[j];

  // Keys of digit d in tile t, a full one, from the source.
  auto count_tile = [&](int t, uint32_t d) -> uint32_t {
    const K* other = src_keys + (int64_t)t * TileCfg::kTile;
    uint32_t c = 0;
#pragma unroll 4
    for (int i = 0; i < TileCfg::kTile; ++i) {
      K k = other[i];
      if constexpr (FLOAT_KEYS) k = ordered_bits(k, xf_in);
      c += digit(k) == d;
    }
    return c;
  };
  if constexpr (AT_ONCE) {
    static_assert(BLOCK == 2 * kRadix, "two halves of a thread per digit");
    // Every tile publishes its counts at about the same time, so a walk would meet nothing but counts and take as
    // many round trips as its tile has predecessors in fours.  Instead one half of the block sums
    // the counts of the tiles in front within the group, the other those of the groups in front: two round
    // trips behind each other, since the group's last tile sums its group before the others see it.
    // (Inside a pass of 2^21 u32 keys, 342 tiles, the slowest tile waits 4 us for it instead of 7.6.  Sorts with a copy
    // in front, us, a walk / this: u32 keys 2^20 55.0 / 48.9, 2^21 69.4 / 63.2, below 10^6 2^20 63.1 / 53.6; normal floats
    // 2^20 74.1 / 64.7; pairs of 2^21 u32 85.2 / 77.4, 2^20 Zipf 60.5 / 53.4, of 2^20 u64 with u32 85.7 / 79.2; u16 keys 600 000 35.2 / 30.4, 2^20
    // 39.1 / 32.6, 3 * 10^6 54.2 / 45.0; u8 keys 600 000 28.1 / 26.0, 2^20 30.6 / 27.7, 3 * 10^6 38.0 / 33.5; but 130 000 u16 32.4 / 33.0 and u8 26.7 / 27.2.)
    const uint32_t d = (uint32_t)tid & (kRadix - 1);
    const bool groups = __builtin_amdgcn_readfirstlane(tid) >= kRadix;
    const int group = tile / kLookGroup;
    const int span = groups ? kLookGroup : 1;                       // tiles that a word stands for
    const int words = groups ? group : tile % kLookGroup;           // to be summed
    const int first = groups ? kLookGroup - 1 : group * kLookGroup;  // row of the first one
    // A count has the top bits 11, a group's 10: with this added it is at least kStatusAggregate, and
    // anything else is not.
    const uint32_t to_aggregate = groups ? kStatusAggregate - kStatusGroup : 0u;
    auto word = [&](int row) -> uint32_t {
      return __hip_atomic_load(&status[(int64_t)row * kRadix + d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    uint32_t before = groups ? excl[pass * kRadix + d] : 0u;
    for (int at = 0; at < words; at += kLookGroup) {
      uint32_t sum;
      for (uint32_t polls = 0;; ++polls) {
        uint32_t w[kLookGroup], least = ~0u;
#pragma unroll
        for (int u = 0; u < kLookGroup; ++u) w[u] = word(first + (at + u < words ? at + u : at) * span);
        sum = 0;
#pragma unroll
        for (int u = 0; u < kLookGroup; ++u) {
          least = min(least, w[u] + to_aggregate);
          sum += w[u] & (at + u < words ? kStatusCountMask : 0u);
        }
        if (least >= kStatusAggregate) break;
        if (polls >= spin_limit) {
          // A tile may not be running (see below): what has not been published is counted.
          sum = 0;
          for (int u = at; u < words && u < at + kLookGroup; ++u) {
            const int row = first + u * span;
            const uint32_t whole = word(row);
            if (whole + to_aggregate >= kStatusAggregate) {
              sum += whole & kStatusCountMask;
              continue;
            }
            uint32_t of_row = 0;
            for (int t = row - (span - 1); t <= row; ++t) {
              const uint32_t one = word(t);
              if (one != 0u && !status_is_aggregate(one)) of_row = 0;  // the group's last tile has summed it by now
              of_row += one != 0u ? one & kStatusCountMask : count_tile(t, d);
            }
            sum += of_row;
          }
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
      before += sum;
    }
    if (groups) s_global_off[d] = before;
    else if (tile % kLookGroup == kLookGroup - 1)
      __hip_atomic_store(&tile_status[d], status_group(before + count), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (!groups) s_global_off[d] += before - digit_start;
  } else if (tid < kRadix) {
    // Keys with this digit in earlier tiles: walk back over the status words,
    // kLookback tiles per step.  The loads of a step are unconditional (index
    // clamped) so that they are in flight together; positions in front of
    // tile 0 read as an empty inclusive prefix.  Where a step chose for every word between the load and first_step, the
    // compiler waited for one before it issued the next.  So keys alone have a step's loads at the end of the one in front
    // of it, and pairs, whose registers that spills, one choice for all the words of a step.
    // (Sorts with a copy in front, us, word by word / at the end / one choice: 10^7 normal doubles 331 / 321 / 321, 20 000 003 normal
    // floats 277 / 265 / 272, 14 * 10^6 u32 below 10^6 175 / 171 / 172; pairs of 8 * 10^6 u32 173 / 169 / 169, of 2^26 u32 below 10^6 with
    // their index 1051 / 1034 / 1035, of 12 * 10^6 normal doubles with bytes 451 / 461 / 450.)
    uint32_t before = 0;
    bool done = tile == 0;
    uint32_t s[kLookback];
    if constexpr (!kPairs) {
#pragma unroll
      for (int u = 0; u < kLookback; ++u) s[u] = first_step[u];
    }
    bool preloaded = true;
    for (int t = tile - 1; !done; t -= kLookback) {
      if constexpr (kPairs) {
        if (preloaded) {
#pragma unroll
          for (int u = 0; u < kLookback; ++u) s[u] = first_step[u];
        } else {
#pragma unroll
          for (int u = 0; u < kLookback; ++u) {
            const int idx = t - u < 0 ? 0 : t - u;
            s[u] = __hip_atomic_load(&status[(int64_t)idx * kRadix + tid], __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
          }
        }
        preloaded = false;
      }
#pragma unroll
      for (int u = 0; u < kLookback; ++u)
        if (t - u < 0) s[u] = status_prefix(0u);
#pragma unroll
      for (int u = 0; u < kLookback; ++u) {
        if (done) continue;
        uint32_t polls = 0;
        while (s[u] == 0u) {
          if (polls++ >= spin_limit) {
            // Nobody has published tile t - u: its owner may not be running.
            // Count this thread's digit in that tile from the source keys (a
            // full tile: it precedes this one) and go on as if the tile had
            // published its own count.  Slow, and never needed while every
            // group of blocks is resident.
            s[u] = status_aggregate(count_tile(t - u, (uint32_t)tid));
            break;
          }
          __builtin_amdgcn_s_sleep(1);
          s[u] = __hip_atomic_load(&status[(int64_t)(t - u) * kRadix + tid],
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        before += status_value(s[u]);
        done = !status_is_aggregate(s[u]);
      }
      if constexpr (!kPairs) {
        if (done) break;
#pragma unroll
        for (int u = 0; u < kLookback; ++u) {
          const int next = t - kLookback - u;
          s[u] = __hip_atomic_load(&status[(int64_t)(next < 0 ? 0 : next) * kRadix + tid],
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    }
    if (tile > 0)
      __hip_atomic_store(&tile_status[tid], status_prefix(before + count),
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_global_off[tid] = excl[pass * kRadix + tid] + before - digit_start;
  }
  __syncthreads();

  uint32_t gpos[kPairs ? kItems : 1];
  asm volatile("" : "+v"(tid));
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const int i = j * BLOCK + tid;
    if (FULL || i < valid) {
      const K k = s_keys[i];
      const uint32_t g = s_global_off[digit(k)] + (uint32_t)i;
      if constexpr (FLOAT_KEYS) dst_keys[g] = out_raw ? raw_bits(k, xf) : k;
      else dst_keys[g] = k;
      if constexpr (kPairs) gpos[j] = g;
    }
    constexpr int kWriteGroup = kPairs ? ILGPU_HIP_SORT_PAIR_WRITE_GROUP : ILGPU_HIP_SORT_WRITE_GROUP;
    if (j % kWriteGroup == kWriteGroup - 1) __builtin_amdgcn_sched_barrier(0);
  }

  if constexpr (kPairs) {
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
      const uint32_t lo = (uint32_t)r * kValuesPerRound;
      __syncthreads();  // the stage buffer is free again
#pragma unroll
      for (int j = 0; j < kItems; ++j) {
        const uint32_t pos = j % 2 == 0 ? packed[j / 2] & 0xFFFFu : packed[j / 2] >> 16;
        if (pos - lo < (uint32_t)kValuesPerRound) s_vals[pos - lo] = val[j];
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < kItems; ++j) {
        const uint32_t i = (uint32_t)(j * BLOCK + tid);
        if ((FULL || i < (uint32_t)valid) && i - lo < (uint32_t)kValuesPerRound)
          dst_vals[gpos[j]] = s_vals[i - lo];
      }
    }
  }
}

// AT_ONCE: one tile per block, which is not handed out (see below), and a look-back for tiles that all run at the same
// time.
template <int KEY_BYTES, int VALUE_BYTES, bool FLOAT_KEYS, int BLOCK, int ITEMS, bool AT_ONCE>
__global__ __launch_bounds__(BLOCK, ILGPU_HIP_SORT_WAVES_PER_EU) ILGPU_HIP_SORT_CODE_ALIGNED
void onesweep_kernel(
    typename KeyOf<KEY_BYTES>::type* keys_a,
    typename KeyOf<KEY_BYTES>::type* keys_b,
    typename ValueOf<VALUE_BYTES>::type* vals_a,
    typename ValueOf<VALUE_BYTES>::type* vals_b, int64_t n, int pass,
    KeyXform xf, const uint32_t* __restrict__ excl, uint32_t* all_status,
    uint32_t* ticket, const SortPlan* __restrict__ plan, int num_tiles,
    int values_from_index, int groups, int chunk_shift, uint32_t spin_limit) {
  using K = typename KeyOf<KEY_BYTES>::type;
  using Val = typename ValueOf<VALUE_BYTES>::type;
  using TileCfg = SortTile<KEY_BYTES, VALUE_BYTES, BLOCK, ITEMS>;
  constexpr int kTile = TileCfg::kTile;
  constexpr int kItems = TileCfg::kItems;

  __shared__ __attribute__((aligned(16))) unsigned char s_stage[TileCfg::kStageBytes];
  __shared__ uint32_t s_global_off[kRadix];
  __shared__ uint32_t s_scan[kRadix / kWaveSize];
  __shared__ int s_tile;

  if (plan->skip[pass]) return;
  const bool src_alt = plan->src_is_alt[pass] != 0;
  constexpr bool kTurns = sort_status_turns(KEY_BYTES, BLOCK, AT_ONCE,
                                            FLOAT_KEYS && KEY_BYTES == 4 && VALUE_BYTES == 0 && ITEMS == kFloatItems);
  const int64_t region_words = (int64_t)num_tiles * kRadix;
  uint32_t* status = all_status + (kTurns ? (src_alt ? region_words : 0) : pass * region_words);
  // (A block of one tile does it when the tile is done: the others wait for its counts.)
  if constexpr (kTurns && !AT_ONCE) clear_next_status(all_status, region_words, plan, pass, BLOCK);
  uint32_t hot[kMaxHot];
#pragma unroll
  for (int h = 0; h < kMaxHot; ++h) hot[h] = plan->hot[pass][h];
  const K* src_keys = src_alt ? keys_b : keys_a;
  K* dst_keys = src_alt ? keys_a : keys_b;
  const Val* src_vals = src_alt ? vals_b : vals_a;
  Val* dst_vals = src_alt ? vals_a : vals_b;
  // 0, or the kind of index values the first pass that runs generates
  const int make_index =
      VALUE_BYTES > 0 && plan->first_executed == (uint32_t)pass ? values_from_index : 0;
  const bool in_raw = plan->first_executed == (uint32_t)pass;
  const bool out_raw = plan->last_executed == (uint32_t)pass;
  const int tid = threadIdx.x;
  const int first_local = (tid / kSubLanes) * TileCfg::kSubTileKeys + tid % kSubLanes;

  auto valid_keys = [&](int t) -> int {
    const int64_t remaining = n - (int64_t)t * kTile;
    return remaining >= kTile ? kTile : (remaining > 0 ? (int)remaining : 0);
  };

  // Tickets: group g (= blockIdx % 8) owns the chunks g, g + 8, g + 16, ... of
  // 2^chunk_shift consecutive tiles and draws their tiles in order from its
  // own counter.  Unlike a single counter this does not start tiles in index
  // order across groups: a tile can find that a predecessor owned by another
  // group has not been started, and if that group had no resident block it
  // would wait for ever.  The look-back therefore never waits without bound:
  // after spin_limit polls of an empty word it counts the tile's digit itself
  // (sort_tile), so every block finishes whatever the other blocks do.
  // A block draws its next tile only when it is about to start it: the time
  // between a tile's ticket and the publication of its digit counts is what
  // every later tile's look-back waits for.  (Drawing it earlier, to load the
  // next keys during the look-back and the write-out, measured 3 to 12 % slower,
  // with the global ticket and again with the per-group ones.)  The key loads
  // fly while the ranking counters are cleared.
  // A grid of as many blocks as there are tiles (a short input) needs no
  // tickets (ticket == nullptr): block b takes tile b and is done, which saves
  // a pass two round trips to the ticket, one of them only to learn that
  // there is nothing left.  Blocks start in index order in practice, so a
  // tile's predecessors are running; where they are not, the bounded look-back
  // covers that as it does with tickets.
  for (int round = 0;; ++round) {
    int tile;
    if (AT_ONCE || ticket == nullptr) {
      if (round > 0) break;
      tile = (int)blockIdx.x;
    } else {
      if (tid == 0) {
        const uint32_t g = blockIdx.x % (uint32_t)groups;
        s_tile = ticket_tile(atomicAdd(ticket + g * kTicketStride, 1u), g, (uint32_t)groups, chunk_shift);
      }
      __syncthreads();  // also: the previous tile's staged keys have been read
      tile = s_tile;
    }
    if (tile >= num_tiles) break;
    const int64_t tile_base = (int64_t)tile * kTile;
    const int valid = valid_keys(tile);
    // Three instantiations of the tile code: full tiles with and without
    // dominant digits, and the tail tile (bounds-checked; the dominant-digit
    // form serves it either way: without such digits every key goes through
    // the counters).  Each loads its keys itself, so that the loads, the
    // clearing of the counters and the ranking are one straight line and the
    // rows are ranked as their keys arrive.
    auto run = [&](auto full, auto with_hot) {
      constexpr bool kFull = decltype(full)::value;
      constexpr bool kHot = decltype(with_hot)::value;
      K key[kItems];
      load_tile_keys<KEY_BYTES, kItems, kFull>(src_keys, tile_base, valid, first_local, key);
      if constexpr (FLOAT_KEYS) {
        if (in_raw) {
#pragma unroll
          for (int j = 0; j < kItems; ++j) key[j] = ordered_bits(key[j], xf);
        }
      }
      {  // clear the ranking counters
        uint4* z = reinterpret_cast<uint4*>(s_stage);
        for (int i = tid; i < TileCfg::kCounterBytes / 16; i += BLOCK)
          z[i] = make_uint4(0u, 0u, 0u, 0u);
      }
      __syncthreads();
      sort_tile<KEY_BYTES, VALUE_BYTES, FLOAT_KEYS, kFull, kHot, BLOCK, ITEMS, AT_ONCE>(
          key, src_keys, dst_keys, src_vals, dst_vals, tile_base, valid, tile, pass, xf, excl,
          status, make_index, s_stage, s_global_off, s_scan, hot, spin_limit, in_raw, out_raw);
    };
    if (valid != kTile) run(std::false_type{}, std::true_type{});
    else if (hot[0] == kNoHotDigit) run(std::true_type{}, std::false_type{});
    else run(std::true_type{}, std::true_type{});
  }
  if constexpr (kTurns && AT_ONCE) clear_next_status(all_status, region_words, plan, pass, BLOCK);
}

// ---- onesweep pass, pipelined form (keys without values, large inputs) --------
// The pass above runs a tile's phases one after the other: while a block waits
// for its keys nothing else happens on its compute unit, and while it ranks,
// walks and stages, no load is in flight.  This form overlaps them.
//
//   * The write-out of a tile is deferred until the next tile is ranked.  Per
//     tile: positions and staging of tile T (its keys leave the registers),
//     load and ranking of the block's next tile T', digit totals of T'
//     published, T written out from LDS, and so on.  The stores of T drain
//     while T' is staged and T'' is loaded; T is resolved (the digit counts of
//     all earlier tiles) while T' is loaded and ranked.
//   * A 1024-thread block is fifteen waves that sort and one that resolves.
//     The sorting waves hold the keys (15 x 64 x kItems per tile).  The other
//     wave holds none and hands the 256 global offsets of a tile over through
//     LDS.  A wave that sorts could not do this beside its loads: vector memory
//     results return to a wave, and to a compute unit, in request order, so a
//     status word asked for behind a tile of keys arrives behind the keys.  For
//     the same reason a look-back step on a compute unit that streams keys
//     takes three times what it takes on an idle one, and a walk of the usual
//     depth (thirty tiles) would outlast the tile.
//   * So the walking is done elsewhere.  Four blocks of the grid sort nothing:
//     their compute units issue no key traffic and their memory round trips are
//     short.  Each takes 64 of the 256 digits and turns the published counts of
//     the tiles into inclusive prefixes, in tile order, a window of 64 tiles per
//     round trip.  A sorting block's sixteenth wave only polls the row of its
//     own tile until the prefixes are there.  Every status row is read by the
//     scanning blocks and by its owner, not by the thirty tiles behind it.
//     Nothing waits without bound: a wave that has polled its row often enough
//     walks back itself (pipelined_walk), and a scanning block that waits for a
//     tile nobody publishes counts that tile's digits itself.
//   * A tile's digit counts are published a fixed time after its ticket is
//     drawn (staging of the previous tile, load, ranking), whatever any other
//     block does and however long the tile before takes to be resolved: a
//     ticket commits the block to the tile, and every later tile waits for
//     those counts.  That is why the sorting waves never meet the sixteenth
//     wave inside their own steps: among themselves they synchronise through
//     counters in LDS (arrive: one add by a wave's first lane; wait: poll), and
//     the block-wide barrier is used once per tile, where the offsets of the
//     tile before are handed over.
//   * The ranking counters have LDS of their own (the tile is 1/16 shorter,
//     which frees it): a wave clears its counters itself as soon as it has read
//     its run starts, and no barrier separates positions from staging.
//
// Floating-point keys are converted by the first pass that runs and back by
// the last one (in_xf, out_xf in the kernel); pairs take the pass above.
template <int KEY_BYTES> struct PipelinedTile {
  static constexpr int kBlock = 1024;
  static constexpr int kSorterWaves = kBlock / kWaveSize - 1;
  static constexpr int kSorters = kSorterWaves * kWaveSize;
  static constexpr int kItems = items_per_thread(KEY_BYTES, 0);
  static constexpr int kSubTileKeys = kWaveSize * kItems;
  static constexpr int kTile = kSorterWaves * kSubTileKeys;
};
constexpr int pipelined_tile_keys(int key_bytes) {
  return (1024 / kWaveSize - 1) * kWaveSize * items_per_thread(key_bytes, 0);
}
#ifndef ILGPU_HIP_SORT_WALK_STEP
#define ILGPU_HIP_SORT_WALK_STEP 4
#endif
constexpr int kWalkStep = ILGPU_HIP_SORT_WALK_STEP;   // tiles per look-back step of a resolving wave that walks back itself
constexpr int kWalkDigits = kRadix / kWaveSize;       // digits per lane of a resolving wave

// Loads the calling wave's keys of one tile into `key` and ranks them on the
// wave's counters, which are zero on entry: as in sort_tile.
template <int KEY_BYTES, bool FULL, bool HOT, bool FLOAT_KEYS>
__device__ __forceinline__ void pipelined_rank(
    typename KeyOf<KEY_BYTES>::type (&key)[(items_per_thread(KEY_BYTES, 0))],
    uint32_t (&packed)[(items_per_thread(KEY_BYTES, 0)) / 2],
    const typename KeyOf<KEY_BYTES>::type* __restrict__ src_keys, int64_t tile_base, int valid,
    int shift, const KeyXform& in_xf, uint32_t* my_counters, int lane, int first_local,
    const uint32_t (&hot)[kMaxHot]) {
  using K = typename KeyOf<KEY_BYTES>::type;
  constexpr int kItems = items_per_thread(KEY_BYTES, 0);
  // Rows whose loads are issued before the ranking starts; the others follow
  // one rank group at a time.
  constexpr int kAhead = ILGPU_HIP_SORT_LOAD_AHEAD < kItems ? ILGPU_HIP_SORT_LOAD_AHEAD : kItems;
  auto load_rows = [&](int j0, int j1) {
#pragma unroll
    for (int j = j0; j < j1 && j < kItems; ++j) {
      const int local = first_local + j * kWaveSize;
      if (FULL || local < valid)
        key[j] = ILGPU_HIP_SORT_NT_LOAD ? __builtin_nontemporal_load(&src_keys[tile_base + local])
                                        : src_keys[tile_base + local];
      else key[j] = 0;
    }
  };
  load_rows(0, kAhead);
  if (kAhead < kItems) __builtin_amdgcn_sched_barrier(0);
  // Float keys leave this function in their ordered form (in_xf is the
  // identity when they arrive in it); integer keys keep their bits.
  auto item_digit = [&](int j) -> uint32_t {
    if constexpr (FLOAT_KEYS) key[j] = ordered_bits(key[j], in_xf);
    const K o = FLOAT_KEYS ? key[j] : (K)(key[j] ^ (K)in_xf.xor_mask);
    const uint32_t d = (uint32_t)(o >> shift) & (kRadix - 1);
    return (FULL || first_local + j * kWaveSize < valid) ? d : (uint32_t)(kRadix - 1);
  };
  uint32_t hot_count[kMaxHot] = {};
  constexpr int kGroup = ILGPU_HIP_SORT_RANK_GROUP;
  static_assert(kGroup % 2 == 0, "ranks are packed in pairs");
#pragma unroll
  for (int j0 = 0; j0 < kItems; j0 += kGroup) {
    uint32_t fetched[kGroup];
    uint32_t offset[kGroup];
    bool broadcast[kGroup];
    if (kAhead < kItems) {
      load_rows(kAhead + j0, kAhead + j0 + kGroup);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int g = 0; g < kGroup; ++g) {
      const int j = j0 + g;
      if (j >= kItems) break;
      const uint32_t d = item_digit(j);
      fetched[g] = 0;
      offset[g] = 0;
      broadcast[g] = false;
      bool through_counter = true;
      if constexpr (HOT) {
#pragma unroll
        for (int h = 0; h < kMaxHot; ++h) {
          if (hot[h] == kNoHotDigit) continue;  // wave-uniform
          const bool is_hot = d == hot[h];
          const uint64_t hot_lanes = __ballot(is_hot);
          if (is_hot) {
            offset[g] = hot_count[h] + (uint32_t)mbcnt(hot_lanes);
            through_counter = false;
          }
          hot_count[h] += (uint32_t)__popcll(hot_lanes);
        }
      } else {
        const uint32_t row_digit = (uint32_t)__builtin_amdgcn_readfirstlane((int)d);
        broadcast[g] = __ballot(d == row_digit) == ~0ull;
        if (broadcast[g]) {
          offset[g] = (uint32_t)lane;
          through_counter = lane == 0;
        }
      }
      if (through_counter)
        fetched[g] = __hip_atomic_fetch_add(my_counters + d,
                                            broadcast[g] ? (uint32_t)kWaveSize : 1u,
                                            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
#pragma unroll
    for (int g = 0; g < kGroup; ++g) {
      const int j = j0 + g;
      if (j >= kItems) break;
      uint32_t rank = fetched[g];
      if constexpr (!HOT) {
        if (broadcast[g]) rank = (uint32_t)__builtin_amdgcn_readfirstlane((int)rank);
      }
      rank += offset[g];
      if (j % 2 == 0) packed[j / 2] = rank;
      else packed[j / 2] |= rank << 16;
    }
#pragma unroll
    for (int g = 0; g < kGroup; g += 2)
      if (j0 + g < kItems) asm volatile("" : "+v"(packed[(j0 + g) / 2]));
  }
  if constexpr (HOT) {
#pragma unroll
    for (int h = 0; h < kMaxHot; ++h)  // these counters are untouched so far: still zero
      if (hot[h] != kNoHotDigit && lane == 0) my_counters[hot[h]] = hot_count[h];
  }
}

// A resolving wave that walks back itself: the digit counts of all earlier tiles by
// look-back, the tile's inclusive counts published, the global offsets of its
// 256 runs into s_global_off.  Lane l owns digits 4l .. 4l+3, so a tile's
// status row is one 16-byte load per lane: the time of a look-back step grows
// with the number of load instructions in it, not with their width.
typedef uint32_t StatusVec __attribute__((ext_vector_type(4)));
constexpr int kStatusCoherent = 16;  // cache policy of the buffer operations: sc1, agent scope
__device__ __forceinline__ StatusVec load_status_row(__amdgpu_buffer_rsrc_t rsrc, int tile,
                                                      int lane) {
  return __builtin_amdgcn_raw_buffer_load_b128(rsrc, (tile * kRadix + lane * kWalkDigits) * 4, 0,
                                               kStatusCoherent);
}

template <int KEY_BYTES, bool FLOAT_KEYS>
__device__ __forceinline__ void pipelined_walk(
    const typename KeyOf<KEY_BYTES>::type* __restrict__ src_keys, int tile, int shift,
    const KeyXform& in_xf, __amdgpu_buffer_rsrc_t status,
    const uint32_t* __restrict__ excl_row, const uint32_t* s_total, const uint32_t* s_start,
    uint32_t* s_global_off, int lane, uint32_t spin_limit) {
  using K = typename KeyOf<KEY_BYTES>::type;
  constexpr int kTile = PipelinedTile<KEY_BYTES>::kTile;
  static_assert(kWalkDigits == 4, "a lane's digits are one 16-byte vector");
  auto digit = [&](K k) -> uint32_t {  // of a key as the source holds it
    const K o = FLOAT_KEYS ? ordered_bits(k, in_xf) : (K)(k ^ (K)in_xf.xor_mask);
    return (uint32_t)(o >> shift) & (kRadix - 1);
  };
  const StatusVec my_count = reinterpret_cast<const StatusVec*>(s_total)[lane];
  const StatusVec my_excl = reinterpret_cast<const StatusVec*>(excl_row)[lane];
  uint32_t before[kWalkDigits];
  bool done[kWalkDigits];
#pragma unroll
  for (int c = 0; c < kWalkDigits; ++c) {
    before[c] = 0;
    done[c] = tile == 0;
  }
  for (int t = tile - 1; t >= 0; t -= kWalkStep) {
    bool all_done = true;
#pragma unroll
    for (int c = 0; c < kWalkDigits; ++c) all_done = all_done && done[c];
    if (__all(all_done)) break;
    // The loads of a step are unconditional (index clamped) so that they are in
    // flight together; positions in front of tile 0 read as an empty prefix.
    StatusVec s[kWalkStep];
#pragma unroll
    for (int u = 0; u < kWalkStep; ++u)
      s[u] = load_status_row(status, t - u < 0 ? 0 : t - u, lane);
#pragma unroll
    for (int u = 0; u < kWalkStep; ++u) {
      if (t - u < 0) s[u] = StatusVec{status_prefix(0u), status_prefix(0u), status_prefix(0u),
                                      status_prefix(0u)};
      // Words of tile t - u that this lane still needs and that are empty:
      // the tile's row is polled until they are there, never without bound.
      uint32_t polls = 0;
      while (true) {
        bool missing = false;
#pragma unroll
        for (int c = 0; c < kWalkDigits; ++c) missing = missing || (!done[c] && s[u][c] == 0u);
        if (!__any(missing)) break;
        if (polls++ >= spin_limit) {
          // Nobody has published tile t - u: its owner may not be running.
          // Count the digits of that (full) tile from the source keys and go
          // on as if the tile had published its own counts.  Slow, and never
          // needed while every group of blocks is resident.
          const K* other = src_keys + (int64_t)(t - u) * kTile;
          uint32_t cnt[kWalkDigits] = {};
#pragma unroll 4
          for (int i = 0; i < kTile; ++i) {
            K k = other[i];
            const uint32_t d = digit(k);
#pragma unroll
            for (int c = 0; c < kWalkDigits; ++c) cnt[c] += d == (uint32_t)(lane * kWalkDigits + c);
          }
#pragma unroll
          for (int c = 0; c < kWalkDigits; ++c)
            if (s[u][c] == 0u) s[u][c] = status_aggregate(cnt[c]);
          break;
        }
        __builtin_amdgcn_s_sleep(1);
        s[u] = load_status_row(status, t - u, lane);
      }
#pragma unroll
      for (int c = 0; c < kWalkDigits; ++c) {
        if (!done[c]) {
          before[c] += status_value(s[u][c]);
          done[c] = !status_is_aggregate(s[u][c]);
        }
      }
    }
  }
  StatusVec prefix, offset;
  const StatusVec start = reinterpret_cast<const StatusVec*>(s_start)[lane];
#pragma unroll
  for (int c = 0; c < kWalkDigits; ++c) {
    prefix[c] = status_prefix(before[c] + my_count[c]);
    offset[c] = my_excl[c] + before[c] - start[c];
  }
  if (tile > 0)
    __builtin_amdgcn_raw_buffer_store_b128(prefix, status, (tile * kRadix + lane * kWalkDigits) * 4,
                                           0, kStatusCoherent);
  reinterpret_cast<StatusVec*>(s_global_off)[lane] = offset;
}

#ifndef ILGPU_HIP_SORT_OWN_ROW_SLEEP
#define ILGPU_HIP_SORT_OWN_ROW_SLEEP 20
#endif
// Rows (tiles) a scanning block takes per round trip: four per wave, and as
// many again requested ahead.  (A wave with more than about 24 dwords per lane
// in flight stalls: measured.)
#ifndef ILGPU_HIP_SORT_SCAN_SEG_ROWS
#define ILGPU_HIP_SORT_SCAN_SEG_ROWS 4
#endif
constexpr int kScanSegRows = ILGPU_HIP_SORT_SCAN_SEG_ROWS;
constexpr int kScanSegs = 16;
constexpr int kScanWindow = kScanSegs * kScanSegRows;
constexpr int kScanBlocks = kRadix / kWaveSize;  // one scanning block per 64 digits
// Polls of its own row before a resolving wave stops waiting for the scanning
// block and walks back itself.
constexpr uint32_t kScannerPolls = 64;

// A scanning block's loop: status words of the tiles in order, counts into
// inclusive prefixes, for the 64 digits of the block (lane = digit).  Wave w
// takes the rows 4w .. 4w+3 of a window of 64 tiles: one round trip reads the
// window, the rows that are complete at its front are scanned (four rows per
// thread in registers, the sixteen waves combined through LDS) and their
// prefixes written back.  A row's word either adds its count or (tile 0, or a
// tile whose owner walked back itself) sets the running value.
// s_lds: 16 + 17 x 64 words.
template <int KEY_BYTES, bool FLOAT_KEYS>
__device__ __forceinline__ void pipelined_scan(
    const typename KeyOf<KEY_BYTES>::type* __restrict__ src_keys, int shift,
    const KeyXform& in_xf, uint32_t* status, int num_tiles, uint32_t spin_limit,
    uint32_t* s_lds) {
  using K = typename KeyOf<KEY_BYTES>::type;
  constexpr int kTile = PipelinedTile<KEY_BYTES>::kTile;
  uint32_t* s_avail = s_lds;                          // [segments]: leading complete rows of every wave's segment
  uint32_t* s_part = s_lds + kScanSegs;               // [segments][64]: what a segment's rows do to the running value
  uint32_t* s_prefix = s_part + kScanSegs * kWaveSize;  // [64]: the running inclusive counts
  static_assert(kScanSegs * kWaveSize >= kRadix, "the fallback counts 256 digit values in s_part");
  constexpr uint32_t kAbsolute = 0x80000000u; // a segment that sets the running value
  const int tid = threadIdx.x;
  const int lane = tid & (kWaveSize - 1);
  const int wave = tid / kWaveSize;
  const int quarter = blockIdx.x;  // this block's 64 digits
  const int seg = wave;            // this wave's rows of the window
  const int dgt = quarter * kWaveSize + lane;
  auto combine = [&](uint32_t running, uint32_t part) -> uint32_t {
    return (part & kAbsolute) ? (part & ~kAbsolute) : running + part;
  };
  if (seg == 0) s_prefix[lane] = 0u;
  __syncthreads();
  uint32_t polls = 0;
  int t = 0;
  uint32_t w[kScanSegRows], w_next[kScanSegRows];
  bool ahead = false;  // w already holds the window at t
  auto load_window = [&](int first_tile, uint32_t (&words)[kScanSegRows]) {
#pragma unroll
    for (int u = 0; u < kScanSegRows; ++u) {
      int row = first_tile + seg * kScanSegRows + u;
      row = row < num_tiles ? row : num_tiles - 1;
      words[u] = __hip_atomic_load(&status[(int64_t)row * kRadix + dgt], __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
    }
  };
  while (t < num_tiles) {
    const int first_row = t + seg * kScanSegRows;
    // The window was requested by the previous turn if that consumed a whole
    // window (the scan is behind and the rows are there); the next one is
    // requested before this one is worked on, so that its round trip runs
    // beside the scan and ahead of this window's stores.
    if (!ahead) load_window(t, w);
    load_window(t + kScanWindow, w_next);
    int there = 0;  // complete rows at the front of this wave's segment (wave-uniform)
    bool open = true;
#pragma unroll
    for (int u = 0; u < kScanSegRows; ++u) {
      open = open && first_row + u < num_tiles && __all(w[u] != 0u);
      there += open ? 1 : 0;
    }
    if (lane == 0) s_avail[seg] = (uint32_t)there;
    __syncthreads();
    // Complete rows at the front of the window.
    int avail = 0;
    {
      bool full = true;
#pragma unroll
      for (int g = 0; g < kScanSegs; ++g) {
        const int a = (int)s_avail[g];
        avail += full ? a : 0;
        full = full && a == kScanSegRows;
      }
    }
    int mine = avail - seg * kScanSegRows;  // rows of this segment that are consumed
    mine = mine < 0 ? 0 : (mine > kScanSegRows ? kScanSegRows : mine);
    uint32_t value = 0;
    bool absolute = false;
    uint32_t was_aggregate = 0;  // bit u: row u held a count
#pragma unroll
    for (int u = 0; u < kScanSegRows; ++u) {
      if (u < mine) {
        if (status_is_aggregate(w[u])) {
          value += w[u] & kStatusCountMask;
          was_aggregate |= 1u << u;
        } else {
          value = w[u] - 1u;
          absolute = true;
        }
      }
      // From here w[u] is the running value within the segment, and whether it
      // is already absolute rides in the top bit.
      w[u] = value | (absolute ? kAbsolute : 0u);
    }
    s_part[seg * kWaveSize + lane] = value | (absolute ? kAbsolute : 0u);
    __syncthreads();
    uint32_t running = s_prefix[lane];
    uint32_t base = running;
#pragma unroll
    for (int g = 0; g < kScanSegs; ++g) {
      const uint32_t part = s_part[g * kWaveSize + lane];
      if (g < seg) base = combine(base, part);
      running = combine(running, part);
    }
#pragma unroll
    for (int u = 0; u < kScanSegRows; ++u) {
      if (u < mine && ((was_aggregate >> u) & 1u))
        __hip_atomic_store(&status[(int64_t)(first_row + u) * kRadix + dgt],
                           status_prefix(combine(base, w[u])), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();  // the segment results and the running counts have been read
    if (seg == 0) s_prefix[lane] = running;
    t += avail;
    ahead = avail == kScanWindow;
    if (ahead) {
#pragma unroll
      for (int u = 0; u < kScanSegRows; ++u) w[u] = w_next[u];
    }
    if (avail != 0) {
      polls = 0;
    } else if (polls++ >= spin_limit) {
      // Nobody has published tile t: its owner may not be running.  Count its
      // digits from the source keys (a full tile: the last one is left to its
      // owner) and go on; the owner, if it ever runs, resolves itself.  Slow,
      // and never needed while every block is resident.
      if (t == num_tiles - 1) return;
      if (tid < kRadix) s_part[tid] = 0u;
      __syncthreads();
      const K* other = src_keys + (int64_t)t * kTile;
      for (int i = tid; i < kTile; i += kScanSegs * kWaveSize) {
        const K k = other[i];
        const K o = FLOAT_KEYS ? ordered_bits(k, in_xf) : (K)(k ^ (K)in_xf.xor_mask);
        atomicAdd(&s_part[(uint32_t)(o >> shift) & (kRadix - 1)], 1u);
      }
      __syncthreads();
      if (seg == 0) s_prefix[lane] += s_part[dgt];
      __syncthreads();
      ++t;
      polls = 0;
    } else {
      __builtin_amdgcn_s_sleep(2);
    }
  }
}

template <int KEY_BYTES, bool FLOAT_KEYS>
__global__ __launch_bounds__(1024, ILGPU_HIP_SORT_WAVES_PER_EU) ILGPU_HIP_SORT_CODE_ALIGNED
void onesweep_pipelined_kernel(
    typename KeyOf<KEY_BYTES>::type* keys_a, typename KeyOf<KEY_BYTES>::type* keys_b, int64_t n,
    int pass, KeyXform xf, const uint32_t* __restrict__ excl, uint32_t* all_status, uint32_t* ticket,
    const SortPlan* __restrict__ plan, int num_tiles, int groups, int chunk_shift,
    uint32_t spin_limit, int with_scanner) {
  using K = typename KeyOf<KEY_BYTES>::type;
  using Cfg = PipelinedTile<KEY_BYTES>;
  constexpr int kTile = Cfg::kTile;
  constexpr int kItems = Cfg::kItems;
  constexpr int kSorterWaves = Cfg::kSorterWaves;
  constexpr int kDigitWaves = kRadix / kWaveSize;
  constexpr int kDrawThread = kRadix;  // first lane of the first wave without digits
  static_assert(kItems % 2 == 0 && kTile <= 65536,
                "ranks and tile positions are packed two to a register");

  __shared__ __attribute__((aligned(16))) K s_keys[kTile];
  __shared__ __attribute__((aligned(16))) uint32_t s_counter[kSorterWaves * kRadix];
  // Handed between the sorting waves and the resolving wave, which runs up to a
  // tile behind: two copies each, by the parity of the block's tile count.
  __shared__ __attribute__((aligned(16))) uint32_t s_total[2][kRadix];
  __shared__ __attribute__((aligned(16))) uint32_t s_start[2][kRadix];
  __shared__ __attribute__((aligned(16))) uint32_t s_global_off[2][kRadix];
  __shared__ int s_next[2];
  __shared__ uint32_t s_scan[kDigitWaves];
  __shared__ uint32_t s_bar[4];

  if (plan->skip[pass]) return;
  const bool src_alt = plan->src_is_alt[pass] != 0;
  const int64_t region_words = (int64_t)num_tiles * kRadix;
  uint32_t* status = all_status + (src_alt ? region_words : 0);
  clear_next_status(all_status, region_words, plan, pass, 1024);
  const K* src_keys = src_alt ? keys_b : keys_a;
  K* dst_keys = src_alt ? keys_a : keys_b;
  const int shift = pass * 8;
  const uint32_t group = blockIdx.x % (uint32_t)groups;
  uint32_t* my_ticket = ticket + group * kTicketStride;
  // Float keys travel between the passes in their ordered form: the first pass
  // that runs converts them as it ranks them, the last one converts them back
  // as it writes them, and in between a digit is a shift and a mask (in_xf and
  // out_xf are the identity then).  Integer keys keep their bits throughout;
  // their order is one xor wherever a digit is taken.
  KeyXform in_xf = xf, out_xf = xf;
  if constexpr (FLOAT_KEYS) {
    if (plan->first_executed != (uint32_t)pass) in_xf = KeyXform{0, 0, 0};
    if (plan->last_executed != (uint32_t)pass) out_xf = KeyXform{0, 0, 0};
  }

  if (with_scanner && blockIdx.x < kScanBlocks) {
    // ---- a scanning block: the prefixes of 64 digits ----
    pipelined_scan<KEY_BYTES, FLOAT_KEYS>(src_keys, shift, in_xf, status, num_tiles,
                                          spin_limit, s_counter);
    return;
  }
  if (threadIdx.x == 0)
    s_next[0] = ticket_tile(atomicAdd(my_ticket, 1u), group, (uint32_t)groups, chunk_shift);
  if (threadIdx.x < 4) s_bar[threadIdx.x] = 0u;
  for (int i = threadIdx.x; i < kSorterWaves * kRadix / 4; i += Cfg::kBlock)
    reinterpret_cast<uint4*>(s_counter)[i] = make_uint4(0u, 0u, 0u, 0u);
  __syncthreads();
  int tile = s_next[0];
  __syncthreads();  // s_next[0] is written again by the first tile
  auto is_full = [&](int t) -> bool { return n - (int64_t)t * kTile >= kTile; };

  // Synchronisation.  The block-wide barrier (all sixteen waves) is used once
  // per tile, where the sixteenth wave hands over: it must never be waited for
  // inside the sorting waves' steps, or the publication of a tile's counts
  // would wait for the resolution of the tile before.  Among themselves the
  // sorting waves meet at counters in LDS: a wave arrives with one add by its
  // first lane (after its own LDS operations have completed) and, where it
  // needs the others, polls the counter.  it = tiles this block has finished.

  if (__builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize) == kSorterWaves) {
    // ---- the resolving wave ----
    const int lane = threadIdx.x & (kWaveSize - 1);
    // The status words of this pass as a buffer: 16-byte loads and stores with
    // the cache policy of an agent-scope atomic.
    const __amdgpu_buffer_rsrc_t status_rows = __builtin_amdgcn_make_buffer_rsrc(
        status, 0, num_tiles * kRadix * 4, 0x00027000);
    uint32_t it = 0;
    __syncthreads();  // the first tile's totals and run starts are there, or there is no tile
    while (tile < num_tiles) {
      const uint32_t par = it & 1u;
      bool resolved = false;
      if (!resolved && with_scanner && tile > 0) {
        // The scanning block turns this tile's counts into prefixes; its row is
        // polled until it has, but never without bound.
        const StatusVec my_count = reinterpret_cast<const StatusVec*>(s_total[par])[lane];
        for (uint32_t polls = 0; polls <= spin_limit && polls < kScannerPolls; ++polls) {
          __builtin_amdgcn_s_sleep(ILGPU_HIP_SORT_OWN_ROW_SLEEP);
          const StatusVec row = load_status_row(status_rows, tile, lane);
          bool all = true;
#pragma unroll
          for (int c = 0; c < kWalkDigits; ++c)
            all = all && row[c] != 0u && !status_is_aggregate(row[c]);
          if (__all(all)) {
            const StatusVec my_excl =
                reinterpret_cast<const StatusVec*>(excl + pass * kRadix)[lane];
            const StatusVec start = reinterpret_cast<const StatusVec*>(s_start[par])[lane];
            StatusVec offset;
#pragma unroll
            for (int c = 0; c < kWalkDigits; ++c)
              offset[c] = my_excl[c] + (status_value(row[c]) - my_count[c]) - start[c];
            reinterpret_cast<StatusVec*>(s_global_off[par])[lane] = offset;
            resolved = true;
            break;
          }
        }
      }
      if (!resolved)
        pipelined_walk<KEY_BYTES, FLOAT_KEYS>(src_keys, tile, shift, in_xf, status_rows,
                                              excl + pass * kRadix, s_total[par], s_start[par],
                                              s_global_off[par], lane, spin_limit);
      __syncthreads();  // this tile is resolved; the next one's totals are there, if there is one
      tile = s_next[par];
      ++it;
    }
    return;
  }

  // ---- the sorting waves ----
  uint32_t hot[kMaxHot];
#pragma unroll
  for (int h = 0; h < kMaxHot; ++h) hot[h] = plan->hot[pass][h];
  auto digit = [&](K k) -> uint32_t {  // of a ranked or staged key
    const K o = FLOAT_KEYS ? k : (K)(k ^ (K)xf.xor_mask);
    return (uint32_t)(o >> shift) & (kRadix - 1);
  };
  auto arrive = [&](int which, int lane) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    if (lane == 0)
      __hip_atomic_fetch_add(&s_bar[which], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  auto wait_for = [&](int which, uint32_t target, int lane) {
    if (lane == 0) {
      while (__hip_atomic_load(&s_bar[which], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) <
             target)
        __builtin_amdgcn_s_sleep(1);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  };
  // Tile-local positions from the run starts, the wave's counters cleared for
  // the next tile, the keys staged in digit order.
  auto stage = [&](auto full, K (&key)[kItems], uint32_t (&packed)[kItems / 2], int valid,
                   uint32_t* my_counters, int lane, int first_local) {
    constexpr bool kFull = decltype(full)::value;
    auto item_digit = [&](int j) -> uint32_t {
      return (kFull || first_local + j * kWaveSize < valid) ? digit(key[j])
                                                             : (uint32_t)(kRadix - 1);
    };
#pragma unroll
    for (int j = 0; j < kItems; j += 2) {
      const uint32_t p0 = my_counters[item_digit(j)] + (packed[j / 2] & 0xFFFFu);
      const uint32_t p1 = my_counters[item_digit(j + 1)] + (packed[j / 2] >> 16);
      packed[j / 2] = p0 | (p1 << 16);
      if (j % 8 == 6) __builtin_amdgcn_sched_barrier(0);
    }
    reinterpret_cast<uint4*>(my_counters)[lane] = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
    for (int j = 0; j < kItems; ++j)
      s_keys[j % 2 == 0 ? packed[j / 2] & 0xFFFFu : packed[j / 2] >> 16] = key[j];
  };
  auto write_out = [&](auto full, int valid, const uint32_t* global_off) {
    constexpr bool kFull = decltype(full)::value;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const int i = j * Cfg::kSorters + tid;
      if (kFull || i < valid) {
        const K k = s_keys[i];
        const uint32_t g = global_off[digit(k)] + (uint32_t)i;
        const K out = FLOAT_KEYS ? raw_bits(k, out_xf) : k;
        if (ILGPU_HIP_SORT_NT_STORE) __builtin_nontemporal_store(out, &dst_keys[g]);
        else dst_keys[g] = out;
      }
      if (j % ILGPU_HIP_SORT_WRITE_GROUP == ILGPU_HIP_SORT_WRITE_GROUP - 1)
        __builtin_amdgcn_sched_barrier(0);
    }
  };
  // What follows the ranking of a tile, up to the point where its keys are
  // staged in LDS: digit totals published, run starts, the hand-over with the
  // resolving wave, the write-out of the tile before, staging.
  uint32_t it = 0;       // tiles this block has finished
  bool pending = false;  // a staged tile waits to be written out
  auto after_ranking = [&](auto full, K (&key)[kItems], uint32_t (&packed)[kItems / 2],
                           int valid) {
    // The thread index is made opaque per tile: see sort_tile.
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & (kWaveSize - 1);
    const int wave = tid / kWaveSize;
    const int first_local = wave * Cfg::kSubTileKeys + lane;
    uint32_t* my_counters = s_counter + wave * kRadix;
    const uint32_t par = it & 1u;
    arrive(0, lane);  // ranked
    uint32_t drawn = 0;
    if (tid < kRadix) {
      // One thread per digit (waves 0..3): totals over the sub-tiles, published
      // at once; then the tile-local start of every (sub-tile, digit) run.
      wait_for(0, (it + 1u) * kSorterWaves, lane);
      uint32_t count = 0;
#pragma unroll
      for (int s = 0; s < kSorterWaves; ++s) count += s_counter[s * kRadix + tid];
      __hip_atomic_store(&status[(int64_t)tile * kRadix + tid],
                         tile == 0 ? status_prefix(count) : status_aggregate(count),
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_total[par][tid] = count;
      uint32_t inc = count;
#pragma unroll
      for (int s = 1; s < kWaveSize; s <<= 1) {
        const uint32_t o = shfl_up(inc, s);
        if (lane >= s) inc += o;
      }
      if (lane == kWaveSize - 1) s_scan[wave] = inc;
      arrive(1, lane);
      wait_for(1, (it + 1u) * kDigitWaves, lane);
      uint32_t run = inc - count;
      for (int w = 0; w < wave; ++w) run += s_scan[w];
      s_start[par][tid] = run;
#pragma unroll
      for (int s = 0; s < kSorterWaves; ++s) {
        const uint32_t c = s_counter[s * kRadix + tid];
        s_counter[s * kRadix + tid] = run;
        run += c;
      }
    } else if (tid == kDrawThread) {
      // The block's next tile is drawn now: its keys are loaded as soon as this
      // tile is staged, and its counts are published right after their ranking,
      // whatever the look-back of this tile does.
      drawn = atomicAdd(my_ticket, 1u);
    }
    __syncthreads();  // run starts and totals are there; the tile before is resolved
    if (pending) write_out(std::true_type{}, kTile, s_global_off[par ^ 1u]);
    if (tid == kDrawThread) s_next[par] = ticket_tile(drawn, group, (uint32_t)groups, chunk_shift);
    arrive(2, lane);  // the staged tile has been read
    wait_for(2, (it + 1u) * kSorterWaves, lane);
    stage(full, key, packed, valid, my_counters, lane, first_local);
    pending = true;
    const int next_tile = s_next[par];
    ++it;
    return next_tile;
  };

  auto full_tiles = [&](auto with_hot) {
    constexpr bool kHot = decltype(with_hot)::value;
    if (!(tile < num_tiles && is_full(tile))) return;
    K key[kItems];
    uint32_t packed[kItems / 2];
    {
      int tid = threadIdx.x;
      asm volatile("" : "+v"(tid));
      const int lane = tid & (kWaveSize - 1), wave = tid / kWaveSize;
      pipelined_rank<KEY_BYTES, true, kHot, FLOAT_KEYS>(
          key, packed, src_keys, (int64_t)tile * kTile, kTile, shift, in_xf, s_counter + wave * kRadix,
          lane, wave * Cfg::kSubTileKeys + lane, hot);
    }
    bool ranked = true;
    while (ranked) {
      const int next_tile = after_ranking(std::true_type{}, key, packed, kTile);
      ranked = next_tile < num_tiles && is_full(next_tile);
      if (ranked) {
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lane = tid & (kWaveSize - 1), wave = tid / kWaveSize;
        pipelined_rank<KEY_BYTES, true, kHot, FLOAT_KEYS>(
            key, packed, src_keys, (int64_t)next_tile * kTile, kTile, shift, in_xf,
            s_counter + wave * kRadix, lane, wave * Cfg::kSubTileKeys + lane, hot);
      }
      tile = next_tile;
    }
  };
  if (hot[0] == kNoHotDigit) full_tiles(std::false_type{});
  else full_tiles(std::true_type{});
  // Here the block's next tile, if any, is the one at the end of the input; it
  // is the last of its group and so of this block.
  int last_valid = kTile;
  if (tile < num_tiles) {
    const int tid = threadIdx.x;
    const int lane = tid & (kWaveSize - 1);
    const int wave = tid / kWaveSize;
    last_valid = (int)(n - (int64_t)tile * kTile);
    K key[kItems];
    uint32_t packed[kItems / 2];
    pipelined_rank<KEY_BYTES, false, true, FLOAT_KEYS>(
        key, packed, src_keys, (int64_t)tile * kTile, last_valid, shift, in_xf,
        s_counter + wave * kRadix, lane, wave * Cfg::kSubTileKeys + lane, hot);
    after_ranking(std::false_type{}, key, packed, last_valid);
  }
  __syncthreads();  // the last tile is resolved
  if (pending) {
    if (last_valid == kTile) write_out(std::true_type{}, kTile, s_global_off[(it & 1u) ^ 1u]);
    else write_out(std::false_type{}, last_valid, s_global_off[(it & 1u) ^ 1u]);
  }
}

// ---- inputs of one tile ---------------------------------------------------------
// A sort of at most one 512-thread tile runs as one block and one launch: the
// keys (and values) stay in registers, every pass ranks them like a pass above,
// moves them through LDS into digit order and takes them back in memory order
// (lane l of wave w holds positions w*64*I + j*64 + l again; small_sort_block says how many threads), and the last pass
// is followed by one coalesced write.  No histogram, plan, tickets, look-back
// or temp memory.  ITEMS keys per thread: every row costs its rank, its
// staging and its share of five barriers per pass whether it holds keys or
// not, so short inputs take an instantiation with few rows (4, 12 or 24:
// 32 to 2048 u32 keys 8 to 9 us instead of 24 to 27, up to 6144 keys 13
// instead of 31).
//
// A chain of dependent steps bounds it, the passes above all (some 1.4 us each with four rows), so as few
// of them run as order the keys.  A digit that all keys share takes none (the block ORs what
// differs between integer keys; floats vary in every digit, and two digits are not worth it).  And
// a tile has so few keys that of 8-byte keys the three topmost digits that differ (up to 2048
// integers) or the four topmost tell all but a few pairs apart: only those run, and where
// neighbours are then in the wrong order every key looks for the ones of its prefix that go the
// other way round.  Which pays while few different keys share a prefix, so 512 keys from all over the input
// are asked: each takes its prefix's slot in LDS and looks at the one before, and those that meet another key of
// their prefix are counted.  (Copies of a key need no order.)  Where a prefix has more than kSmallSortReach keys all the
// same, and they are in the wrong order, all the digits follow.
// (Kernel, us, every digit / this: 2000 int64 uniform 13.6 / 7.4, with u32 index values 14.9 / 8.3, below 10^6
// 13.2 / 6.5, time stamps within 17 s 13.7 / 11.7, normal doubles 14.6 / 10.6; 9000 uniform 32.3 / 21.1, 18 000 u32 below
// 10^6 31.2 / 22.1.  A prefix of 30 of 2000 keys 13.6 / 13.3, of 9000 32.3 / 30.2; of a tenth, all digits, 13.5 / 14.3 and
// 32.2 / 33.6, signed numbers of 40 bits 13.3 / 13.8 and 31.3 / 32.5: the question.  With 8 keys of a row and wave asked, and
// runs of up to 24 taken: a tenth 36.7 and 116, 40 bits 14.8 and 165, where many runs of some 20 were looked through,
// or the prefix's passes were for nothing.)
// (Two digits and the same of 4-byte keys: a key in four has a neighbour to look at, 18 000 keys 68 us
// instead of 34.6.)
constexpr int kSmallSortReach = 256;
constexpr int kSmallSortAlike = 12;  // of a wave's keys asked
constexpr int kAskedSlotsLog2 = 11;
// `clashes`: keys asked that meet another of their prefix.  Half a key beside every key is too many: all
// waves would look at neighbours (7000 keys in 20 bursts, 1.4 others per key, 35.2 us all digits, 40.7 by prefix; 2000 in
// 20 bursts, 0.4 per key, 17.5 and 15.3).
__device__ __forceinline__ bool small_sort_few_meet(int clashes, int n) {
  return (int64_t)clashes * (n > kSortBlock ? n : kSortBlock) <= kSortBlock * kSortBlock / 4;
}
// `pairs`: of the keys asked that differ from another of their prefix.  Of a run of L keys some k = 512 L / n are asked, which
// makes k^2 / 2 and fewer of them; the runs that cost as much to look through as the passes that are saved have some
// 35 keys of 2000, 80 of 9000.
__device__ __forceinline__ bool small_sort_spreads(int pairs, int n) {
  const int64_t m = n > kSortBlock ? n : kSortBlock;
  const int64_t run = kSortBlock * (30 + m / 256);
  return 2 * pairs * m * m <= run * run;
}

constexpr int kSmallSortItemsA = 4, kSmallSortItemsB = 12, kSmallSortItemsC = 24;
// Threads of the block for tiles of `rows` keys per 512 threads: twice that many with half of the rows, which wait for the
// LDS together, where there are more rows than four; of 8-byte keys, which sort few digits and look at their neighbours, the
// floating-point ones, which sort all digits; of shorter keys, which have one or two digits, only the longest tiles.  (Sorts with a copy in front, us, 512 / 1024 threads: u32 keys 4000 12.6 / 11.8,
// 9000 20.1 / 18.1, 18 000 30.1 / 24.8, below 10^6 24.3 / 20.5; normal floats 6000 19.0 / 16.4, 18 000 49.2 / 36.5; normal doubles 9000
// 32.4 / 30.2; but u64 keys below 10^6 9000 17.7 / 18.2, Zipf 17.2 / 18.1, pairs of 5000 u64 21.6 / 23.7, u16 keys 6000 11.4 / 12.9, 18 000 16.8 / 14.3.
// Pairs of integers whose rows do not halve into an even number keep 512: 7000 u32 with u64 15.9 / 17.1 in the kernel.)
constexpr int small_sort_block(int key_bytes, int value_bytes, bool floats, int rows) {
  const bool wide = key_bytes == 8 ? floats && value_bytes == 0 && rows > kSmallSortItemsA
                                   : rows > (key_bytes == 4 ? kSmallSortItemsA : kSmallSortItemsC) &&
                                         (value_bytes == 0 || rows % 4 == 0 || floats);
  return wide ? 2 * kSortBlock : kSortBlock;
}
constexpr int small_sort_items(int block, int rows) { return block == kSortBlock ? rows : (rows / 2 + 1) / 2 * 2; }
// (One block runs: registers and LDS are not shared with others.)
template <int KEY_BYTES, int VALUE_BYTES, bool FLOAT_KEYS, int BLOCK, int ITEMS>
__global__ __launch_bounds__(BLOCK, BLOCK == kSortBlock && KEY_BYTES == 8 ? 2 : ILGPU_HIP_SORT_WAVES_PER_EU)
void small_sort_kernel(typename KeyOf<KEY_BYTES>::type* keys,
                       typename ValueOf<VALUE_BYTES>::type* vals, int n, KeyXform xf,
                       int values_from_index) {
  using K = typename KeyOf<KEY_BYTES>::type;
  using Val = typename ValueOf<VALUE_BYTES>::type;
  using TileCfg = SortTile<KEY_BYTES, VALUE_BYTES, BLOCK>;
  constexpr int kItems = ITEMS;
  constexpr int kSubTiles = TileCfg::kSubTiles;
  constexpr int kSubTileKeys = kSubLanes * kItems;
  constexpr bool kPairs = VALUE_BYTES > 0;
  static_assert(kItems % 2 == 0 && kItems <= TileCfg::kItems, "ranks are packed in pairs");
  // Counters, then the keys, then the values of the tile share these bytes.
  constexpr int kEntryBytes = KEY_BYTES > VALUE_BYTES ? KEY_BYTES : VALUE_BYTES;
  constexpr int kStageBytes = BLOCK * kItems * kEntryBytes > TileCfg::kCounterBytes
                                  ? BLOCK * kItems * kEntryBytes
                                  : TileCfg::kCounterBytes;

  __shared__ __attribute__((aligned(16))) unsigned char s_stage[kStageBytes];
  __shared__ uint32_t s_scan[kRadix / kWaveSize];
  __shared__ uint64_t s_diff[kSubTiles];
  __shared__ uint32_t s_inverted, s_far;
  __shared__ int s_clashes[kSubTiles], s_pairs[kSubTiles];
  __shared__ uint64_t s_asked[KEY_BYTES == 8 ? kSortBlock : 1];
  __shared__ uint16_t s_to[KEY_BYTES == 8 ? BLOCK * kItems : 1];  // where a staged key belongs
  uint32_t* s_counter = reinterpret_cast<uint32_t*>(s_stage);
  K* s_keys = reinterpret_cast<K*>(s_stage);
  Val* s_vals = reinterpret_cast<Val*>(s_stage);

  const int tid = threadIdx.x;
  const int lane = tid & (kWaveSize - 1);
  const int wave = tid / kWaveSize;
  const int first_local = wave * kSubTileKeys + lane;
  uint32_t* my_counters = s_counter + wave * kRadix;

  K key[kItems], asked = 0;
  Val val[kPairs ? kItems : 1];
  uint32_t* s_words = reinterpret_cast<uint32_t*>(s_stage);  // two tables of kAskedSlotsLog2
  if constexpr (KEY_BYTES == 8) {
    static_assert(8 << kAskedSlotsLog2 <= kStageBytes && (8 << kAskedSlotsLog2) % (16 * BLOCK) == 0, "");
    // (The first kSortBlock threads ask.)
    if (tid < kSortBlock) asked = keys[(uint32_t)tid * (uint32_t)n / kSortBlock];
#pragma unroll
    for (int i = 0; i < (8 << kAskedSlotsLog2) / (16 * BLOCK); ++i)
      reinterpret_cast<uint4*>(s_stage)[i * BLOCK + tid] = make_uint4(0u, 0u, 0u, 0u);
  }
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const int local = first_local + j * kSubLanes;
    key[j] = 0;
    if (local < n) {
      key[j] = keys[local];
      if constexpr (FLOAT_KEYS) key[j] = ordered_bits(key[j], xf);
      if constexpr (kPairs) {
        if (values_from_index) {
          val[j] = index_value<VALUE_BYTES>(local, values_from_index);
        } else {
          val[j] = vals[local];
        }
      }
    }
  }

  auto ordered = [&](K k) -> K {  // of a key as it is held
    if constexpr (FLOAT_KEYS) return k;
    else return (K)(k ^ (K)xf.xor_mask);
  };
  // The bits in which keys differ, and the prefix that is sorted first.
  // (4-byte keys with fewer rows: half a microsecond for the question, which a digit less gives back
  // where there is one: 2000 uniform u32 keys 6.8 -> 7.4 us, below 10^6 6.8 -> 6.0.)
  constexpr bool kAsks = KEY_BYTES == 8 || (KEY_BYTES == 4 && !FLOAT_KEYS && BLOCK * kItems > kSortBlock * kSmallSortItemsC);
  constexpr int kPrefixDigits = BLOCK * kItems <= kSortBlock * kSmallSortItemsA && !FLOAT_KEYS ? 3 : 4;
  uint64_t diff = ~0ull;
  int top_bits = 8 * KEY_BYTES, prefix_shift = 0;
  bool by_prefix = false;
  if constexpr (kAsks) {
    const K first = FLOAT_KEYS ? ordered_bits(keys[0], xf) : keys[0];
    K mine = 0;
#pragma unroll
    for (int j = 0; j < kItems; ++j)
      if (first_local + j * kSubLanes < n) mine |= (K)(key[j] ^ first);
    diff = wave_or((uint32_t)mine);
    if constexpr (KEY_BYTES == 8) diff |= (uint64_t)wave_or((uint32_t)((uint64_t)mine >> 32)) << 32;
    if (lane == 0) s_diff[wave] = diff;
    if (tid == 0) s_inverted = s_far = 0u;
    if constexpr (KEY_BYTES == 8) {
      if constexpr (FLOAT_KEYS) asked = ordered_bits(asked, xf);
      else asked = ordered(asked);
      if (tid < kSortBlock) s_asked[tid] = asked;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kSubTiles; ++w) diff |= s_diff[w];
    diff = readfirstlane_key(diff);
    top_bits = diff != 0 ? 64 - __builtin_clzll(diff) : 0;
  }
  if constexpr (KEY_BYTES == 8) {
    int digits = 0;  // that differ
#pragma unroll
    for (int p = 0; p < KEY_BYTES; ++p) digits += (diff >> (8 * p) & 0xFFull) != 0 ? 1 : 0;
    prefix_shift = top_bits > 8 * kPrefixDigits ? top_bits - 8 * kPrefixDigits : 0;
    by_prefix = digits > kPrefixDigits;
    if (by_prefix) {
      const uint64_t prefix = (uint64_t)asked >> prefix_shift;
      const uint32_t slot = ((uint32_t)prefix * 0x9E3779B1u) >> (32 - kAskedSlotsLog2);
      // (A wave that sees many of one prefix asks no more: all would wait for one word.)
      const int alike = __popcll(__ballot(prefix == readfirstlane_key(prefix) &&
                                          (uint64_t)asked != readfirstlane_key((uint64_t)asked)));
      bool clash = false;
      if (tid < kSortBlock && alike <= kSmallSortAlike) {
        const uint32_t before = __hip_atomic_exchange(&s_words[slot], (uint32_t)tid + 1u, __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_WORKGROUP);
        if (before != 0u) {
          const uint64_t other = s_asked[before - 1u];
          clash = other >> prefix_shift == prefix && other != (uint64_t)asked;
        }
      }
      int clashes = __popcll(__ballot(clash));
      if (lane == 0) s_clashes[wave] = tid >= kSortBlock ? 0 : (alike <= kSmallSortAlike ? clashes : 1 << 20);
      __syncthreads();
      clashes = 0;
#pragma unroll
      for (int w = 0; w < kSubTiles; ++w) clashes += s_clashes[w];
      clashes = __builtin_amdgcn_readfirstlane(clashes);
      by_prefix = small_sort_few_meet(clashes, n);
      if (by_prefix && clashes != 0) {  // how many of them share a prefix
        int pairs = 0;
        if (clash)
          pairs = (int)__hip_atomic_fetch_add(&s_words[(1 << kAskedSlotsLog2) + slot], 1u, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_WORKGROUP);
        pairs = wave_sum(pairs);
        if (lane == 0) s_pairs[wave] = pairs;
        __syncthreads();
        pairs = 0;
#pragma unroll
        for (int w = 0; w < kSubTiles; ++w) pairs += s_pairs[w];
        by_prefix = small_sort_spreads(__builtin_amdgcn_readfirstlane(pairs), n);
      }
    }
  }
  int shift = by_prefix ? prefix_shift : 0;
#pragma unroll 1
  for (; shift < top_bits; shift += 8) {
    const bool last_of_prefix = by_prefix && shift + 8 >= top_bits;
    if (!by_prefix && (diff >> shift & 0xFFull) == 0) continue;
    // Positions past the end take digit 255 and come last in memory order, so
    // they stay behind every key through every pass.  (The length is made opaque: held from one pass to the
    // next the rows' masks spill.)
    int length = n;
    asm volatile("" : "+s"(length));
    auto item_digit = [&](int j) -> uint32_t {
      if (first_local + j * kSubLanes >= length) return (uint32_t)(kRadix - 1);
      return (uint32_t)(ordered(key[j]) >> shift) & (kRadix - 1);
    };
    __syncthreads();  // the stage of the previous pass has been read
    // (A wave clears its own counters, and needs no barrier for that.)
    static_assert(kRadix == 4 * kSubLanes, "four counters per lane");
    reinterpret_cast<uint4*>(my_counters)[lane] = make_uint4(0u, 0u, 0u, 0u);
    __builtin_amdgcn_wave_barrier();

    uint32_t packed[kItems / 2];  // rank in the sub-tile, then position in the tile
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const uint32_t d = item_digit(j);
      // a row that is all one digit: lane 0 adds for the row (see sort_tile)
      const uint32_t row_digit = (uint32_t)__builtin_amdgcn_readfirstlane((int)d);
      const bool whole_row = __ballot(d == row_digit) == ~0ull;
      uint32_t rank = 0;
      if (!whole_row || lane == 0)
        rank = __hip_atomic_fetch_add(my_counters + d, whole_row ? (uint32_t)kSubLanes : 1u,
                                      __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (whole_row) rank = (uint32_t)__builtin_amdgcn_readfirstlane((int)rank) + (uint32_t)lane;
      if (j % 2 == 0) packed[j / 2] = rank;
      else packed[j / 2] |= rank << 16;
    }
    __syncthreads();

    // One thread per digit: totals over the sub-tiles, exclusive scan over the
    // digits, then the tile position of the first key of every (sub-tile, digit).
    uint32_t count = 0, inc = 0;
    if (tid < kRadix) {
#pragma unroll
      for (int s = 0; s < kSubTiles; ++s) count += s_counter[s * kRadix + tid];
      inc = count;
#pragma unroll
      for (int s = 1; s < kWaveSize; s <<= 1) {
        const uint32_t o = shfl_up(inc, s);
        if (lane >= s) inc += o;
      }
      if (lane == kWaveSize - 1) s_scan[wave] = inc;
    }
    __syncthreads();
    if (tid < kRadix) {
      uint32_t run = inc - count;
      for (int w = 0; w < wave; ++w) run += s_scan[w];
#pragma unroll
      for (int s = 0; s < kSubTiles; ++s) {
        const uint32_t t = s_counter[s * kRadix + tid];
        s_counter[s * kRadix + tid] = run;
        run += t;
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kItems; j += 2) {
      const uint32_t p0 = my_counters[item_digit(j)] + (packed[j / 2] & 0xFFFFu);
      const uint32_t p1 = my_counters[item_digit(j + 1)] + (packed[j / 2] >> 16);
      packed[j / 2] = p0 | (p1 << 16);
    }
    __syncthreads();  // the run starts have been read; the same bytes stage the keys
#pragma unroll
    for (int j = 0; j < kItems; ++j)
      s_keys[j % 2 == 0 ? packed[j / 2] & 0xFFFFu : packed[j / 2] >> 16] = key[j];
    __syncthreads();
    if constexpr (KEY_BYTES == 8) {
      if (last_of_prefix) {
        bool inverted = false;
#pragma unroll
        for (int j = 0; j < kItems; ++j) {
          const int at = j * BLOCK + tid;
          if (at + 1 < length) inverted = inverted || ordered(s_keys[at]) > ordered(s_keys[at + 1]);
        }
        if (inverted) s_inverted = 1u;
        __syncthreads();
        if (s_inverted != 0u) {
          // Keys of the same prefix are next to each other, equal keys in their order: a key moves
          // by the smaller ones behind it and the larger ones in front of it.
          for (int at = tid; at < length; at += BLOCK) {
            const K o = ordered(s_keys[at]);
            const K prefix = (K)(o >> prefix_shift);
            int to = at;
            auto look = [&](int step) {
              const int next = at + step;
              if (next < 0 || next >= length || (K)(ordered(s_keys[next]) >> prefix_shift) != prefix) return;
              for (int q = next;; q += 4 * step) {  // four keys at a time
                K other[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  const int from = q + e * step;
                  other[e] = ordered(s_keys[from < 0 ? 0 : (from < length ? from : length - 1)]);
                }
                bool same = true;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  const int from = q + e * step;
                  same = same && from >= 0 && from < length && (K)(other[e] >> prefix_shift) == prefix;
                  if (same) to += step > 0 ? (other[e] < o ? 1 : 0) : (other[e] > o ? -1 : 0);
                }
                if (!same) break;
                if ((q - at) * step > kSmallSortReach) {
                  s_far = 1u;
                  break;
                }
              }
            };
            look(1);
            look(-1);
            s_to[at] = (uint16_t)to;
          }
          __syncthreads();
          if (s_far != 0u) {  // from the order before this pass, which the registers still hold
            by_prefix = false;
            shift = -8;
            continue;
          }
#pragma unroll
          for (int j = 0; j < kItems; j += 2) {
            // (Positions behind the keys keep their places.)
            const uint32_t p0 = packed[j / 2] & 0xFFFFu, p1 = packed[j / 2] >> 16;
            packed[j / 2] = ((int)p0 < length ? s_to[p0] : p0) | ((int)p1 < length ? s_to[p1] : p1) << 16;
          }
#pragma unroll
          for (int j = 0; j < kItems; ++j)
            s_keys[j % 2 == 0 ? packed[j / 2] & 0xFFFFu : packed[j / 2] >> 16] = key[j];
          __syncthreads();
        }
      }
    }
#pragma unroll
    for (int j = 0; j < kItems; ++j) key[j] = s_keys[first_local + j * kSubLanes];
    if constexpr (kPairs) {
      __syncthreads();
#pragma unroll
      for (int j = 0; j < kItems; ++j)
        s_vals[j % 2 == 0 ? packed[j / 2] & 0xFFFFu : packed[j / 2] >> 16] = val[j];
      __syncthreads();
#pragma unroll
      for (int j = 0; j < kItems; ++j) val[j] = s_vals[first_local + j * kSubLanes];
    }
  }

#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const int local = first_local + j * kSubLanes;
    if (local < n) {
      if constexpr (FLOAT_KEYS) keys[local] = raw_bits(key[j], xf);
      else keys[local] = key[j];
      if constexpr (kPairs) vals[local] = val[j];
    }
  }
}

// ---- finish ----------------------------------------------------------------
template <int KEY_BYTES, int VALUE_BYTES>
__device__ __forceinline__ void finish(
    typename KeyOf<KEY_BYTES>::type* keys_a,
    const typename KeyOf<KEY_BYTES>::type* keys_b,
    typename ValueOf<VALUE_BYTES>::type* vals_a,
    const typename ValueOf<VALUE_BYTES>::type* vals_b, int64_t n,
    const SortPlan* __restrict__ plan, int values_from_index) {
  const bool copy_back = plan->final_in_alt != 0;
  const bool fill_index =
      VALUE_BYTES > 0 && values_from_index && plan->executed == 0;
  if (!copy_back && !fill_index) return;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += stride) {
    if (copy_back) {
      keys_a[i] = keys_b[i];
      if constexpr (VALUE_BYTES > 0) vals_a[i] = vals_b[i];
    } else {
      if constexpr (VALUE_BYTES > 0) vals_a[i] = index_value<VALUE_BYTES>(i, values_from_index);
    }
  }
}

template <int KEY_BYTES, int VALUE_BYTES>
__global__ __launch_bounds__(256) void finish_kernel(
    typename KeyOf<KEY_BYTES>::type* keys_a,
    const typename KeyOf<KEY_BYTES>::type* keys_b,
    typename ValueOf<VALUE_BYTES>::type* vals_a,
    const typename ValueOf<VALUE_BYTES>::type* vals_b, int64_t n,
    const SortPlan* __restrict__ plan, int values_from_index) {
  finish<KEY_BYTES, VALUE_BYTES>(keys_a, keys_b, vals_a, vals_b, n, plan, values_from_index);
}

// ---- ties of the upper half --------------------------------------------------
// After the passes over the upper half (plan->ties_left): keys whose upper halves
// are the same stand next to each other in their original order.  Every run of such
// keys is put into the order of the whole key, equal keys left in their order.
// Nobody else writes the run, and whoever looks at its neighbours compares upper
// halves, which do not change.
//
// A read of the keys, then: a lane takes kTieRows keys, a row of a wave 64
// neighbouring ones, and the runs of all rows are ordered together, since each
// costs a chain of two or three memory round trips.  Runs of two or three keys, which nearly
// all of them are, are ordered by the lane that sees the first one, longer ones by 8 to
// 64 lanes with a key per lane, or a wave with two.  Runs of 128 keys and more wait until
// the block's waves have seen all of their keys, and are then ordered by the block.
constexpr int kTieRows = 8;
constexpr int kTieChunk = kTieRows * kWaveSize;
constexpr int kTieBlock = 256;
constexpr int kTieWaves = kTieBlock / kWaveSize;
constexpr int kTieItems = 8;        // keys per thread that are ordered in LDS at a time
constexpr int kTieMerges = 4;       // memory reads of a thread in flight where runs are merged
// Runs of 128 keys and more that can start in one chunk.
constexpr int kTieLongsPerChunk = kTieChunk / 128;

// Runs of fewer than `width` keys, one by each `width` lanes (start: of the lane's run, if
// there is one for it; width: 8 to 64).  A key's place is the number of keys that go in
// front of it.
template <int VALUE_BYTES, typename Val>
__device__ __forceinline__ void order_runs(uint64_t* keys, Val* vals, uint32_t start, bool any, uint32_t n,
                                           const KeyXform& xf, int lane, int width) {
  const int first = lane & ~(width - 1);
  const uint32_t at = start + (uint32_t)(lane - first);
  const bool have = any && at < n;
  uint64_t k = 0;
  Val v{};
  if (have) {
    k = keys[at];
    if constexpr (VALUE_BYTES > 0) v = vals[at];
  }
  const bool same = have && (uint32_t)(k >> 32) == (uint32_t)__shfl((int)(uint32_t)(k >> 32), first);
  const int end = first + __builtin_ctzll(~(__ballot(same) >> first));
  const uint32_t o = (uint32_t)ordered_bits(k, xf);  // the upper halves agree
  int rank = first;
  if (width == kWaveSize) {  // one run: `end` is the same in every lane
    const int len = __builtin_amdgcn_readfirstlane(end);
    for (int j = 0; j < len; ++j) {
      const uint32_t q = (uint32_t)__builtin_amdgcn_readlane((int)o, j);
      if (q < o || (q == o && j < lane)) ++rank;
    }
  } else {
#pragma unroll 4
    for (int j = 0; j < width; ++j) {
      const int other = first + j;
      const uint32_t q = (uint32_t)__shfl((int)o, other);
      if (other < end && (q < o || (q == o && other < lane))) ++rank;
    }
  }
  if (lane < end && rank != lane) {
    keys[start + (uint32_t)(rank - first)] = k;
    if constexpr (VALUE_BYTES > 0) vals[start + (uint32_t)(rank - first)] = v;
  }
}

// A run of 64 to 127 keys, by a wave with two keys per lane.
template <int VALUE_BYTES, typename Val>
__device__ __forceinline__ void order_two_rows(uint64_t* keys, Val* vals, uint32_t start, uint32_t n,
                                               const KeyXform& xf, int lane) {
  const uint32_t first = start + lane;
  const uint32_t second = min(first + kWaveSize, n - 1);
  const uint64_t k0 = keys[first], k1 = keys[second];
  Val v0{}, v1{};
  if constexpr (VALUE_BYTES > 0) {
    v0 = vals[first];
    v1 = vals[second];
  }
  const bool same = first + kWaveSize < n &&
                    (uint32_t)(k1 >> 32) == (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(k0 >> 32));
  const int more = __builtin_ctzll(~__ballot(same));  // not all of them
  const uint32_t o0 = (uint32_t)ordered_bits(k0, xf), o1 = (uint32_t)ordered_bits(k1, xf);
  int rank0 = 0, rank1 = 0;
  for (int j = 0; j < kWaveSize; ++j) {
    const uint32_t q = (uint32_t)__builtin_amdgcn_readlane((int)o0, j);
    if (q < o0 || (q == o0 && j < lane)) ++rank0;
    if (q <= o1) ++rank1;
  }
  for (int j = 0; j < more; ++j) {
    const uint32_t q = (uint32_t)__builtin_amdgcn_readlane((int)o1, j);
    if (q < o0) ++rank0;
    if (q < o1 || (q == o1 && j < lane)) ++rank1;
  }
  keys[start + rank0] = k0;
  if constexpr (VALUE_BYTES > 0) vals[start + rank0] = v0;
  if (lane < more) {
    keys[start + rank1] = k1;
    if constexpr (VALUE_BYTES > 0) vals[start + rank1] = v1;
  }
}

// `count` elements from one buffer to the other, kTieMerges of a thread in flight.
template <typename E>
__device__ __forceinline__ void copy_rows(E* to, const E* from, uint32_t count, int t) {
  for (uint32_t row = t; row < count; row += kTieMerges * kTieBlock) {
    E e[kTieMerges];
#pragma unroll
    for (int u = 0; u < kTieMerges; ++u) e[u] = from[min(row + u * kTieBlock, count - 1)];
#pragma unroll
    for (int u = 0; u < kTieMerges; ++u)
      if (row + u * kTieBlock < count) to[row + u * kTieBlock] = e[u];
  }
}

// LDS in which a block orders a piece of a run.
struct TiePiece {
  static constexpr int kKeys = kTieBlock * kTieItems;
  uint32_t o[kKeys];   // ordered lower halves
  uint16_t from[kKeys];  // places they came from
  uint32_t counts[kTieWaves][kRadix];
  uint32_t totals[kTieWaves];
};
static_assert(kRadix == kTieBlock, "a thread scans the counts of one digit");

// Exclusive sums of the digit counts of all waves, digits first, in their place.
__device__ __forceinline__ void scan_counts(TiePiece& p, uint32_t* s_totals, int t) {
  const int lane = t & (kWaveSize - 1);
  uint32_t total = 0;
#pragma unroll
  for (int w = 0; w < kTieWaves; ++w) total += p.counts[w][t];
  uint32_t sum = total;
#pragma unroll
  for (int step = 1; step < kWaveSize; step <<= 1) {
    const uint32_t other = shfl_up(sum, step);
    if (lane >= step) sum += other;
  }
  if (lane == kWaveSize - 1) s_totals[t / kWaveSize] = sum;
  __syncthreads();
  uint32_t off = sum - total;
  for (int w = 0; w < t / kWaveSize; ++w) off += s_totals[w];
#pragma unroll
  for (int w = 0; w < kTieWaves; ++w) {
    const uint32_t c = p.counts[w][t];
    p.counts[w][t] = off;
    off += c;
  }
}

// Puts a piece, whose lower halves are in p.o, into their order, stable: four digits, each as a
// pass of the sort ranks it (returning LDS adds on counters of the wave, which serve
// lanes in lane order).  A wave holds kTieItems rows of 64 neighbouring keys.
__device__ __forceinline__ void sort_piece(TiePiece& p, uint32_t* s_totals, int t) {
  const int lane = t & (kWaveSize - 1), wave = t / kWaveSize;
  const int base = wave * (kTieItems * kWaveSize) + lane;
  uint32_t* counts = p.counts[wave];
  for (int shift = 0; shift < 32; shift += 8) {
    uint32_t o[kTieItems], from[kTieItems];  // from: place it came from, and above it the rank
#pragma unroll
    for (int q = 0; q < kRadix / kWaveSize; ++q) counts[q * kWaveSize + lane] = 0u;
#pragma unroll
    for (int u = 0; u < kTieItems; ++u) {
      o[u] = p.o[base + u * kWaveSize];
      from[u] = shift == 0 ? (uint32_t)(base + u * kWaveSize) : p.from[base + u * kWaveSize];
    }
    // (The counters are the wave's own, and its LDS instructions run in order.)
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int u = 0; u < kTieItems; ++u) from[u] |= atomicAdd(&counts[(o[u] >> shift) & (kRadix - 1)], 1u) << 16;
    __syncthreads();
    scan_counts(p, s_totals, t);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kTieItems; ++u) {
      const uint32_t at = counts[(o[u] >> shift) & (kRadix - 1)] + (from[u] >> 16);
      p.o[at] = o[u];
      p.from[at] = (uint16_t)from[u];
    }
    __syncthreads();
  }
}

// (Whole sorts of 2^21 u64 keys, us: uniform 115; one cluster of 1000, 2000 and 3000 keys 127,
// 125 and 153, where a wave that merged it in memory, with an agent-scope fence per
// level, took 305, 549 and 811; 1 % of the keys in runs of 32 with neighbouring upper
// halves 160 / 314, of 2^27 keys 2687 / 6656.  By a bitonic sort of 1024 keys at a time
// 3000 keys took 206, by merges alone in LDS 200.)

// A run of 128 keys or more, by a block.  Pieces of kTieItems keys per thread are
// ordered in LDS, by their lower halves; a piece that is in order (many copies of
// one key) is left alone.  Then pieces are merged through memory if they have to
// be, every key finding its place in the other piece by bisection, first among every
// 2^k-th key, which LDS holds.  The other buffer's same range is scratch.
// (Not inlined: its registers made the loop that every input goes through spill,
// 29.1 us instead of 26.4 at 2^24 uniform keys.)
template <typename Val, int VALUE_BYTES>
__device__ __attribute__((noinline)) void order_long_run(
    uint64_t* keys, uint64_t* other_keys, Val* vals, Val* other_vals, uint32_t start, uint32_t n,
    uint64_t xor_mask, uint64_t reference_term, uint64_t total_term,
    __attribute__((address_space(3))) TiePiece* lds_piece) {
  const KeyXform xf{xor_mask, reference_term, total_term};
  TiePiece& p = *(TiePiece*)lds_piece;
  uint32_t* s_totals = p.totals;
  const int t = threadIdx.x;
  constexpr int kPiece = TiePiece::kKeys;
  uint64_t* src = keys + start;
  uint64_t* dst = other_keys + start;
  Val* src_vals = VALUE_BYTES > 0 ? vals + start : nullptr;
  Val* dst_vals = VALUE_BYTES > 0 ? other_vals + start : nullptr;
  const uint64_t first_key = src[0];
  const uint64_t upper_ordered = ordered_bits(first_key, xf) & ~0xFFFFFFFFull;
  const uint32_t left = n - start;
  uint32_t total = 0, largest = 0;
  bool merge = false;
  for (;;) {
    int count = 0;
#pragma unroll
    for (int u = 0; u < kTieItems; ++u) {
      const uint32_t i = u * kTieBlock + t;
      const uint64_t k = src[total + i < left ? total + i : left - 1];
      const bool same = total + i < left && (k >> 32) == (first_key >> 32);
      p.o[i] = same ? (uint32_t)ordered_bits(k, xf) : 0xFFFFFFFFu;  // what is behind the run stays there
      count += __popcll(__ballot(same));
    }
    if (t % kWaveSize == 0) s_totals[t / kWaveSize] = (uint32_t)count;
    __syncthreads();
    count = 0;
    for (int w = 0; w < kTieWaves; ++w) count += (int)s_totals[w];
    bool inverted = false;
    for (int i = t; i + 1 < count; i += kTieBlock) inverted |= p.o[i] > p.o[i + 1];
    if (__syncthreads_or(inverted)) {
      sort_piece(p, s_totals, t);
      for (int i = t; i < count; i += kTieBlock)
        src[total + i] = raw_bits((uint64_t)(upper_ordered | p.o[i]), xf);
      if constexpr (VALUE_BYTES > 0) {
        for (int row = t; row < count; row += kTieMerges * kTieBlock) {
          Val v[kTieMerges];
#pragma unroll
          for (int u = 0; u < kTieMerges; ++u) v[u] = src_vals[total + p.from[min(row + u * kTieBlock, count - 1)]];
#pragma unroll
          for (int u = 0; u < kTieMerges; ++u)
            if (row + u * kTieBlock < count) dst_vals[total + row + u * kTieBlock] = v[u];
        }
        __syncthreads();
        copy_rows(src_vals + total, dst_vals + total, (uint32_t)count, t);
      }
    }
    if (count > 0) {
      merge |= total > 0 && p.o[0] < largest;
      largest = p.o[count - 1];
    }
    total += (uint32_t)count;
    __syncthreads();
    if (count < kPiece) break;
  }
  if (!merge) return;
  uint32_t* s_samples = reinterpret_cast<uint32_t*>(&p);
  // Every piece begins with a sample, or there are none (beyond 2^23 keys).
  int shift = 0;
  while (((total - 1) >> shift) + 1 > (uint32_t)(sizeof(p) / 4)) ++shift;
  const bool sampled = 1 << shift <= kPiece;
  for (uint32_t width = kPiece; width < total; width <<= 1) {
#pragma unroll 4
    for (uint32_t i = t; sampled && i << shift < total; i += kTieBlock)
      s_samples[i] = (uint32_t)ordered_bits(src[i << shift], xf);
    __syncthreads();
    // kTieMerges keys of a thread at once: a bisection is a chain of loads.
    for (uint32_t row = t; row < total; row += kTieMerges * kTieBlock) {
      uint32_t o[kTieMerges], lo[kTieMerges], hi[kTieMerges];
      auto middle_of = [&](uint32_t i) {
        const uint32_t pair = i & ~(2 * width - 1);
        return total - pair > width ? pair + width : total;
      };
#pragma unroll
      for (int u = 0; u < kTieMerges; ++u) {
        const uint32_t i = min(row + u * kTieBlock, total - 1);
        o[u] = (uint32_t)ordered_bits(src[i], xf);
      }
      // Keys of the other piece that go in front of this one: among the samples, ...
      auto bounds = [&](uint32_t i, uint32_t& first, uint32_t& end) {
        const uint32_t pair = i & ~(2 * width - 1), middle = middle_of(i);
        first = i < middle ? middle : pair;
        end = i < middle ? (total - pair > 2 * width ? pair + 2 * width : total) : middle;
      };
#pragma unroll
      for (int u = 0; u < kTieMerges; ++u) {
        uint32_t first, end;
        bounds(min(row + u * kTieBlock, total - 1), first, end);
        lo[u] = first >> shift;
        hi[u] = sampled && first < end ? ((end - 1) >> shift) + 1 : lo[u];
      }
      for (uint32_t step = width >> shift; step > 0; step >>= 1) {
#pragma unroll
        for (int u = 0; u < kTieMerges; ++u) {
          if (lo[u] >= hi[u]) continue;
          const uint32_t i = row + u * kTieBlock, m = (lo[u] + hi[u]) >> 1;
          const uint32_t q = s_samples[m];
          if (i < middle_of(i) ? q < o[u] : q <= o[u]) lo[u] = m + 1;
          else hi[u] = m;
        }
      }
      // ... then among the keys between two of them.
#pragma unroll
      for (int u = 0; u < kTieMerges; ++u) {
        uint32_t first, end;
        bounds(min(row + u * kTieBlock, total - 1), first, end);
        const uint32_t sample = lo[u];
        hi[u] = sampled && sample << shift < end ? sample << shift : end;
        lo[u] = sampled && sample << shift > first ? ((sample - 1) << shift) + 1 : first;
      }
      for (uint32_t step = sampled ? (1u << shift) >> 1 : width; step > 0; step >>= 1) {
#pragma unroll
        for (int u = 0; u < kTieMerges; ++u) {
          if (lo[u] >= hi[u]) continue;
          const uint32_t i = row + u * kTieBlock, m = (lo[u] + hi[u]) >> 1;
          const uint32_t q = (uint32_t)ordered_bits(src[m], xf);
          if (i < middle_of(i) ? q < o[u] : q <= o[u]) lo[u] = m + 1;
          else hi[u] = m;
        }
      }
#pragma unroll
      for (int u = 0; u < kTieMerges; ++u) {
        const uint32_t i = row + u * kTieBlock;
        lo[u] += i - middle_of(i);  // its place, from either half
        if (i < total) dst[lo[u]] = raw_bits((uint64_t)(upper_ordered | o[u]), xf);
      }
      if constexpr (VALUE_BYTES > 0) {
        Val v[kTieMerges];
#pragma unroll
        for (int u = 0; u < kTieMerges; ++u) v[u] = src_vals[min(row + u * kTieBlock, total - 1)];
#pragma unroll
        for (int u = 0; u < kTieMerges; ++u)
          if (row + u * kTieBlock < total) dst_vals[lo[u]] = v[u];
      }
    }
    __syncthreads();  // the next step reads what other threads wrote
    uint64_t* k = src; src = dst; dst = k;
    Val* v = src_vals; src_vals = dst_vals; dst_vals = v;
  }
  if (src != keys + start) {
    copy_rows(dst, src, total, t);
    if constexpr (VALUE_BYTES > 0) copy_rows(dst_vals, src_vals, total, t);
  }
  __syncthreads();
}

// (Compiled for 32 waves per CU, as the copy of finish() wants them too.)  long_starts:
// scratch, kTieLongsPerChunk words for every chunk that a block's waves take.
template <int VALUE_BYTES>
__global__ __launch_bounds__(kTieBlock, 8) void ties_kernel(
    uint64_t* keys_a, uint64_t* keys_b, typename ValueOf<VALUE_BYTES>::type* vals_a,
    typename ValueOf<VALUE_BYTES>::type* vals_b, int64_t n, KeyXform xf,
    const SortPlan* __restrict__ plan, int values_from_index, uint32_t* long_starts) {
  using Val = typename ValueOf<VALUE_BYTES>::type;
  __shared__ TiePiece s_piece;
  __shared__ uint32_t s_longs;
  if (plan->local_from != 0) return;  // local_sort_kernel has done it
  if (plan->ties_left == 0) {  // every digit was sorted
    finish<8, VALUE_BYTES>(keys_a, keys_b, vals_a, vals_b, n, plan, values_from_index);
    return;
  }
  uint64_t* keys = keys_a;  // an even number of passes ran
  Val* vals = vals_a;
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int64_t wave = (int64_t)blockIdx.x * kTieWaves + threadIdx.x / kWaveSize;
  const int64_t waves = (int64_t)gridDim.x * kTieWaves;
  const int64_t rounds = (n + waves * kTieChunk - 1) / (waves * kTieChunk);
  long_starts += (int64_t)blockIdx.x * rounds * (kTieWaves * kTieLongsPerChunk);
  if (threadIdx.x == 0) s_longs = 0u;
  __syncthreads();
  for (int64_t base = wave * kTieChunk; base < n; base += waves * kTieChunk) {
    // Upper halves of the rows; what lies outside of the input repeats the
    // nearest key and is masked below.
    uint32_t upper[kTieRows];
#pragma unroll
    for (int r = 0; r < kTieRows; ++r) {
      const int64_t i = base + r * kWaveSize + lane;
      upper[r] = (uint32_t)(keys[i < n ? i : n - 1] >> 32);
    }
    uint32_t before = (uint32_t)(keys[base > 0 ? base - 1 : 0] >> 32);
    const uint32_t after = (uint32_t)(keys[base + kTieChunk < n ? base + kTieChunk : n - 1] >> 32);
    uint32_t leads = 0;  // rows in which this lane holds a run's first key
#pragma unroll
    for (int r = 0; r < kTieRows; ++r) {
      const int64_t i = base + r * kWaveSize + lane;
      const uint32_t last = (uint32_t)__builtin_amdgcn_readlane((int)upper[r], kWaveSize - 1);
      const uint32_t following =
          r + 1 < kTieRows ? (uint32_t)__builtin_amdgcn_readfirstlane((int)upper[r + 1 < kTieRows ? r + 1 : r])
                           : after;
      uint32_t prev = shfl_up(upper[r], 1);
      uint32_t next = __shfl_down(upper[r], 1);
      if (lane == 0) prev = before;
      if (lane == kWaveSize - 1) next = following;
      if (i + 1 < n && next == upper[r] && (i == 0 || prev != upper[r])) leads |= 1u << r;
      before = last;
    }
    while (__ballot(leads != 0) != 0ull) {
      uint32_t start = 0;  // n is below 2^31
      int places = 0;      // more than the run has keys: 0 if this lane has ordered it
      if (leads != 0) {
        start = (uint32_t)base + (uint32_t)(__builtin_ctz(leads) * kWaveSize + lane);
        leads &= leads - 1;
        const uint32_t last = (uint32_t)n - 1;
        const uint64_t k0 = keys[start], k1 = keys[start + 1], k2 = keys[min(start + 2, last)],
                       k3 = keys[min(start + 3, last)];
        auto same = [&](uint64_t k, uint32_t j) { return start + j <= last && (k >> 32) == (k0 >> 32); };
        if (!same(k2, 2)) {  // by itself: as two of the three below it cost 2^27 uniform pairs 1 %
          if (ordered_bits(k1, xf) < ordered_bits(k0, xf)) {
            if constexpr (VALUE_BYTES > 0) {
              const Val v = vals[start];
              vals[start] = vals[start + 1];
              vals[start + 1] = v;
            }
            keys[start] = k1;
            keys[start + 1] = k0;
          }
        } else if (!same(k3, 3)) {
          // Lower halves with their places, so that equal keys keep their order.
          uint64_t x[3] = {ordered_bits(k0, xf) << 32, ordered_bits(k1, xf) << 32 | 1u,
                           same(k2, 2) ? ordered_bits(k2, xf) << 32 | 2u : ~0ull << 32 | 2u};
          auto order = [&](int i, int j) {
            const uint64_t lo = x[i] < x[j] ? x[i] : x[j];
            x[j] = x[i] < x[j] ? x[j] : x[i];
            x[i] = lo;
          };
          order(0, 1); order(1, 2); order(0, 1);
          const uint64_t upper_ordered = ordered_bits(k0, xf) & ~0xFFFFFFFFull;
          Val v[3];
          if constexpr (VALUE_BYTES > 0) {
#pragma unroll
            for (int j = 0; j < 3; ++j)
              if ((uint32_t)x[j] != (uint32_t)j) v[j] = vals[start + (uint32_t)x[j]];
          }
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            if ((uint32_t)x[j] == (uint32_t)j) continue;
            keys[start + j] = raw_bits((uint64_t)(upper_ordered | x[j] >> 32), xf);
            if constexpr (VALUE_BYTES > 0) vals[start + j] = v[j];
          }
        } else {
          const uint64_t k7 = keys[min(start + 7, last)], k15 = keys[min(start + 15, last)],
                         k31 = keys[min(start + 31, last)], k63 = keys[min(start + 63, last)],
                         k127 = keys[min(start + 127, last)];
          places = 8 << (int)same(k7, 7) << (int)same(k15, 15) << (int)same(k31, 31) << (int)same(k63, 63)
                     << (int)same(k127, 127);
          if (places == 256) long_starts[atomicAdd(&s_longs, 1u)] = start;
        }
      }
      if (__ballot(places != 0) == 0ull) continue;
      // As many runs at once as the wave has room for.
      for (int width = 8; width <= kWaveSize; width <<= 1) {
        for (uint64_t owners = __ballot(places == width); owners != 0ull;) {
          int mine = -1;
          for (int first = 0; first < kWaveSize && owners != 0ull; first += width, owners &= owners - 1)
            if ((lane & ~(width - 1)) == first) mine = __builtin_ctzll(owners);
          const uint32_t s = (uint32_t)__shfl((int)start, mine < 0 ? 0 : mine);
          order_runs<VALUE_BYTES>(keys, vals, s, mine >= 0, (uint32_t)n, xf, lane, width);
        }
      }
      for (uint64_t owners = __ballot(places == 128); owners != 0ull; owners &= owners - 1)
        order_two_rows<VALUE_BYTES>(
            keys, vals, (uint32_t)__builtin_amdgcn_readlane((int)start, __builtin_ctzll(owners)), (uint32_t)n, xf,
            lane);
    }
  }
  __syncthreads();
  const uint32_t longs = s_longs;
  for (uint32_t r = 0; r < longs; ++r)  // the same in every thread
    order_long_run<Val, VALUE_BYTES>(keys, keys_b, vals, vals_b, long_starts[r], (uint32_t)n, xf.xor_mask,
                                     xf.reference_term, xf.total_term,
                                     (__attribute__((address_space(3))) TiePiece*)&s_piece);
}

#include "radix_sort_local.hpp"

// ---- host side -------------------------------------------------------------

struct TempLayout {
  int64_t alt_keys, alt_vals, excl, plan, zero_begin, hist, tickets, status,
      status_stride, total;
  int64_t tiles;
};

// Layout for tiles of `block` threads.  Temp views are sized for the small
// block (more tiles, more status words); the large block's layout fits inside.
// Keys per thread of the class of short tiles an input takes (the shortest
// that makes at most `max_tiles` tiles), or 0: full tiles.
inline int pick_short_items(int64_t n, int key_bytes, int value_bytes, int64_t max_tiles) {
  if (value_bytes != 0) return 0;
  // 8-byte keys: their full tiles are half as long to begin with, and beyond
  // 128 short ones the longer look-back costs what the shorter tiles save.
  if (key_bytes == 8 && max_tiles > kShortTileMaxTiles / 4) max_tiles = kShortTileMaxTiles / 4;
  for (int c = 0; c < kShortTileClasses; ++c) {
    const int items = short_items_per_thread(key_bytes, c);
    if (div_up(n, (int64_t)kSortBlock * items) <= max_tiles) return items;
  }
  return 0;
}
// With the defaults (what temp views are sized by) the layout is that of the
// shortest tiles the input can be given: the 512-thread block's, or short
// tiles where they apply.
TempLayout make_layout(int64_t n, int key_bytes, int value_bytes, int block = kSortBlock,
                       int64_t tile_override = 0) {
  TempLayout L;
  int64_t tile = tile_override > 0 ? tile_override : tile_keys(key_bytes, value_bytes, block);
  if (tile_override <= 0 && block == kSortBlock) {
    const int short_items = pick_short_items(n, key_bytes, value_bytes, kShortTileMaxTiles);
    if (short_items > 0) tile = (int64_t)kSortBlock * short_items;
  }
  L.tiles = div_up(n, tile);
  int64_t off = 0;
  L.alt_keys = off; off += align_up(n * key_bytes, 256);
  L.alt_vals = off; off += align_up(n * value_bytes, 256);
  L.excl = off; off += kMaxPasses * kRadix * 4;
  L.plan = off; off += 256;
  L.zero_begin = off;
  L.hist = off; off += kMaxPasses * kRadix * 4;
  L.tickets = off; off += kMaxPasses * kTicketGroups * kTicketStride * 4;
  L.status = off;
  L.status_stride = L.tiles * kRadix * 4;
  // One status array per pass, or two by turns (sort_status_turns).
  off += L.status_stride * key_bytes;
  L.total = off;
  return L;
}

// Lengths at which the local sort is offered.  Below the first its draws would not fit the alternate
// keys.  8-byte keys between the other two (2^21 to 2^23) are sorted by their upper half (TieSampling), in
// four passes.  The local sort would be faster there where it is taken, and slower where the draws refuse it and the
// upper half follows (with a copy in front, us, the upper half / the local sort offered: u64 2^21 uniform 119 / 101, time stamps
// 139 / 106, Zipf 84 / 87, below 10^6 101 / 105, six copies 182 / 184; 2^22 148 / 124, 175 / 134, 101 / 106, 128 / 133, 229 / 234;
// 2^23 225 / 180, 273 / 195, 148 / 153, 195 / 199).  The line has nothing else for it than that these are the lengths at which the
// upper half was proven.
constexpr int64_t kLocalMinKeys = 1ll << 14;
constexpr int64_t kLocalMinKeysAfterTies = (1ll << 23) + 1;
static_assert(kLocalMinKeys >= 1ll << kLocalMinDrawBits, "the draws lie in the alternate keys");
static_assert(kLocalMinKeysAfterTies * 8 >= kLocalDrawsOffset + (8ll << kLocalMaxDrawBits),
              "the draws lie in the alternate keys, behind the table");
inline bool local_wanted(int64_t n, int key_bytes) {
  return n >= kLocalMinKeys && (key_bytes != 8 || n < kTieMinKeys || n >= kLocalMinKeysAfterTies);
}

KeyXform make_xform(int32_t key_type, int32_t flags) {
  const int bits = elem_size(key_type) * 8;
  const uint64_t all = bits == 64 ? ~0ull : ((1ull << bits) - 1ull);
  const uint64_t sign = 1ull << (bits - 1);
  KeyXform xf{0, 0, 0};
  switch (key_type) {
    case ILGPU_HIP_I8: case ILGPU_HIP_I16: case ILGPU_HIP_I32: case ILGPU_HIP_I64:
      xf.xor_mask = sign;
      break;
    case ILGPU_HIP_F16: case ILGPU_HIP_F32: case ILGPU_HIP_F64:
      if (flags & ILGPU_HIP_SORT_FLOAT_TOTAL_ORDER) {
        xf.xor_mask = sign;
        xf.total_term = sign - 1ull;
      } else {
        // Half: (uint)~bits >> 15 keeps the sign-extended upper ones, so bits
        // 1..15 are always flipped (RadixSortOperations.tt:77-80).
        xf.xor_mask = key_type == ILGPU_HIP_F16 ? 0xFFFEull : sign;
        xf.reference_term = 1ull;
      }
      break;
    default:
      break;
  }
  if (flags & ILGPU_HIP_SORT_DESCENDING) xf.xor_mask ^= all;
  return xf;
}

// The passes of one sort with tiles of BLOCK threads and ITEMS keys per thread.
// AT_ONCE: a block for every tile.
template <int KEY_BYTES, int VALUE_BYTES, int BLOCK, bool AT_ONCE = false,
          int ITEMS = items_per_thread(KEY_BYTES, VALUE_BYTES)>
int32_t launch_passes(hipStream_t stream, const SortArgs& a, const TempLayout& L, char* base,
                      const KeyXform& xf, int cus) {
  using K = typename KeyOf<KEY_BYTES>::type;
  using Val = typename ValueOf<VALUE_BYTES>::type;
  K* keys_a = static_cast<K*>(a.keys);
  K* keys_b = reinterpret_cast<K*>(base + L.alt_keys);
  Val* vals_a = static_cast<Val*>(a.values);
  Val* vals_b = reinterpret_cast<Val*>(base + L.alt_vals);
  uint32_t* excl = reinterpret_cast<uint32_t*>(base + L.excl);
  SortPlan* plan = reinterpret_cast<SortPlan*>(base + L.plan);
  uint32_t* tickets = reinterpret_cast<uint32_t*>(base + L.tickets);
  const int passes = KEY_BYTES;
  const int from_index = a.value_source == ILGPU_HIP_VALUES_FROM_INDEX
                             ? 1
                             : (a.value_source == ILGPU_HIP_VALUES_FROM_INDEX_AS_FLOAT ? 2 : 0);
  const bool float_keys = (xf.reference_term | xf.total_term) != 0;
  constexpr bool kOfKeys = KEY_BYTES == 4 && VALUE_BYTES == 0 && BLOCK == kSortBlock;
  constexpr bool kOnlyFloats = kOfKeys && ITEMS == kFloatItems, kNoFloats = kOfKeys && ITEMS == ILGPU_HIP_SORT_ITEMS;
  auto* pass_kernel = onesweep_kernel<KEY_BYTES, VALUE_BYTES, kOnlyFloats, BLOCK, ITEMS, AT_ONCE>;
  if constexpr (KEY_BYTES >= 2 && !kNoFloats) {  // there is no 1-byte floating-point key
    if (float_keys) pass_kernel = onesweep_kernel<KEY_BYTES, VALUE_BYTES, true, BLOCK, ITEMS, AT_ONCE>;
  }
  int64_t grid = L.tiles;
  if constexpr (!AT_ONCE) {
    // Resident blocks per CU of this instantiation: asked once per device and
    // kernel (the query costs microseconds, which small sorts would feel).
    static std::atomic<int> cached_per_cu[kMaxCachedDevices][2];  // per instantiation
    const int device = current_device();
    std::atomic<int>* cached =
        device >= 0 && device < kMaxCachedDevices ? &cached_per_cu[device][float_keys ? 1 : 0]
                                                  : nullptr;
    int per_cu = cached ? cached->load(std::memory_order_relaxed) : 0;
    if (per_cu == 0) {
      ILGPU_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
          &per_cu, pass_kernel, BLOCK, 0));
      if (per_cu < 1) per_cu = 1;
      if (cached) cached->store(per_cu, std::memory_order_relaxed);
    }
    grid = std::min((int64_t)cus * per_cu, L.tiles);
  }
  // Every group of blocks needs a block: a grid below eight blocks (few tiles, or
  // a device with very few compute units) forms as many groups as it has blocks.
  const int groups = grid < kTicketGroups ? (int)grid : kTicketGroups;
  // Chunks as long as leave every block of the grid a tile of its own in the
  // first round (short inputs: single tiles, handed out round-robin).
  int chunk_shift = 0;
  while (chunk_shift < kMaxChunkShift && (grid << (chunk_shift + 1)) <= L.tiles) ++chunk_shift;
  const uint32_t spin_limit = g_sort_spin_limit.load(std::memory_order_relaxed);
  uint32_t* status = reinterpret_cast<uint32_t*>(base + L.status);
  for (int p = 0; p < passes; ++p) {
    {
      ProfileScope scope(stream, "sort_onesweep");
      hipLaunchKernelGGL(pass_kernel,
                         dim3((unsigned)grid), dim3(BLOCK), 0, stream,
                         keys_a, keys_b, vals_a, vals_b, a.n, p, xf, excl,
                         status,
                         grid == L.tiles ? nullptr : tickets + p * kTicketGroups * kTicketStride,
                         plan, (int)L.tiles, from_index, groups, chunk_shift, spin_limit);
    }
    ILGPU_HIP_CHECK(hipGetLastError());
  }
  return ILGPU_HIP_SUCCESS;
}

// The passes of a keys-only sort in the pipelined form (one block per compute unit).
template <int KEY_BYTES>
int32_t launch_passes_pipelined(hipStream_t stream, const SortArgs& a, const TempLayout& L,
                                char* base, const KeyXform& xf, int cus) {
  using K = typename KeyOf<KEY_BYTES>::type;
  K* keys_a = static_cast<K*>(a.keys);
  K* keys_b = reinterpret_cast<K*>(base + L.alt_keys);
  uint32_t* excl = reinterpret_cast<uint32_t*>(base + L.excl);
  SortPlan* plan = reinterpret_cast<SortPlan*>(base + L.plan);
  uint32_t* tickets = reinterpret_cast<uint32_t*>(base + L.tickets);
  auto* pass_kernel = onesweep_pipelined_kernel<KEY_BYTES, false>;
  if constexpr (KEY_BYTES >= 2) {  // there is no 1-byte floating-point key
    if ((xf.reference_term | xf.total_term) != 0)
      pass_kernel = onesweep_pipelined_kernel<KEY_BYTES, true>;
  }
  int64_t grid = cus;  // 1024 threads and 150 KiB of LDS: one block per compute unit
  if (grid > L.tiles) grid = L.tiles;
  const int groups = grid < kTicketGroups ? (int)grid : kTicketGroups;
  // Chunks of 16 and 32 tiles, which the write pattern by itself prefers
  // (bench_bounds scatter), lose here: 0.492 and 0.572 ms per pass against 0.484.
  int chunk_shift = 0;
  while (chunk_shift < kMaxChunkShift && (grid << (chunk_shift + 1)) <= L.tiles) ++chunk_shift;
  const uint32_t spin_limit = g_sort_spin_limit.load(std::memory_order_relaxed);
#ifndef ILGPU_HIP_SORT_SCANNER
#define ILGPU_HIP_SORT_SCANNER 1
#endif
  // One block scans instead of sorting when the grid can spare it.
  const int with_scanner = ILGPU_HIP_SORT_SCANNER && grid >= 64 ? 1 : 0;
  uint32_t* status = reinterpret_cast<uint32_t*>(base + L.status);
  for (int p = 0; p < KEY_BYTES; ++p) {
    {
      ProfileScope scope(stream, "sort_onesweep");
      hipLaunchKernelGGL(pass_kernel, dim3((unsigned)grid), dim3(1024), 0, stream, keys_a, keys_b,
                         a.n, p, xf, excl, status, tickets + p * kTicketGroups * kTicketStride,
                         plan, (int)L.tiles, groups, chunk_shift, spin_limit, with_scanner);
    }
    ILGPU_HIP_CHECK(hipGetLastError());
  }
  return ILGPU_HIP_SUCCESS;
}

template <int KEY_BYTES, int VALUE_BYTES>
int32_t launch_sized(hipStream_t stream, const SortArgs& a) {
  using K = typename KeyOf<KEY_BYTES>::type;
  using Val = typename ValueOf<VALUE_BYTES>::type;
  if (a.n <= (int64_t)tile_keys(KEY_BYTES, VALUE_BYTES, kSortBlock) &&
      g_sort_small_kernel.load(std::memory_order_relaxed) != 0) {
    // one tile: one block, one launch, no temp
    const KeyXform xf = make_xform(a.key_type, a.flags);
    constexpr int kFullItems = items_per_thread(KEY_BYTES, VALUE_BYTES);
    auto launch_small = [&](auto items) -> int32_t {
      constexpr int kRows = decltype(items)::value;
      constexpr int kBlock = small_sort_block(KEY_BYTES, VALUE_BYTES, false, kRows);
      constexpr int kFloatBlock = small_sort_block(KEY_BYTES, VALUE_BYTES, true, kRows);
      auto* kernel = small_sort_kernel<KEY_BYTES, VALUE_BYTES, false, kBlock, small_sort_items(kBlock, kRows)>;
      unsigned block = kBlock;
      if constexpr (KEY_BYTES >= 2) {  // there is no 1-byte floating-point key
        if ((xf.reference_term | xf.total_term) != 0) {
          kernel = small_sort_kernel<KEY_BYTES, VALUE_BYTES, true, kFloatBlock, small_sort_items(kFloatBlock, kRows)>;
          block = kFloatBlock;
        }
      }
      ProfileScope scope(stream, "sort_small");
      hipLaunchKernelGGL(kernel, dim3(1), dim3(block), 0, stream, static_cast<K*>(a.keys),
                         static_cast<Val*>(a.values), (int)a.n, xf,
                         a.value_source == ILGPU_HIP_VALUES_FROM_INDEX
                               ? 1
                               : (a.value_source == ILGPU_HIP_VALUES_FROM_INDEX_AS_FLOAT ? 2 : 0));
      ILGPU_HIP_CHECK(hipGetLastError());
      return ILGPU_HIP_SUCCESS;
    };
    if constexpr (kSmallSortItemsA < kFullItems) {
      if (a.n <= (int64_t)kSortBlock * kSmallSortItemsA)
        return launch_small(std::integral_constant<int, kSmallSortItemsA>{});
    }
    if constexpr (kSmallSortItemsB < kFullItems) {
      if (a.n <= (int64_t)kSortBlock * kSmallSortItemsB)
        return launch_small(std::integral_constant<int, kSmallSortItemsB>{});
    }
    if constexpr (kSmallSortItemsC < kFullItems) {
      if (a.n <= (int64_t)kSortBlock * kSmallSortItemsC)
        return launch_small(std::integral_constant<int, kSmallSortItemsC>{});
    }
    return launch_small(std::integral_constant<int, kFullItems>{});
  }
  const int cus = device_cu_count();
  int64_t min_tiles_per_cu = g_sort_large_min_tiles_per_cu.load(std::memory_order_relaxed);
  if (min_tiles_per_cu < 0)
    min_tiles_per_cu = VALUE_BYTES > 0 ? kLargeMinTilesPerCuPairs : kLargeMinTilesPerCuKeys;
  const bool use_large =
      div_up(a.n, (int64_t)tile_keys(KEY_BYTES, VALUE_BYTES, kSortBlockLarge)) >=
      min_tiles_per_cu * cus;
  const KeyXform xf = make_xform(a.key_type, a.flags);
#ifndef ILGPU_HIP_SORT_PIPELINED
#define ILGPU_HIP_SORT_PIPELINED 1
#endif
#ifndef ILGPU_HIP_SORT_PIPELINED_FLOAT
#define ILGPU_HIP_SORT_PIPELINED_FLOAT 1
#endif
  // Large keys-only sorts take the pipelined form of the pass.
  const bool use_pipelined =
      ILGPU_HIP_SORT_PIPELINED && VALUE_BYTES == 0 && use_large &&
      (ILGPU_HIP_SORT_PIPELINED_FLOAT || (xf.reference_term | xf.total_term) == 0);
  // Short inputs of keys take short tiles (the parameter can only lower the
  // limit: temp views are sized by the default).
  int64_t short_max_tiles = g_sort_short_tile_max_tiles.load(std::memory_order_relaxed);
  if (short_max_tiles < 0 || short_max_tiles > kShortTileMaxTiles)
    short_max_tiles = kShortTileMaxTiles;
  // Two 512-thread blocks are resident per compute unit; a second round of
  // short tiles would cost more than full tiles do.
  if (short_max_tiles > 2 * (int64_t)cus) short_max_tiles = 2 * (int64_t)cus;
  const int short_items =
      use_large ? 0 : pick_short_items(a.n, KEY_BYTES, VALUE_BYTES, short_max_tiles);
  const bool float_tiles = KEY_BYTES == 4 && VALUE_BYTES == 0 && (xf.reference_term | xf.total_term) != 0 &&
                           !use_large && short_items == 0;
  TempLayout L =
      make_layout(a.n, KEY_BYTES, VALUE_BYTES, use_large ? kSortBlockLarge : kSortBlock,
                  use_pipelined ? pipelined_tile_keys(KEY_BYTES)
                                : (short_items > 0 ? kSortBlock * short_items
                                   : float_tiles   ? kSortBlock * kFloatItems
                                                   : tile_keys(KEY_BYTES, VALUE_BYTES,
                                                               use_large ? kSortBlockLarge : kSortBlock)));
  // (What the temp view is sized for: the layout's own, or somewhat less where its tiles are shorter than full ones, which two
  // status arrays fit all the same.)
  static_assert(2 * ILGPU_HIP_SORT_ITEMS < 4 * kFloatItems, "two arrays for these tiles in four for full ones");
  L.total = std::min(L.total, make_layout(a.n, KEY_BYTES, VALUE_BYTES).total);
  char* base = reinterpret_cast<char*>(align_up((int64_t)(uintptr_t)a.temp, 256));
  K* keys_a = static_cast<K*>(a.keys);
  K* keys_b = reinterpret_cast<K*>(base + L.alt_keys);
  Val* vals_a = static_cast<Val*>(a.values);
  Val* vals_b = reinterpret_cast<Val*>(base + L.alt_vals);
  uint32_t* excl = reinterpret_cast<uint32_t*>(base + L.excl);
  SortPlan* plan = reinterpret_cast<SortPlan*>(base + L.plan);
  uint32_t* hist = reinterpret_cast<uint32_t*>(base + L.hist);
  const int passes = KEY_BYTES;
  const int from_index = a.value_source == ILGPU_HIP_VALUES_FROM_INDEX
                             ? 1
                             : (a.value_source == ILGPU_HIP_VALUES_FROM_INDEX_AS_FLOAT ? 2 : 0);

  int shift = 0;  // replicas of the histogram: as many as kHistLdsWords of LDS counters hold
  while ((1 << (shift + 1)) <= 32 &&
         ((passes * kRadix) << (shift + 1)) <= kHistLdsWords)
    ++shift;
  const size_t hist_lds = (size_t)((passes * kRadix) << shift) * 4;
  // A block's fixed cost is its flush, one global atomic per digit value and
  // position, which all blocks issue at about the same time.  Up to half a
  // block per CU as soon as every thread has four vectors to count, more
  // only when every thread has sixteen (2^20 u32 keys: 7.5 us instead of
  // 15.5 with one vector per thread; 2^22: 12.3 instead of 17.1).
  const int64_t vectors = div_up(a.n, Vec16<K>::N);
  const int64_t few = std::min<int64_t>(div_up(vectors, kHistBlock * 4), std::max(cus / 2, 1));
  int64_t hist_blocks = std::max(few, div_up(vectors, kHistBlock * 16));
  // Two blocks of 64 KiB of counters are resident per CU: no second round.
  if (hist_blocks > (int64_t)cus * ILGPU_HIP_SORT_HIST_BLOCKS_PER_CU)
    hist_blocks = (int64_t)cus * ILGPU_HIP_SORT_HIST_BLOCKS_PER_CU;
  if (hist_blocks < 1) hist_blocks = 1;

  TieSampling ties{};
  int64_t table_words = 0;
  if (KEY_BYTES == 8 && a.n >= kTieMinKeys) {
    uint32_t bits = kTieMinSampleBits;
    while (bits < kTieMaxSampleBits && a.n >> (bits + 9) != 0) ++bits;
    while ((1ll << bits) > hist_blocks * kHistBlock) --bits;  // few compute units
    ties.table = reinterpret_cast<unsigned long long*>(keys_b);
    // Words of the first tickets' lines that no group uses, cleared with them.
    ties.counts = reinterpret_cast<uint32_t*>(base + L.tickets) + 1;
    ties.sample_bits = bits;
    ties.max_doubles = (uint32_t)((1ull << (2 * bits)) / (uint64_t)a.n);
    ties.max_pairs = (uint32_t)((3ull << (2 * bits)) / (uint64_t)a.n);
    table_words = 2ll << (bits + kTieSlotsPerDrawLog2);
  }
  // The local sort: inputs whose topmost digit alone can make runs that fit a window ask the
  // digit's counts, longer ones the draws.
  constexpr bool kLocal = local_sorts(KEY_BYTES, VALUE_BYTES);
  LocalSampling local{};
  if constexpr (kLocal) {
    constexpr int64_t kWindow = local_window(KEY_BYTES, VALUE_BYTES);
    if (local_wanted(a.n, KEY_BYTES) &&
        local_deferred_bytes(a.n, local_blocks(a.n, cus), (uint32_t)kWindow) <= L.total - L.status) {
      local.limits = local_limits(a.n, KEY_BYTES, VALUE_BYTES);
      local.draws = reinterpret_cast<char*>(keys_b) + (ties.table != nullptr ? kLocalDrawsOffset : 0);
      // Words of the first ticket's line that no group uses, cleared with it.
      local.from = reinterpret_cast<uint32_t*>(base + L.tickets) + 4;
    }
  }
  int32_t rc;
  // Full tiles, no more of them than run at the same time, two per compute unit, look back as short ones do.
  // (Not every value size is worth two more kernels.
  // Full tiles of 4-byte keys would spill: 2^23 u32 keys 125 -> 132 us.)  Two tiles walk: the second one needs one word, for which
  // the other look-back has a barrier more (pairs with a copy in front, us, at once / a walk: 13 619 u32 with u64 53.6 / 52.3, 15 564 floats
  // with u32 56.0 / 54.3, 9728 doubles with u64 83.7 / 82.2; but 9318 doubles with u32, whose walk spills, 101.4 / 104).
  constexpr bool kAtOnce = VALUE_BYTES == 0 ? KEY_BYTES == 8 : KEY_BYTES >= 4 && (VALUE_BYTES == 4 || VALUE_BYTES == 8);
  const bool full_at_once = kAtOnce && !use_large && short_items == 0 && !float_tiles &&
                            L.tiles > (KEY_BYTES == 8 && VALUE_BYTES == 4 ? 0 : 2) && L.tiles <= 2 * (int64_t)cus;
  const bool turns = sort_status_turns(KEY_BYTES, use_large ? kSortBlockLarge : kSortBlock,
                                       short_items > 0 || full_at_once, float_tiles);
  const int64_t words = ((turns ? L.status + L.status_stride : L.total) - L.zero_begin) / 4;
  if (local.draws != nullptr) {
    auto* draw_kernel = sort_draw_kernel<K, false>;
    if ((xf.reference_term | xf.total_term) != 0) draw_kernel = sort_draw_kernel<K, true>;
    const int64_t blocks = std::min<int64_t>(
        div_up(std::max(std::max(words, table_words), (int64_t)1 << local.limits.draw_bits), 256), (int64_t)cus * 8);
    ProfileScope scope(stream, "zero_words");
    hipLaunchKernelGGL(draw_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, hist, words,
                       reinterpret_cast<uint32_t*>(ties.table), table_words, keys_a, a.n, xf,
                       static_cast<K*>(const_cast<void*>(local.draws)), local.limits.draw_bits);
    ILGPU_HIP_CHECK(hipGetLastError());
  } else {
    rc = launch_zero_words(stream, hist, words,
                           reinterpret_cast<uint32_t*>(ties.table), table_words);
    if (rc != ILGPU_HIP_SUCCESS) return rc;
  }

  {
    ProfileScope scope(stream, "sort_histogram");
    auto* histogram_kernel = sort_histogram_kernel<K, false>;
    if constexpr (KEY_BYTES >= 2) {  // there is no 1-byte floating-point key
      if ((xf.reference_term | xf.total_term) != 0) histogram_kernel = sort_histogram_kernel<K, true>;
    }
    // (One block more looks at the draws, unless that would start a second round.)
    if (local.draws != nullptr && (hist_blocks < (int64_t)cus * ILGPU_HIP_SORT_HIST_BLOCKS_PER_CU || hist_blocks < 2))
      ++hist_blocks;
    hipLaunchKernelGGL(histogram_kernel, dim3((unsigned)hist_blocks),
                       dim3(kHistBlock), hist_lds, stream, keys_a, a.n, xf, passes,
                       shift, hist, ties, local);
    ILGPU_HIP_CHECK(hipGetLastError());
  }
  {
    ProfileScope scope(stream, "sort_plan");
    hipLaunchKernelGGL(plan_kernel, dim3(1), dim3(kPlanBlock), 0, stream, hist, excl,
                       plan, passes, (uint32_t)a.n, ties, local.from, local.limits.max_run,
                       (uint32_t)local_window(KEY_BYTES, VALUE_BYTES));
  }
  ILGPU_HIP_CHECK(hipGetLastError());

  if (use_pipelined) {
    if constexpr (VALUE_BYTES == 0)
      rc = launch_passes_pipelined<KEY_BYTES>(stream, a, L, base, xf, cus);
  } else if (use_large) {
    rc = launch_passes<KEY_BYTES, VALUE_BYTES, kSortBlockLarge>(stream, a, L, base, xf, cus);
  } else if (short_items > 0) {
    if constexpr (VALUE_BYTES == 0) {
      constexpr int kA = short_items_per_thread(KEY_BYTES, 0);
      constexpr int kB = short_items_per_thread(KEY_BYTES, 1);
      constexpr int kC = short_items_per_thread(KEY_BYTES, 2);
      if (short_items == kA)
        rc = launch_passes<KEY_BYTES, 0, kSortBlock, true, kA>(stream, a, L, base, xf, cus);
      else if (short_items == kB)
        rc = launch_passes<KEY_BYTES, 0, kSortBlock, true, kB>(stream, a, L, base, xf, cus);
      else
        rc = launch_passes<KEY_BYTES, 0, kSortBlock, true, kC>(stream, a, L, base, xf, cus);
    }
  } else if (float_tiles) {
    if constexpr (KEY_BYTES == 4 && VALUE_BYTES == 0)
      rc = L.tiles <= 2 * (int64_t)cus
               ? launch_passes<4, 0, kSortBlock, true, kFloatItems>(stream, a, L, base, xf, cus)
               : launch_passes<4, 0, kSortBlock, false, kFloatItems>(stream, a, L, base, xf, cus);
  } else if (full_at_once) {
    if constexpr (kAtOnce)
      rc = launch_passes<KEY_BYTES, VALUE_BYTES, kSortBlock, true>(stream, a, L, base, xf, cus);
  } else {
    rc = launch_passes<KEY_BYTES, VALUE_BYTES, kSortBlock>(stream, a, L, base, xf, cus);
  }
  if (rc != ILGPU_HIP_SUCCESS) return rc;
  if constexpr (kLocal) {
    if (local.draws != nullptr) {
      const int64_t blocks = local_blocks(a.n, cus);
      const int finishes = ties.table == nullptr ? 1 : 0;
      auto* kernel = local_sort_kernel<KEY_BYTES, VALUE_BYTES, false>;
      if ((xf.reference_term | xf.total_term) != 0) kernel = local_sort_kernel<KEY_BYTES, VALUE_BYTES, true>;
      ProfileScope scope(stream, "sort_local");
      hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(LocalBlock::kBlock), 0, stream, keys_a, keys_b,
                         vals_a, vals_b, (uint32_t)a.n, xf, plan, excl, from_index, finishes,
                         reinterpret_cast<uint2*>(base + L.status));
      ILGPU_HIP_CHECK(hipGetLastError());
      if (finishes) return ILGPU_HIP_SUCCESS;
    }
  }
  if constexpr (KEY_BYTES == 8) {
    if (ties.table != nullptr) {
      int64_t blocks = div_up(a.n, kTieBlock * kTieRows);
      if (blocks > (int64_t)cus * 8) blocks = (int64_t)cus * 8;
      // The list of long runs lies in the status words, which the passes are done
      // with: kTieLongsPerChunk words per chunk, for at most twice as many chunks as
      // there are (the last round of a grid), against 256 words per tile and digit position.
      static_assert(2 * kTieLongsPerChunk * 4 * (tile_keys(8, 0, kSortBlockLarge) / kTieChunk + 1) <= 8 * kRadix * 4,
                    "room for the list of long runs");
      ProfileScope scope(stream, "sort_finish");
      hipLaunchKernelGGL((ties_kernel<VALUE_BYTES>), dim3((unsigned)blocks), dim3(kTieBlock), 0, stream,
                         keys_a, keys_b, vals_a, vals_b, a.n, xf, plan, from_index,
                         reinterpret_cast<uint32_t*>(base + L.status));
      ILGPU_HIP_CHECK(hipGetLastError());
      return ILGPU_HIP_SUCCESS;
    }
  }
  {
    // Mostly there is nothing to copy and every block returns at once; 16
    // keys per thread are few enough blocks for that and enough for the copy.
    int64_t blocks = div_up(a.n, 256 * 16);
    if (blocks > (int64_t)cus * 8) blocks = (int64_t)cus * 8;
    ProfileScope scope(stream, "sort_finish");
    hipLaunchKernelGGL((finish_kernel<KEY_BYTES, VALUE_BYTES>),
                       dim3((unsigned)blocks), dim3(256), 0, stream, keys_a,
                       keys_b, vals_a, vals_b, a.n, plan, from_index);
    ILGPU_HIP_CHECK(hipGetLastError());
  }
  return ILGPU_HIP_SUCCESS;
}

template <int KEY_BYTES>
int32_t launch_value(hipStream_t stream, const SortArgs& a) {
  switch (a.value_bytes) {
    case 0: return launch_sized<KEY_BYTES, 0>(stream, a);
    case 1: return launch_sized<KEY_BYTES, 1>(stream, a);
    case 2: return launch_sized<KEY_BYTES, 2>(stream, a);
    case 4: return launch_sized<KEY_BYTES, 4>(stream, a);
    case 8: return launch_sized<KEY_BYTES, 8>(stream, a);
    case 16: return launch_sized<KEY_BYTES, 16>(stream, a);
    default: return ILGPU_HIP_ERROR_NOT_SUPPORTED;
  }
}


}  // namespace

}  // namespace ilgpu_hip
