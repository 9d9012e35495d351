// Part of radix_sort_impl.hpp: what is left after passes over the upper digits.
//
// After the passes over the digits from plan->local_from on, keys that agree in
// those digits stand next to each other, in their original order: a run.  A run
// of some thousand keys fits the LDS of a block, where all of its lower digits are
// sorted at once, however many there are: one read and one write of the keys
// instead of a pass for every digit.
//
// A block owns the runs that start in its part of the input and takes as many
// whole runs as fit its LDS at a time: a window.  The keys of a window lie in a
// known range (the upper digits of its first and last run), which is cut into 2^15
// equal bins, some four for every key.  One returning LDS add per key on the
// count of its bin gives the keys of a bin different places; a scan over the
// counts gives the bins theirs; the few bins that hold two keys or more are put
// into order afterwards.  Four bins share a word, 4 bits of count each, with the
// place of the first of them in the upper half.
//
// What bounds it: 41 vector operations per key and row (60 % of the time busy), next to seven LDS
// operations (half of it) and the 16 bytes that 2^28 u32 keys move each (540 us against 330 for a copy).
// Sorting a window by digits takes eight LDS operations for two digits and twelve where a window
// holds more than one run; bins take the same seven whatever is left of the key.  Four bins for
// every key: with one, a key in four would have to be put into order with others.  Blocks of 256
// threads, four on a compute unit, so that some load and store while others count.
// (With a copy in front, us, every digit by passes / this: u32 keys 2^28 2378 / 2049, 2^26 648 / 567, 2^24
// 238 / 193, 2^20 71.5 / 52.0; u64 keys with index values 2^27 3572 / 2723, where four passes and the ties
// came before; 300 000 u64 keys with values 120 / 54.)
//
// Values that come half a time or more each on average share more bins than the list of them holds in a full window: there
// every thread looks at its places for keys in the wrong order instead.  (u32 keys with a copy in front, us, every digit / such
// windows by digits / this: 2^28 keys, each value once on average, 2365 / 4525 / 2385, 2^26 656 / 1129 / 665, 2 000 000 92 / 116 / 86.)
//
// Windows whose keys crowd a bin with sixteen or more (many copies of a key,
// keys clustered within a run) are sorted digit by digit in LDS, like a tile of
// the sort; a run longer than a window digit by digit through memory, by its
// block.  Both are decided from the keys themselves: the answer is right whatever
// the plan believed of them.

struct LocalLds {
  __attribute__((aligned(16))) unsigned char stage[LocalBlock::kStageBytes];
  uint16_t list[LocalBlock::kList];
  uint32_t sums[LocalBlock::kWaves];
  uint32_t bounds[2];
  uint32_t listed;
  uint32_t deferred;  // windows and runs that wait until the others are done
};
static_assert(sizeof(LocalLds) <= 40 * 1024, "four blocks on a compute unit");

// The first position from x on that starts a run (n if there is none): by one wave, 64 keys
// at growing distances until one of them has another prefix, then between the last
// two.
template <typename K>
__device__ __forceinline__ uint32_t local_run_start(const K* src, uint32_t x, uint32_t n, const KeyXform& xf,
                                                    int below, int lane) {
  if (x == 0 || x >= n) return x < n ? x : n;
  uint32_t same = x - 1;  // a position of the run that x - 1 is in
  const K prefix = (K)(ordered_bits(src[same], xf) >> below);
  int step_log2 = 0;
  bool grow = true;
  while (true) {
    const uint64_t at = (uint64_t)same + ((uint64_t)(lane + 1) << step_log2);
    const bool other = at >= n || (K)(ordered_bits(src[at], xf) >> below) != prefix;
    const uint64_t others = __ballot(other);
    if (others == 0ull) {
      same += 64u << step_log2;
      if (grow) step_log2 += 6;
      continue;
    }
    grow = false;
    same += (uint32_t)__builtin_ctzll(others) << step_log2;
    if (step_log2 == 0) return same + 1;
    step_log2 -= 6;
  }
}

// The same where one pass has run, whose digits are the runs: by their offsets, one round trip instead of three.
__device__ __forceinline__ uint32_t local_digit_start(const uint32_t* excl, uint32_t x, uint32_t n, int lane) {
  const uint4 at = reinterpret_cast<const uint4*>(excl)[lane];
  uint32_t start = n;
  start = at.w >= x && at.w < start ? at.w : start;
  start = at.z >= x && at.z < start ? at.z : start;
  start = at.y >= x && at.y < start ? at.y : start;
  start = at.x >= x && at.x < start ? at.x : start;
#pragma unroll
  for (int s = 1; s < kWaveSize; s <<= 1) {
    const uint32_t other = shfl(start, lane ^ s);
    start = other < start ? other : start;
  }
  return start;
}

// `count` elements, by `blocks` blocks (this one: `block`): four neighbouring ones at a time, the
// grid's next to each other, past the caches: HBM bounds it.  (Two loads of a thread in flight and plain
// stores, keys below 10^6 with a copy in front, us, before / now: u32 2^23 135.8 / 132.6, 2^24 217.6 / 211.4, 2^26
// 632.9 / 617.8, pairs of 2^24 u32 343.9 / 328.5; four loads, each a grid further on: 2^24 225.)
template <typename E>
__device__ __forceinline__ void local_copy(const E* from, E* to, uint32_t count, uint32_t block, uint32_t blocks) {
  typedef E Four __attribute__((ext_vector_type(4), aligned(sizeof(E))));
  constexpr uint32_t kBlock = (uint32_t)LocalBlock::kBlock;
  const uint32_t t = threadIdx.x;
  const uint32_t fours = count / 4;
  const Four* f = reinterpret_cast<const Four*>(from);
  Four* g = reinterpret_cast<Four*>(to);
  for (uint32_t i = block * kBlock + t; i < fours; i += blocks * kBlock) __builtin_nontemporal_store(f[i], &g[i]);
  if (block == 0)
    for (uint32_t i = fours * 4 + t; i < count; i += kBlock) to[i] = from[i];
}

// ---- digit by digit -------------------------------------------------------------
// Ranks the block's keys (lane l of wave w holds the elements w * 64 * rows + j * 64 + l) by
// one digit: rank[j] becomes the element's place, starts (thread t: of digit t) that of
// a digit's first key, counts its keys.  Counters as in sort_tile; the stage holds them.
template <typename K, int ITEMS>
__device__ __forceinline__ void local_rank(const K (&key)[ITEMS], uint32_t (&rank)[ITEMS], int rows,
                                           uint32_t first_local, uint32_t count, int shift, LocalLds& lds,
                                           uint32_t& digit_start, uint32_t& digit_count) {
  constexpr int kWaves = LocalBlock::kWaves;
  const int t = threadIdx.x, lane = t & (kWaveSize - 1), wave = t / kWaveSize;
  uint32_t* counter = reinterpret_cast<uint32_t*>(lds.stage);
  uint32_t* mine = counter + wave * kRadix;
  __syncthreads();  // the stage has been read
#pragma unroll
  for (int q = 0; q < kRadix / kWaveSize; ++q) mine[q * kWaveSize + lane] = 0u;
  // What is behind the keys takes digit 255 and stays behind them.
  auto digit = [&](int j) -> uint32_t {
    return first_local + j * kWaveSize < count ? (uint32_t)(key[j] >> shift) & (kRadix - 1) : (uint32_t)(kRadix - 1);
  };
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    rank[j] = 0;
    if (j < rows) {
      const uint32_t d = digit(j);
      // a row that is all one digit: lane 0 adds for the row (see sort_tile)
      const bool whole = __ballot(d == (uint32_t)__builtin_amdgcn_readfirstlane((int)d)) == ~0ull;
      uint32_t r = 0;
      if (!whole || lane == 0)
        r = __hip_atomic_fetch_add(mine + d, whole ? (uint32_t)kWaveSize : 1u, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
      if (whole) r = (uint32_t)__builtin_amdgcn_readfirstlane((int)r) + (uint32_t)lane;
      rank[j] = r;
    }
  }
  __syncthreads();
  static_assert(LocalBlock::kBlock == kRadix, "a thread scans the counts of one digit");
  digit_count = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) digit_count += counter[w * kRadix + t];
  uint32_t sum = digit_count;
#pragma unroll
  for (int s = 1; s < kWaveSize; s <<= 1) {
    const uint32_t o = shfl_up(sum, s);
    if (lane >= s) sum += o;
  }
  if (lane == kWaveSize - 1) lds.sums[wave] = sum;
  __syncthreads();
  uint32_t run = sum - digit_count;
  for (int w = 0; w < wave; ++w) run += lds.sums[w];
  digit_start = run;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const uint32_t c = counter[w * kRadix + t];
    counter[w * kRadix + t] = run;
    run += c;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < ITEMS; ++j)
    if (j < rows) rank[j] += mine[digit(j)];
  __syncthreads();  // the run starts have been read; the stage is free
}

// A window whose keys crowd a bin: `digits` digits of key - low, in LDS.
template <int KEY_BYTES, int VALUE_BYTES>
__device__ __attribute__((noinline)) void local_window_by_digits(
    const typename KeyOf<KEY_BYTES>::type* src, typename KeyOf<KEY_BYTES>::type* dst,
    const typename ValueOf<VALUE_BYTES>::type* src_vals, typename ValueOf<VALUE_BYTES>::type* dst_vals,
    uint32_t count, int below, uint64_t xor_mask, uint64_t reference_term, uint64_t total_term,
    __attribute__((address_space(3))) LocalLds* lds_in) {
  using K = typename KeyOf<KEY_BYTES>::type;
  using Val = typename ValueOf<VALUE_BYTES>::type;
  constexpr bool kPairs = VALUE_BYTES > 0;
  constexpr int kItems = local_items(KEY_BYTES, VALUE_BYTES);
  const KeyXform xf{xor_mask, reference_term, total_term};
  LocalLds& lds = *(LocalLds*)lds_in;
  const int t = threadIdx.x, lane = t & (kWaveSize - 1), wave = t / kWaveSize;
  const int rows = (int)((count + LocalBlock::kBlock - 1) / LocalBlock::kBlock);
  const uint32_t first_local = (uint32_t)(wave * rows * kWaveSize + lane);
  K* s_keys = reinterpret_cast<K*>(lds.stage);
  uint16_t* s_from = reinterpret_cast<uint16_t*>(lds.stage + local_window(KEY_BYTES, VALUE_BYTES) * KEY_BYTES);
  const K low = (K)((K)(ordered_bits(src[0], xf) >> below) << below);
  const K span = (K)((ordered_bits(src[count - 1], xf) | (K)((((K)1) << below) - 1)) - low);
  const int bits = KEY_BYTES == 8 ? 64 - __builtin_clzll((uint64_t)span) : 32 - __builtin_clz((uint32_t)span);
  K key[kItems];
  uint32_t from[kPairs ? kItems : 1];
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const uint32_t local = first_local + j * kWaveSize;
    key[j] = 0;
    if (j < rows && local < count) key[j] = (K)(ordered_bits(src[local], xf) - low);
    if constexpr (kPairs) from[j] = local;
  }
#pragma unroll 1
  for (int shift = 0; shift < bits; shift += 8) {
    uint32_t rank[kItems], digit_start, digit_count;
    local_rank<K, kItems>(key, rank, rows, first_local, count, shift, lds, digit_start, digit_count);
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      if (j < rows) {
        s_keys[rank[j]] = key[j];
        if constexpr (kPairs) s_from[rank[j]] = (uint16_t)from[j];
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      if (j < rows) {
        key[j] = s_keys[first_local + j * kWaveSize];
        if constexpr (kPairs) from[j] = s_from[first_local + j * kWaveSize];
      }
    }
  }
  // (Every key and value has been read before the first one is written: the window may be
  // sorted in place.)
  Val value[kPairs ? kItems : 1];
  if constexpr (kPairs) {
#pragma unroll
    for (int j = 0; j < kItems; ++j)
      if (j < rows && first_local + j * kWaveSize < count) value[j] = src_vals[from[j]];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const uint32_t local = first_local + j * kWaveSize;
    if (j < rows && local < count) {
      dst[local] = raw_bits((K)(key[j] + low), xf);
      if constexpr (kPairs) dst_vals[local] = value[j];
    }
  }
}

// A run longer than a window: by the block, through memory, one pass for each of its lower
// digits that differ between its keys.  (Of one digit there are none, of two the counts allow n / 256 keys and a
// window, or n / 4096 keys: local_counts_allow.  A run of 9300 keys takes 27 to 45 us more than short ones, of 50 000 u32 110 to
// 190, of 25 000 u64 250 to 330, copies of a key the most.)  `other` is scratch at the run's own place; the
// result ends in `result`, which is one of the two.
template <int KEY_BYTES, int VALUE_BYTES>
__device__ __attribute__((noinline)) void local_long_run(
    typename KeyOf<KEY_BYTES>::type* src, typename KeyOf<KEY_BYTES>::type* other,
    typename KeyOf<KEY_BYTES>::type* result, typename ValueOf<VALUE_BYTES>::type* src_vals,
    typename ValueOf<VALUE_BYTES>::type* other_vals, uint32_t total, int digits, uint64_t xor_mask,
    uint64_t reference_term, uint64_t total_term, __attribute__((address_space(3))) LocalLds* lds_in) {
  using K = typename KeyOf<KEY_BYTES>::type;
  using Val = typename ValueOf<VALUE_BYTES>::type;
  constexpr bool kPairs = VALUE_BYTES > 0;
  constexpr int kItems = local_items(KEY_BYTES, VALUE_BYTES);
  constexpr uint32_t kTile = (uint32_t)local_window(KEY_BYTES, VALUE_BYTES);
  const KeyXform xf{xor_mask, reference_term, total_term};
  LocalLds& lds = *(LocalLds*)lds_in;
  const int t = threadIdx.x, lane = t & (kWaveSize - 1), wave = t / kWaveSize;
  K* s_keys = reinterpret_cast<K*>(lds.stage);
  uint16_t* s_from = reinterpret_cast<uint16_t*>(lds.stage + kTile * KEY_BYTES);
  uint32_t* s_base = reinterpret_cast<uint32_t*>(lds.list);  // where a digit's next key of a tile goes, less its place there
  static_assert(sizeof(lds.list) >= kRadix * 4, "one word per digit");
#pragma unroll 1
  for (int d = 0; d < digits; ++d) {
    const int shift = 8 * d;
    __syncthreads();  // what the pass before wrote is there, and s_base has been read
    s_base[t] = 0u;
    __syncthreads();
    for (uint32_t tile = 0; tile < total; tile += kTile) {
      K key[kItems];
#pragma unroll
      for (int j = 0; j < kItems; ++j) {
        const uint32_t i = tile + j * LocalBlock::kBlock + t;
        key[j] = src[i < total ? i : total - 1];
      }
#pragma unroll
      for (int j = 0; j < kItems; ++j)
        if (tile + j * LocalBlock::kBlock + t < total)
          atomicAdd(&s_base[(uint32_t)(ordered_bits(key[j], xf) >> shift) & (kRadix - 1)], 1u);
    }
    __syncthreads();
    const uint32_t mine = s_base[t];
    if (t == 0) lds.listed = 0u;
    __syncthreads();
    if (mine == total) lds.listed = 1u;
    __syncthreads();
    if (lds.listed != 0u) continue;  // all keys share the digit
    uint32_t sum = mine;
#pragma unroll
    for (int s = 1; s < kWaveSize; s <<= 1) {
      const uint32_t o = shfl_up(sum, s);
      if (lane >= s) sum += o;
    }
    if (lane == kWaveSize - 1) lds.sums[wave] = sum;
    __syncthreads();
    uint32_t next = sum - mine;  // of digit t
    for (int w = 0; w < wave; ++w) next += lds.sums[w];
    for (uint32_t tile = 0; tile < total; tile += kTile) {
      const uint32_t count = total - tile < kTile ? total - tile : kTile;
      const int rows = (int)((count + LocalBlock::kBlock - 1) / LocalBlock::kBlock);
      const uint32_t first_local = (uint32_t)(wave * rows * kWaveSize + lane);
      K key[kItems];
      uint32_t rank[kItems], digit_start, digit_count;
#pragma unroll
      for (int j = 0; j < kItems; ++j) {
        const uint32_t local = first_local + j * kWaveSize;
        key[j] = 0;
        if (j < rows && local < count) key[j] = ordered_bits(src[tile + local], xf);
      }
      local_rank<K, kItems>(key, rank, rows, first_local, count, shift, lds, digit_start, digit_count);
      s_base[t] = next - digit_start;
      next += digit_count;
#pragma unroll
      for (int j = 0; j < kItems; ++j) {
        if (j < rows) {
          s_keys[rank[j]] = key[j];
          if constexpr (kPairs) s_from[rank[j]] = (uint16_t)(first_local + j * kWaveSize);
        }
      }
      __syncthreads();
#pragma unroll 4
      for (uint32_t i = t; i < count; i += LocalBlock::kBlock) {
        const K k = s_keys[i];
        const uint32_t to = s_base[(uint32_t)(k >> shift) & (kRadix - 1)] + i;
        other[to] = raw_bits(k, xf);
        if constexpr (kPairs) other_vals[to] = src_vals[tile + s_from[i]];
      }
      __syncthreads();
    }
    K* k = src; src = other; other = k;
    Val* v = src_vals; src_vals = other_vals; other_vals = v;
  }
  __syncthreads();
  if (src != result) {
    local_copy(src, other, total, 0u, 1u);
    if constexpr (kPairs) local_copy(src_vals, other_vals, total, 0u, 1u);
    __syncthreads();
  }
}

// ---- the kernel -------------------------------------------------------------------
// Rows of a window as a buffer: what lies behind its `count` elements is read as zero and not
// written.  (No scalar offset: it would not be part of what the hardware holds against the
// length.)
template <typename E>
struct LocalRows {
  E* base;
  uint32_t count;
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ LocalRows(const E* from, uint32_t elements)
      : base(const_cast<E*>(from)),
        count(elements),
        rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<E*>(from), 0, (int)(elements * (uint32_t)sizeof(E)),
                                               0x00027000)) {}
  __device__ __forceinline__ E load(int row, uint32_t t) const {
    const int at = (int)((t + (uint32_t)(row * LocalBlock::kBlock)) * (uint32_t)sizeof(E));
    if constexpr (sizeof(E) == 1) return (E)__builtin_amdgcn_raw_buffer_load_b8(rsrc, at, 0, 0);
    else if constexpr (sizeof(E) == 2) return (E)__builtin_amdgcn_raw_buffer_load_b16(rsrc, at, 0, 0);
    else if constexpr (sizeof(E) == 4) return (E)__builtin_amdgcn_raw_buffer_load_b32(rsrc, at, 0, 0);
    else return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b64(rsrc, at, 0, 0));
  }
  __device__ __forceinline__ void store(E e, int row, uint32_t t) const {
    const int at = (int)((t + (uint32_t)(row * LocalBlock::kBlock)) * (uint32_t)sizeof(E));
    typedef uint32_t Two __attribute__((ext_vector_type(2)));
    if constexpr (sizeof(E) == 1) __builtin_amdgcn_raw_buffer_store_b8(e, rsrc, at, 0, 0);
    else if constexpr (sizeof(E) == 2) __builtin_amdgcn_raw_buffer_store_b16(e, rsrc, at, 0, 0);
    else if constexpr (sizeof(E) == 4) __builtin_amdgcn_raw_buffer_store_b32(e, rsrc, at, 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(Two, e), rsrc, at, 0, 0);
  }
  // Rows `row` to row + N - 1, which lie whole within the buffer: N neighbouring elements per
  // thread, in one store of up to 16 bytes (aligned to an element).
  template <int N>
  __device__ __forceinline__ void store_whole(const E (&in)[N], int row, uint32_t t) const {
    struct alignas(sizeof(E)) Pack { E e[N]; } p;
#pragma unroll
    for (int e = 0; e < N; ++e) p.e[e] = in[e];
    *reinterpret_cast<Pack*>(reinterpret_cast<char*>(base + row * LocalBlock::kBlock) +
                             t * (uint32_t)(N * sizeof(E))) = p;
  }
};

template <int KEY_BYTES, int VALUE_BYTES, bool FLOAT_KEYS>
__global__ __launch_bounds__(LocalBlock::kBlock, 4) ILGPU_HIP_SORT_CODE_ALIGNED void local_sort_kernel(
    typename KeyOf<KEY_BYTES>::type* keys_a, typename KeyOf<KEY_BYTES>::type* keys_b,
    typename ValueOf<VALUE_BYTES>::type* vals_a, typename ValueOf<VALUE_BYTES>::type* vals_b, uint32_t n,
    KeyXform xf, const SortPlan* __restrict__ plan, const uint32_t* __restrict__ excl, int values_from_index,
    int finishes, uint2* deferred) {
  using K = typename KeyOf<KEY_BYTES>::type;
  using Val = typename ValueOf<VALUE_BYTES>::type;
  constexpr bool kPairs = VALUE_BYTES > 0;
  constexpr int kBlock = LocalBlock::kBlock;
  constexpr int kWaves = LocalBlock::kWaves;
  constexpr int kItems = local_items(KEY_BYTES, VALUE_BYTES);
  constexpr int kPack = kItems % 4 == 0 ? 4 : 2;  // keys that a thread writes at once
  constexpr uint32_t kWindow = (uint32_t)local_window(KEY_BYTES, VALUE_BYTES);
  static_assert(kWindow <= 65536, "places are packed two to a register");
  static_assert(kItems % kPack == 0 && kItems % 2 == 0, "a thread's keys are whole vectors");
  static_assert(kItems <= 64, "a bit for every place of a thread");
  __shared__ LocalLds lds;

  const int below = 8 * (int)plan->local_from;
  if (below == 0) {  // every digit was sorted
    if (finishes && plan->final_in_alt != 0) {
      local_copy(keys_b, keys_a, n, blockIdx.x, gridDim.x);
      if constexpr (kPairs) local_copy(vals_b, vals_a, n, blockIdx.x, gridDim.x);
    } else if (finishes && kPairs && values_from_index && plan->executed == 0) {
      if constexpr (kPairs)
        for (uint64_t i = blockIdx.x * (uint32_t)kBlock + threadIdx.x; i < n; i += gridDim.x * (uint32_t)kBlock)
          vals_a[i] = index_value<VALUE_BYTES>((int64_t)i, values_from_index);
    }
    return;
  }
  const bool in_b = plan->final_in_alt != 0;
  K* src = in_b ? keys_b : keys_a;
  Val* src_vals = in_b ? vals_b : vals_a;
  const int tid = threadIdx.x;
  const int lane = tid & (kWaveSize - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWaveSize);
  // Float keys are held in their ordered form, others as they are: their order is one xor.
  auto held = [&](K k) -> K {
    if constexpr (FLOAT_KEYS) return ordered_bits(k, xf);
    else return k;
  };
  auto ordered = [&](K k) -> K {  // of a key as it is held
    if constexpr (FLOAT_KEYS) return k;
    else return (K)(k ^ (K)xf.xor_mask);
  };
  // The runs that start in this block's part.
  const uint32_t part = (n + gridDim.x - 1) / gridDim.x;
  if (wave < 2) {
    const uint64_t x = (uint64_t)(blockIdx.x + (uint32_t)wave) * part;
    const uint32_t from = x < n ? (uint32_t)x : n;
    const uint32_t start = plan->executed == 1u
                               ? local_digit_start(excl + plan->last_executed * kRadix, from, n, lane)
                               : local_run_start(src, from, n, xf, below, lane);
    if (lane == 0) lds.bounds[wave] = start;
  }
  if (tid == 0) lds.deferred = 0u;
  deferred += (size_t)blockIdx.x * local_deferred(part, kWindow);
  __syncthreads();
  uint32_t cur = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds.bounds[0]);
  const uint32_t end = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds.bounds[1]);
  K* s_keys = reinterpret_cast<K*>(lds.stage);
  uint16_t* s_from = reinterpret_cast<uint16_t*>(lds.stage + kWindow * KEY_BYTES);
  char* s_words = reinterpret_cast<char*>(lds.stage);
  // The thread index is made opaque for every phase of a window: otherwise the rows' addresses and
  // the masks of their lanes are kept in registers from one phase to the next.
  auto opaque = [&]() -> uint32_t {
    uint32_t t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
  };
  K key[kItems];
  K first = 0, last = 0;
  uint32_t avail = 0;
  // The keys from `cur` on, as many as a window holds.
  auto request = [&]() {
    avail = cur < end ? (end - cur < kWindow ? end - cur : kWindow) : 0u;
    const uint32_t t = opaque();
    const LocalRows<K> in(src + cur, avail);
#pragma unroll
    for (int j = 0; j < kItems; ++j) key[j] = in.load(j, t);
    if (avail != 0) {
      first = src[cur];
      last = src[cur + avail - 1];
    }
  };
  request();

  while (cur < end) {
    {
      uint4* z = reinterpret_cast<uint4*>(lds.stage);
#pragma unroll
      for (int i = 0; i < LocalBlock::kStageBytes / 16 / kBlock; ++i) z[i * kBlock + tid] = make_uint4(0u, 0u, 0u, 0u);
      if (tid == 0) lds.listed = 0u;
    }
    if constexpr (FLOAT_KEYS) {
#pragma unroll
      for (int j = 0; j < kItems; ++j) key[j] = held(key[j]);
    }
    const K first_ordered = ordered(held(first)), last_ordered = ordered(held(last));
    // The last run may go on behind the window: it is left for the next one.
    const K upper_last = (K)((K)(last_ordered >> below) << below);
    const bool cut = cur + avail < end;
    if (cut) {
      uint32_t in_front = 0;
#pragma unroll
      for (int j = 0; j < kItems; ++j) in_front += (uint32_t)__popcll(__ballot(ordered(key[j]) < upper_last));
      if (lane == 0) lds.sums[wave] = in_front;
    }
    __syncthreads();
    uint32_t count = avail;
    const K low = (K)((K)(first_ordered >> below) << below);
    K span = (K)((last_ordered | (K)((((K)1) << below) - 1)) - low);  // of key - low, inclusive
    if (cut) {
      count = 0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) count += lds.sums[w];
      count = (uint32_t)__builtin_amdgcn_readfirstlane((int)count);
      span = (K)(upper_last - low - 1);
    }
    const LocalScale bins_of_span = local_scale<K>(span);
    const int shift = bins_of_span.shift;
    const uint32_t scale = bins_of_span.scale;
    K minus_low = (K)(0 - low);
    if constexpr (sizeof(K) == 4) asm("" : "+v"(minus_low));  // (xor and sum in one instruction)
    auto scaled = [&](K k) -> uint32_t {  // of a key as it is held: its bin in the upper half, 15 bits
      return (uint32_t)__umul24((uint32_t)((K)(ordered(k) + minus_low) >> shift), scale);  // (it returns an int)
    };
    auto bin_of = [&](K k) -> uint32_t { return scaled(k) >> 16; };
    auto codes_of = [&](K k0, K k1) -> uint32_t {  // of two keys
      typedef uint16_t Two __attribute__((ext_vector_type(2)));
      const Two bins = __builtin_bit_cast(Two, __builtin_amdgcn_perm(scaled(k1), scaled(k0), 0x07060302u));
      return __builtin_bit_cast(uint32_t, local_bin_codes(bins));
    };
    auto word_at = [&](uint32_t codes, int which) -> uint32_t* {
      return reinterpret_cast<uint32_t*>(s_words + ((which == 0 ? codes & 0xFFFFu : codes >> 16) & ~3u));
    };
    auto count_at = [&](uint32_t codes, int which) -> uint32_t {  // the bit its count begins at
      return (which == 0 ? codes << 2 : codes >> 14) & 12u;
    };
    constexpr int kRanks = (kItems + 7) / 8;
    uint32_t ranks[kRanks];      // 4 bits each: keys that were in the bin before
    uint32_t place[kItems / 2];  // 16 bits each: the code, then the key's place
#pragma unroll
    for (int q = 0; q < kRanks; ++q) ranks[q] = 0u;
#pragma unroll
    for (int q = 0; q < kItems / 2; ++q) place[q] = 0u;
    // Rows in groups, whose LDS operations are in flight together; the masks of the lanes only
    // where a group is not full of keys.
    constexpr int kGroup = 4;
    {
      const uint32_t t = opaque();
      auto count_group = [&](auto full, int j0) {
        uint32_t old[kGroup];
#pragma unroll
        for (int g = 0; g < kGroup && j0 + g < kItems; ++g) {
          const int j = j0 + g;
          if (g % 2 == 0) place[j / 2] = codes_of(key[j], key[j + 1]);
          old[g] = 0;
          if (decltype(full)::value || (int)t < (int)count - j * kBlock)
            old[g] = __hip_atomic_fetch_add(word_at(place[j / 2], j % 2), 1u << count_at(place[j / 2], j % 2),
                                            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
#pragma unroll
        for (int g = 0; g < kGroup && j0 + g < kItems; ++g) {
          const int j = j0 + g;
          ranks[j / 8] |= __builtin_amdgcn_ubfe(old[g], count_at(place[j / 2], j % 2), 4u) << (4 * (j % 8));
          if (!decltype(full)::value && (int)t >= (int)count - j * kBlock)
            place[j / 2] = local_codes_without(place[j / 2], j % 2);
        }
      };
#pragma unroll
      for (int j0 = 0; j0 < kItems; j0 += kGroup) {
        const int end_of_group = (j0 + kGroup < kItems ? j0 + kGroup : kItems) * kBlock;
        if ((int)count >= end_of_group) count_group(std::true_type{}, j0);
        else if ((int)count > j0 * kBlock) count_group(std::false_type{}, j0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int q = 0; q < kRanks; ++q) asm volatile("" : "+v"(ranks[q]));
#pragma unroll
    for (int q = 0; q < kItems / 2; ++q) asm volatile("" : "+v"(place[q]));
    __syncthreads();
    // Places of the words: 32 per thread, read twice (held in registers they make the keys spill).
    uint4* row = reinterpret_cast<uint4*>(lds.stage + opaque() * (LocalBlock::kRowStride * 4));
    uint32_t sum = 0;
#pragma unroll
    for (int q = 0; q < LocalBlock::kRowWords / 4; ++q) {
      const uint4 w = row[q];
      sum = __builtin_amdgcn_udot8(w.x, 0x1111u, sum, false);
      sum = __builtin_amdgcn_udot8(w.y, 0x1111u, sum, false);
      sum = __builtin_amdgcn_udot8(w.z, 0x1111u, sum, false);
      sum = __builtin_amdgcn_udot8(w.w, 0x1111u, sum, false);
    }
    uint32_t before = sum;
#pragma unroll
    for (int s = 1; s < kWaveSize; s <<= 1) {
      const uint32_t o = shfl_up(before, s);
      if (lane >= s) before += o;
    }
    if (lane == kWaveSize - 1) lds.sums[wave] = before;
    __syncthreads();
    before -= sum;
    uint32_t total = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const uint32_t of_wave = lds.sums[w];
      if (w < wave) before += of_wave;
      total += of_wave;
    }
    // A count that ran over, sixteen keys in a bin, has lost fifteen or sixteen of them, and none
    // gains any.
    bool crowded = (uint32_t)__builtin_amdgcn_readfirstlane((int)total) != count;
    const bool long_run = count == 0;  // one run, and longer than a window
    uint32_t listed = 0;
    if (!crowded && !long_run) {
#pragma unroll
      for (int q = 0; q < LocalBlock::kRowWords / 4; ++q) {
        uint4 w = row[q];
        uint32_t next = __builtin_amdgcn_udot8(w.x, 0x1111u, before, false);
        w.x |= before << 16;
        before = __builtin_amdgcn_udot8(w.y, 0x1111u, next, false);
        w.y |= next << 16;
        next = __builtin_amdgcn_udot8(w.z, 0x1111u, before, false);
        w.z |= before << 16;
        before = __builtin_amdgcn_udot8(w.w, 0x1111u, next, false);
        w.w |= next << 16;
        row[q] = w;
        if (q % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
      auto place_group = [&](int j0) {
        uint32_t w[kGroup], r[kGroup], to[kGroup];
#pragma unroll
        for (int g = 0; g < kGroup && j0 + g < kItems; ++g) {
          const int j = j0 + g;
          r[g] = __builtin_amdgcn_ubfe(ranks[j / 8], 4 * (j % 8), 4u);
          w[g] = *word_at(place[j / 2], j % 2);  // (of the first bin where there is no key)
        }
        uint32_t seconds = 0;
#pragma unroll
        for (int g = 0; g < kGroup && j0 + g < kItems; ++g) {
          const int j = j0 + g;
          const uint32_t lower = __builtin_amdgcn_ubfe(w[g], 0u, count_at(place[j / 2], j % 2));
          to[g] = __builtin_amdgcn_udot8(lower, 0x1111u, (w[g] >> 16) + r[g], false);
          if (g % 2 == 1) place[j / 2] = to[g - 1] | to[g] << 16;
          seconds += (uint32_t)__popcll(__ballot(r[g] == 1u));
        }
        // The second key of a bin lists it.  (Room for the group is taken at once: by and large the
        // second keys are those of the block's last wave.)
        uint32_t slot = 0;
        if (lane == 0) slot = atomicAdd(&lds.listed, seconds);
        slot = (uint32_t)__builtin_amdgcn_readfirstlane((int)slot);
        if (slot + seconds <= (uint32_t)LocalBlock::kList) {
#pragma unroll
          for (int g = 0; g < kGroup && j0 + g < kItems; ++g) {
            const uint64_t second = __ballot(r[g] == 1u);
            if (r[g] == 1u)
              lds.list[__builtin_amdgcn_mbcnt_hi((uint32_t)(second >> 32),
                                                 __builtin_amdgcn_mbcnt_lo((uint32_t)second, slot))] =
                  (uint16_t)(to[g] - 1u);
            slot += (uint32_t)__popcll(second);
          }
        }
      };
#pragma unroll
      for (int j0 = 0; j0 < kItems; j0 += kGroup) {
        if ((int)count > j0 * kBlock) place_group(j0);
#pragma unroll
        for (int g = 0; g < kGroup && j0 + g < kItems; g += 2) asm volatile("" : "+v"(place[(j0 + g) / 2]));
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
      listed = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds.listed);
      {
        const uint32_t t = opaque();
        auto stage_group = [&](auto full, int j0) {
#pragma unroll
          for (int g = 0; g < kGroup && j0 + g < kItems; ++g) {
            const int j = j0 + g;
            if (decltype(full)::value || (int)t < (int)count - j * kBlock) {
              const uint32_t to = j % 2 == 0 ? place[j / 2] & 0xFFFFu : place[j / 2] >> 16;
              s_keys[to] = key[j];
              if constexpr (kPairs) s_from[to] = (uint16_t)(j * kBlock + t);
            }
          }
        };
#pragma unroll
        for (int j0 = 0; j0 < kItems; j0 += kGroup) {
          const int end_of_group = (j0 + kGroup < kItems ? j0 + kGroup : kItems) * kBlock;
          if ((int)count >= end_of_group) stage_group(std::true_type{}, j0);
          else if ((int)count > j0 * kBlock) stage_group(std::false_type{}, j0);
        }
      }
    }
    if (crowded || long_run) {
      __syncthreads();  // everybody has seen it
      if (wave == 0) {
        const uint32_t behind = long_run ? local_run_start(src, cur + avail, n, xf, below, lane) : cur + count;
        if (lane == 0) {
          lds.bounds[0] = behind - cur;
          deferred[lds.deferred++] = make_uint2(cur, behind - cur);
        }
      }
      __syncthreads();
      count = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds.bounds[0]);
    }
    // The next window's keys are on their way while this one is finished.
    const uint32_t at_window = cur;
    cur += count;
    request();
    if (crowded || long_run) continue;
    {
      {
        __syncthreads();
        // Bins of two keys or more.  Where the list has run over (from some half a copy of every key on) those with a
        // key in front of a smaller one (equal keys: of an earlier one): at the first such place of a bin, and
        // all of them are found before any key moves.
        const bool all_listed = listed <= (uint32_t)LocalBlock::kList;
        uint64_t found = 0;  // bit j: place_of(j)
        auto place_of = [&](uint32_t j) -> uint32_t {  // a thread looks at packs of neighbours, as it writes them
          return j / kPack * (kBlock * kPack) + (uint32_t)tid * kPack + j % kPack;
        };
        if (__builtin_expect(!all_listed, 0)) {
          auto inverted = [&](K k0, K k1, uint32_t f0, uint32_t f1) -> bool {  // neighbours
            return ordered(k1) < ordered(k0) || (kPairs && k1 == k0 && f1 < f0);
          };
#pragma unroll 1
          for (int j = 0; j < kItems && j * kBlock < (int)count; j += kPack) {
            const uint32_t at = place_of(j);
            K k[kPack + 1];
            uint32_t f[kPack + 1];
#pragma unroll
            for (int e = 0; e <= kPack; ++e) {
              const uint32_t from = e < kPack || at + kPack < kWindow ? at + e : at;
              k[e] = s_keys[from];
              f[e] = 0;
              if constexpr (kPairs) f[e] = s_from[from];
            }
#pragma unroll
            for (int e = 0; e < kPack; ++e)
              if (at + e + 1 < count && inverted(k[e], k[e + 1], f[e], f[e + 1])) found |= 1ull << (j + e);
          }
          for (uint64_t left = found; left != 0; left &= left - 1) {
            const uint32_t j = (uint32_t)__builtin_ctzll(left);
            const uint32_t at = place_of(j);
            K k = s_keys[at];
            const uint32_t bin = bin_of(k);
            for (uint32_t p = at; p > 0; --p) {
              const K in_front = s_keys[p - 1];
              if (bin_of(in_front) != bin) break;
              uint32_t f0 = 0, f1 = 0;
              if constexpr (kPairs) {
                f0 = s_from[p - 1];
                f1 = s_from[p];
              }
              if (inverted(in_front, k, f0, f1)) {
                found &= ~(1ull << j);
                break;
              }
              k = in_front;
            }
          }
          __syncthreads();
        }
        // Insertion from place i on, for the few that hold three or more.  (It ends at the keys of the bin before, which
        // are smaller.)
        auto insert_from = [&](uint32_t i, uint32_t bin) {
          for (; i < count; ++i) {
            const K k = s_keys[i];
            if (bin_of(k) != bin) break;
            uint32_t f = 0;
            if constexpr (kPairs) f = s_from[i];
            uint32_t to = i;
            while (to > 0) {
              const K p = s_keys[to - 1];
              bool behind = ordered(p) > ordered(k);
              if constexpr (kPairs) behind = behind || (p == k && s_from[to - 1] > f);
              if (!behind) break;
              s_keys[to] = p;
              if constexpr (kPairs) s_from[to] = s_from[to - 1];
              --to;
            }
            if (to != i) {
              s_keys[to] = k;
              if constexpr (kPairs) s_from[to] = (uint16_t)f;
            }
          }
        };
        if (__builtin_expect(!all_listed, 0)) {
          while (found != 0) {
            const uint32_t at = place_of((uint32_t)__builtin_ctzll(found));
            found &= found - 1;
            insert_from(at + 1, bin_of(s_keys[at]));
          }
        } else {
          for (uint32_t e = tid; e < listed; e += kBlock) {
            const uint32_t at = lds.list[e];
            const K k0 = s_keys[at], k1 = s_keys[at + 1];
            uint32_t f0 = 0, f1 = 0;
            if constexpr (kPairs) {
              f0 = s_from[at];
              f1 = s_from[at + 1];
            }
            const uint32_t bin = bin_of(k0);
            bool swap = ordered(k1) < ordered(k0);
            if constexpr (kPairs) swap = swap || (k1 == k0 && f1 < f0);
            if (swap) {
              s_keys[at] = k1;
              s_keys[at + 1] = k0;
              if constexpr (kPairs) {
                s_from[at] = (uint16_t)f1;
                s_from[at + 1] = (uint16_t)f0;
              }
            }
            insert_from(at + 2, bin);
          }
        }
        __syncthreads();
        {
          const uint32_t t = opaque();
          const LocalRows<K> out(keys_a + at_window, count);
          auto final_bits = [&](K k) -> K {
            if constexpr (FLOAT_KEYS) return raw_bits(k, xf);
            else return k;
          };
#pragma unroll
          for (int j = 0; j < kItems; j += kPack) {
            if ((int)count >= (j + kPack) * kBlock) {
              K k[kPack];
#pragma unroll
              for (int e = 0; e < kPack; ++e) k[e] = final_bits(s_keys[j * kBlock + t * kPack + e]);
              out.store_whole(k, j, t);
            } else if ((int)count > j * kBlock) {
#pragma unroll
              for (int e = 0; e < kPack; ++e) out.store(final_bits(s_keys[(j + e) * kBlock + t]), j + e, t);
            }
          }
        }
        if constexpr (kPairs) {
          // The values take the keys' place in LDS, in their own order, and are read in the keys'.
          constexpr int kRoundRows = kItems * KEY_BYTES / VALUE_BYTES < kItems ? kItems * KEY_BYTES / VALUE_BYTES
                                                                               : kItems;
          Val* s_vals = reinterpret_cast<Val*>(lds.stage);
          const LocalRows<Val> in_vals(src_vals + at_window, count), out_vals(vals_a + at_window, count);
          Val moved[kItems];
          const uint32_t t = opaque();
#pragma unroll
          for (int base = 0; base < kItems; base += kRoundRows) {
            Val value[kRoundRows];
#pragma unroll
            for (int j = 0; j < kRoundRows; ++j) value[j] = in_vals.load(base + j, t);
            __syncthreads();
#pragma unroll
            for (int j = 0; j < kRoundRows; ++j)
              if (base + j < kItems) s_vals[j * kBlock + t] = value[j];
            __syncthreads();
#pragma unroll
            for (int j = 0; j < kItems; ++j) {
              if ((int)t < (int)count - j * kBlock) {
                const uint32_t at = (uint32_t)s_from[j * kBlock + t] - (uint32_t)(base * kBlock);
                if (kRoundRows == kItems || at < (uint32_t)(kRoundRows * kBlock)) moved[j] = s_vals[at];
              }
            }
          }
#pragma unroll
          for (int j = 0; j < kItems; ++j) out_vals.store(moved[j], j, t);
        }
        __syncthreads();  // the stage has been read
      }
    }
  }

  // What had to wait.  (In a loop of its own: with the calls in the loop above its registers
  // spill.)
  __syncthreads();
  const uint32_t waiting = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds.deferred);
  for (uint32_t i = 0; i < waiting; ++i) {
    const uint32_t at = (uint32_t)__builtin_amdgcn_readfirstlane((int)deferred[i].x);
    const uint32_t count = (uint32_t)__builtin_amdgcn_readfirstlane((int)deferred[i].y);
    auto* lds_block = (__attribute__((address_space(3))) LocalLds*)&lds;
    K* other = in_b ? keys_a : keys_b;
    Val* other_vals = in_b ? vals_a : vals_b;
    if (count <= kWindow)
      local_window_by_digits<KEY_BYTES, VALUE_BYTES>(src + at, keys_a + at, kPairs ? src_vals + at : nullptr,
                                                     kPairs ? vals_a + at : nullptr, count, below, xf.xor_mask,
                                                     xf.reference_term, xf.total_term, lds_block);
    else
      local_long_run<KEY_BYTES, VALUE_BYTES>(src + at, other + at, keys_a + at, kPairs ? src_vals + at : nullptr,
                                             kPairs ? other_vals + at : nullptr, count, below / 8, xf.xor_mask,
                                             xf.reference_term, xf.total_term, lds_block);
  }
}
