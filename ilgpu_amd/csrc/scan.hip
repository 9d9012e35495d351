// Inclusive / exclusive scan, single pass with decoupled look-back.
//
// Stands in for the Scan delegates of ScanExtensions.cs:930-959.  The
// reference's single-pass kernel (ScanExtensions.cs:530-597) chains the groups
// strictly through one global word (SequentialGroupExecutor.cs:58-77) and reads
// the input twice; here each tile publishes its aggregate as soon as it has
// it, and a tile's first wave resolves the prefix of up to 64 predecessor
// tiles per step, so tiles only wait for data, never for their turn.
//
// Tile layout (kBlock = 512 threads, 8 waves, kVecs = 16 16-byte vectors per
// lane, i.e. 128 KiB per tile: time per launch falls with the number of tiles
// until about this size, then register pressure takes over; inputs of two to 192 such
// tiles, or of a quarter of one, take short ones of 32 KiB):
//   wave w owns a contiguous chunk of kVecs*64 vectors; vector j of lane l is
//   chunk[j*64 + l], so every load/store instruction of a wave covers 1 KiB of
//   consecutive addresses (dwordx4 per lane).  Scan order inside a wave is
//   (j, lane, element): each lane scans its vector, the wave scans the vector
//   totals once per j, and the running totals of earlier j are folded in.
//
// Block b takes tile b.  Blocks start in index order in practice, but nothing promises that a tile's
// predecessors run, so nobody waits without bound: after as many polls as a pass of the sort makes a
// missing tile is folded from the input (resolve_prefix).  Where the output overlaps the input, which may be
// overwritten by then, tile ids come from a global ticket instead, and a tile's predecessors have always
// started; a ticket costs a tile a round trip before its loads and 12 to 18 ns behind the ticket before
// (calls, us, over the input, with tickets / into another view: 2^23 int64 32.2 / 23.1, 2^22 18.8 / 15.0, 2^23 int32
// 17.4 / 14.1, 10^6 double Max 13.2 / 11.2, 2^28 int32 354.6 / 347.4).  Status words are read and written with agent-scope atomics: the
// eight XCDs of the device have separate L2s.
//   4-byte T: one 64-bit word {flag, value} per tile;
//   8-byte T: two such words per tile, one per half of the value.
// Each tile's words sit in a 128-byte line of their own, or in a quarter of one
// where the tiles are short (kShortDivisor).
//
// Algorithmic HBM traffic: 2 * n * sizeof(T) bytes (status: 128 B/tile, 32 B/short tile).
#include <algorithm>
#include <atomic>
#include <mutex>

#include "kernels.hpp"

namespace ilgpu_hip {

namespace {

#ifndef ILGPU_HIP_SCAN_BLOCK
#define ILGPU_HIP_SCAN_BLOCK 512
#endif
#ifndef ILGPU_HIP_SCAN_VECS
#define ILGPU_HIP_SCAN_VECS 16
#endif
#ifndef ILGPU_HIP_SCAN_WAVES_PER_EU
#define ILGPU_HIP_SCAN_WAVES_PER_EU 4
#endif
#ifndef ILGPU_HIP_SCAN_NT_LOAD
#define ILGPU_HIP_SCAN_NT_LOAD 1
#endif
#ifndef ILGPU_HIP_SCAN_NT_STORE
#define ILGPU_HIP_SCAN_NT_STORE 1
#endif
// Measurement only: 1 takes every tile's prefix as the identity (wrong results
// beyond the first tile) to time the kernel without its look-back.
#ifndef ILGPU_HIP_SCAN_PROBE_NO_LOOKBACK
#define ILGPU_HIP_SCAN_PROBE_NO_LOOKBACK 0
#endif
// 1 issues the loads of a tile's second half only after the first half has
// been scanned (half as many bytes in flight per wave).
#ifndef ILGPU_HIP_SCAN_LOAD_HALVES
#define ILGPU_HIP_SCAN_LOAD_HALVES 0
#endif
// 8-byte status words per tile: one 128-byte line each.  Every resident block
// polls the words of the few dozen tiles before it with loads that go past the
// L2; packed eight bytes apart those words share a handful of lines, and the
// memory channels that hold them fall behind on the data streams (measured at
// 2^28 int32: 0.384 ms packed, 0.363 at 64 bytes per tile, 0.360 at 128 to 512).
constexpr int kStatusStride = 16;
constexpr int64_t kStatusBytes = 8 * kStatusStride;
constexpr int kBlock = ILGPU_HIP_SCAN_BLOCK;
constexpr int kWaves = kBlock / kWaveSize;
constexpr int kVecs = ILGPU_HIP_SCAN_VECS;
#ifndef ILGPU_HIP_SCAN_VECS8
#define ILGPU_HIP_SCAN_VECS8 16
#endif
// 16-byte vectors per thread and tile, by element size (the same 128 KiB tile
// for both: measured at 2^27 int64 in the register-lean form, 10 vectors
// 0.456 ms, 12: 0.401, 14: 0.394, 16: 0.382, 18 and 20 the same as 16 for Add
// but 0.48 and 0.54 for the floating-point Max, which then spills).
template <typename T> constexpr int scan_vecs() {
  return sizeof(T) == 8 ? ILGPU_HIP_SCAN_VECS8 : kVecs;
}
constexpr uint32_t kNoLimit = ~0u;  // of polls
constexpr uint32_t kFlagInvalid = 0, kFlagAggregate = 1, kFlagPrefix = 2;
constexpr int64_t kHeaderBytes = 256;  // ticket counter, padded

template <typename T> constexpr int tile_elems() {
  return kBlock * scan_vecs<T>() * Vec16<T>::N;
}
// Short tiles, a quarter as long: an input of a few dozen full tiles leaves most
// compute units idle, and the scan lasts as long as one tile takes from its
// loads to its stores.  Inputs of two to kShortMaxTiles full tiles take them, or to
// kShortMaxTilesTicketed where the tiles are handed out by tickets, one after the other (12 to 18 ns each).
// Their status words stand a quarter of a line apart, so that they fit the
// temp view of the full tiles; that few words are not what such an input waits for.
// So does an input of one short tile, which is one launch like one full tile, with a quarter of its rows (calls, us,
// full / short: 1000 and 4000 double Max 12.3 and 12.3 / 7.1 and 7.1); between one short tile and one full one the launch that
// clears the status words costs more than the short tiles save (16384 int64 7.4 / 10.0).
// (Calls, us, full tiles / short ones: 2^21 double Max 18.4 / 12.8, 3 * 10^6 18.6 / 14.9, 2.5 * 10^6 int32 10.9 / 9.4,
// 6.3 * 10^6 12.0 / 11.9, 2^21 int64 12.3 / 10.3, 3 * 10^6 12.6 / 12.1, but 3.5 * 10^6, 214 full tiles, 13.3 / 18.4, double Max
// 18.7 / 22.3, and 2^22 int64 14.6 / 21.1.  With tickets, which come one after the other, 2^21 int64 13.0.
// Tiles an eighth as long: 10^6 double Max 12.3 against 11.1, 2^21 int64 16.1 against 10.6.)
#ifndef ILGPU_HIP_SCAN_SHORT_DIVISOR
#define ILGPU_HIP_SCAN_SHORT_DIVISOR 4
#endif
#ifndef ILGPU_HIP_SCAN_SHORT_MAX_TILES
#define ILGPU_HIP_SCAN_SHORT_MAX_TILES 192
#endif
constexpr int kShortDivisor = ILGPU_HIP_SCAN_SHORT_DIVISOR;
constexpr int64_t kShortMaxTiles = ILGPU_HIP_SCAN_SHORT_MAX_TILES;
constexpr int64_t kShortMaxTilesTicketed = 64;
static_assert(kStatusStride / kShortDivisor >= 2, "two status words per tile of 8-byte elements");
// Status words per tile of VECS vectors per thread.
template <typename T, int VECS> constexpr int status_stride() {
  return VECS == scan_vecs<T>() ? kStatusStride : kStatusStride / kShortDivisor;
}

template <typename T> struct Bits;
template <> struct Bits<int32_t> { using type = uint32_t; };
template <> struct Bits<uint32_t> { using type = uint32_t; };
template <> struct Bits<float> { using type = uint32_t; };
template <> struct Bits<int64_t> { using type = uint64_t; };
template <> struct Bits<uint64_t> { using type = uint64_t; };
template <> struct Bits<double> { using type = uint64_t; };

template <typename T>
__device__ __forceinline__ typename Bits<T>::type to_bits(T v) {
  typename Bits<T>::type b;
  __builtin_memcpy(&b, &v, sizeof(T));
  return b;
}
template <typename T>
__device__ __forceinline__ T from_bits(typename Bits<T>::type b) {
  T v;
  __builtin_memcpy(&v, &b, sizeof(T));
  return v;
}

// Look-back state in temp memory; STRIDE words from one tile's to the next one's.
// (A constant: as a member of the structure it cost unique_kernel<uint32_t> two
// vector registers and four more spilled scalar ones, 1 % of a call on 2^26 keys.)
template <typename T, int STRIDE = kStatusStride, int SIZE = sizeof(T)> struct TileState;

template <typename T, int STRIDE> struct TileState<T, STRIDE, 4> {
  uint64_t* words;
  __device__ __forceinline__ void publish(int tile, uint32_t flag, T v) const {
    const uint64_t w = ((uint64_t)flag << 32) | to_bits(v);
    __hip_atomic_store(&words[(int64_t)tile * STRIDE], w, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  }
  // What the tile has published: its flag, and the value unless that is kFlagInvalid.
  __device__ __forceinline__ uint32_t read(int tile, T* v) const {
    const uint64_t w = __hip_atomic_load(&words[(int64_t)tile * STRIDE], __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t flag = (uint32_t)(w >> 32);
    if (flag != kFlagInvalid) *v = from_bits<T>((uint32_t)w);
    return flag;
  }
};

// 8-byte values: two 64-bit words in the tile's line, {flag, low half} and
// {flag, high half}, each written and read with one relaxed atomic.  A tile writes each
// state (aggregate, then prefix) once, so two words with the same flag hold
// the halves of the same value; to a reader that catches the words in different
// states nothing has been published yet.  No fences: an agent-scope release would write back the
// whole L2 of the XCD for every tile.
template <typename T, int STRIDE> struct TileState<T, STRIDE, 8> {
  uint64_t* words;
  __device__ __forceinline__ void publish(int tile, uint32_t flag, T v) const {
    const uint64_t bits = to_bits(v);
    uint64_t* w = &words[(int64_t)tile * STRIDE];
    __hip_atomic_store(&w[0], ((uint64_t)flag << 32) | (uint32_t)bits,
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&w[1], ((uint64_t)flag << 32) | (bits >> 32),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __device__ __forceinline__ uint32_t read(int tile, T* v) const {
    const uint64_t* w = &words[(int64_t)tile * STRIDE];
    const uint64_t lo = __hip_atomic_load(&w[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint64_t hi = __hip_atomic_load(&w[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((uint32_t)(lo >> 32) == kFlagInvalid || (lo >> 32) != (hi >> 32)) return kFlagInvalid;
    *v = from_bits<T>((uint64_t)(uint32_t)lo | (hi << 32));
    return (uint32_t)(lo >> 32);
  }
};

// Data-parallel-primitive move: lane i receives `v` of the lane that the
// control word CTRL names (row_shr:n = 0x110 + n within rows of 16 lanes,
// row_bcast:15 = 0x142, row_bcast:31 = 0x143, wave_shr:1 = 0x138); lanes
// without a source, and rows outside ROW_MASK, receive `fill`.
template <typename T, int CTRL, int ROW_MASK>
__device__ __forceinline__ T dpp_move(T fill, T v) {
  if constexpr (sizeof(T) == 8) {
    union { T t; int32_t w[2]; } f, a, b;
    f.t = fill;
    a.t = v;
    b.w[0] = __builtin_amdgcn_update_dpp(f.w[0], a.w[0], CTRL, ROW_MASK, 0xf, false);
    b.w[1] = __builtin_amdgcn_update_dpp(f.w[1], a.w[1], CTRL, ROW_MASK, 0xf, false);
    return b.t;
  } else {
    union { T t; int32_t w; } f, a, b;
    f.t = fill;
    a.t = v;
    b.w = __builtin_amdgcn_update_dpp(f.w, a.w, CTRL, ROW_MASK, 0xf, false);
    return b.t;
  }
}

// Inclusive scan over the 64 lanes of a wave: four shifted steps inside each
// row of 16 lanes, then the last lane of row 0 (2) is folded into row 1 (3),
// then lane 31 into rows 2 and 3.
template <typename T, int OP>
__device__ __forceinline__ T wave_inclusive_scan(T v, int) {
  using F = Functor<T, OP>;
  const T id = F::identity();
  v = F::apply(dpp_move<T, 0x111, 0xf>(id, v), v);
  v = F::apply(dpp_move<T, 0x112, 0xf>(id, v), v);
  v = F::apply(dpp_move<T, 0x114, 0xf>(id, v), v);
  v = F::apply(dpp_move<T, 0x118, 0xf>(id, v), v);
  v = F::apply(dpp_move<T, 0x142, 0xa>(id, v), v);
  v = F::apply(dpp_move<T, 0x143, 0xc>(id, v), v);
  return v;
}

// Value of `v` in lane `src` as a wave-uniform (scalar register) value.
template <typename T>
__device__ __forceinline__ T read_lane(T v, int src) {
  if constexpr (sizeof(T) == 8) {
    union { T t; int32_t w[2]; } a, b;
    a.t = v;
    b.w[0] = __builtin_amdgcn_readlane(a.w[0], src);
    b.w[1] = __builtin_amdgcn_readlane(a.w[1], src);
    return b.t;
  } else {
    union { T t; int32_t w; } a, b;
    a.t = v;
    b.w = __builtin_amdgcn_readlane(a.w, src);
    return b.t;
  }
}

// Keeps a value where it is in program order: the scheduler otherwise
// interleaves the row scans of a tile and keeps a copy of every row alive.
template <typename T> __device__ __forceinline__ void pin(T& v) {
  if constexpr (sizeof(T) == 8) {
    union { T t; int32_t w[2]; } a;
    a.t = v;
    asm volatile("" : "+v"(a.w[0]), "+v"(a.w[1]));
    v = a.t;
  } else {
    union { T t; int32_t w; } a;
    a.t = v;
    asm volatile("" : "+v"(a.w));
    v = a.t;
  }
}

// Value of the previous lane; lane 0 receives `fill`.
template <typename T>
__device__ __forceinline__ T lane_shift_up(T fill, T v) {
  return dpp_move<T, 0x138, 0xf>(fill, v);
}

// Fold over the lanes of a wave, from lane 0 to lane 63 in this order, in every lane.
template <typename T, int OP>
__device__ __forceinline__ T wave_fold(T v, int lane) {
  return read_lane<T>(wave_inclusive_scan<T, OP>(v, lane), kWaveSize - 1);
}

// The aggregate of tile t, a full one, from the input, by one wave.  In the order in which the tile itself
// adds up (the vectors of a row, the rows of a wave, the waves), so that it is the same value bit for bit and a sum of
// floating-point numbers is no less exact for it.  Row after row: it runs where a tile is late, while the tile of
// its own block is held in registers, which more loads in flight would spill.
template <typename T, int OP, bool VECTOR, int VECS>
__device__ __forceinline__ T fold_tile(const T* __restrict__ in, int64_t in_stride, int t, int lane) {
  using F = Functor<T, OP>;
  using V = typename Vec16<T>::type;
  constexpr int VN = Vec16<T>::N;
  const T* row = in + (int64_t)t * (kBlock * VECS * VN) * (VECTOR ? 1 : in_stride);  // (wave-uniform)
  T total = F::identity(), wave_total = F::identity();
#pragma unroll 1
  for (int j = 0; j < kWaves * VECS; ++j) {
    T sum;
    if constexpr (VECTOR) {
      const V v = reinterpret_cast<const V*>(row)[lane];
      sum = v[0];
#pragma unroll
      for (int k = 1; k < VN; ++k) sum = F::apply(sum, v[k]);
    } else {
      const T* p = row + (int64_t)(lane * VN) * in_stride;
      sum = *p;
#pragma unroll 1
      for (int k = 1; k < VN; ++k) sum = F::apply(sum, *(p += in_stride));
    }
    row += kWaveSize * VN * (VECTOR ? 1 : in_stride);
    sum = wave_fold<T, OP>(sum, lane);
    wave_total = j % VECS == 0 ? sum : F::apply(wave_total, sum);
    if (j % VECS == VECS - 1) total = j == VECS - 1 ? wave_total : F::apply(total, wave_total);
  }
  return total;
}

// Tiles that begin with the launch, two per compute unit, wait for the one round trip in front of them.  Those
// that begin when one of these has ended find their predecessors at work, and poll 16 times as seldom: the polls go past the
// L2 and take from the data.  (us, all every 64 cycles / these every 1024: 2^27 int64 377 / 371, 2^27 double Max
// 397 / 393, 2^25 int64 97.0 / 96.1, 2^28 int32 350.6 both; and if all poll seldom, 2^23 int32 13.1 / 13.3, 2^22 int64 16.0 / 16.2.)
constexpr int kFirstTiles = 512;

// Executed by the first wave of the block.  Publishes the tile's aggregate,
// resolves the exclusive prefix of the tile and publishes the inclusive one.
// `fold(t)` is the aggregate of tile t from the input, by the whole wave, for a tile that has not published it
// within `limit` polls.
template <typename T, int OP, int STRIDE, typename Fold>
__device__ __forceinline__ T resolve_prefix(const TileState<T, STRIDE>& st, int tile,
                                            T aggregate, int lane, uint32_t limit, const Fold& fold) {
  using F = Functor<T, OP>;
  if (tile == 0) {
    if (lane == 0) st.publish(0, kFlagPrefix, aggregate);
    return F::identity();
  }
  if (lane == 0) st.publish(tile, kFlagAggregate, aggregate);
  T exclusive = F::identity();
  int base = tile - 1;
  while (true) {
    const int idx = base - (kWaveSize - 1 - lane);  // in the input's order: of two NaNs the first wins
    T val = F::identity();
    uint32_t flag = idx >= 0 ? kFlagInvalid : kFlagPrefix;  // virtual prefix in front of tile 0
    // The nearest inclusive prefix ends the walk; what lies in front of it is in it, and is not waited for.
    uint64_t has_prefix;
    int nearest;
    for (uint32_t polls = 0;; ++polls) {
      if (flag == kFlagInvalid) flag = st.read(idx, &val);
      has_prefix = __ballot(flag == kFlagPrefix);
      nearest = has_prefix != 0 ? kWaveSize - 1 - __builtin_clzll(has_prefix) : 0;
      const uint64_t missing = __ballot(flag == kFlagInvalid) >> nearest;
      if (missing == 0) break;
      if (limit == kNoLimit || polls < limit) {
        if (tile < kFirstTiles) __builtin_amdgcn_s_sleep(1);
        else __builtin_amdgcn_s_sleep(16);
        continue;
      }
      const int late = nearest + kWaveSize - 1 - __builtin_clzll(missing);  // (the nearest; then all are asked again)
      const T folded = fold(base - (kWaveSize - 1 - late));
      if (lane == late) {
        val = folded;
        flag = kFlagAggregate;
      }
    }
    const T contrib = lane >= nearest ? val : F::identity();
    exclusive = F::apply(wave_fold<T, OP>(contrib, lane), exclusive);
    if (has_prefix != 0) break;  // wave-uniform
    base -= kWaveSize;
  }
  if (lane == 0) st.publish(tile, kFlagPrefix, F::apply(exclusive, aggregate));
  return exclusive;
}

// Of a short tile, by the whole block: thread t waits for two neighbouring tiles, so the prefix is one round trip
// behind the slowest aggregate in front of it (a walk by one wave takes one per 64 tiles: 10^6 double Max 12.4
// against 11.4 us a call, 500 000 11.9 against 10.8).  Only aggregates are published.  Called by every thread; ends with a
// barrier.  (Not behind tickets, which come one after the other: 10^6 int64 11.2 against 10.5 by a walk.)
template <typename T, int OP, int STRIDE, typename Fold>
__device__ __forceinline__ T resolve_prefix_at_once(const TileState<T, STRIDE>& st, int tile, T aggregate,
                                                    int wave, int lane, T* s_front, uint32_t limit,
                                                    const Fold& fold) {
  using F = Functor<T, OP>;
  if (threadIdx.x == 0) st.publish(tile, kFlagAggregate, aggregate);
  constexpr int kPer = (int)(kShortMaxTiles * kShortDivisor + kBlock - 1) / kBlock;
  T of_tile[kPer];
  uint32_t waits = 0;  // a bit per tile
#pragma unroll
  for (int p = 0; p < kPer; ++p) {
    of_tile[p] = F::identity();
    if ((int)threadIdx.x * kPer + p < tile) waits |= 1u << p;
  }
  for (uint32_t polls = 0;; ++polls) {
#pragma unroll
    for (int p = 0; p < kPer; ++p)
      if ((waits >> p & 1u) != 0u && st.read((int)threadIdx.x * kPer + p, &of_tile[p]) != kFlagInvalid)
        waits &= ~(1u << p);
    const uint64_t missing = __ballot(waits != 0u);
    if (missing == 0) break;
    if (polls < limit) {
      __builtin_amdgcn_s_sleep(1);
      continue;
    }
    const int late = __builtin_ctzll(missing);
    const int of_late = __builtin_ctz((uint32_t)__builtin_amdgcn_readlane((int)waits, late));
    const int front = (wave * kWaveSize + late) * kPer + of_late;
    const T folded = fold(front);
    // (For the tiles behind, which wait for it as well; the tile itself publishes the same bits.)
    if (lane == 0) st.publish(front, kFlagAggregate, folded);
#pragma unroll
    for (int p = 0; p < kPer; ++p) {
      if (lane != late || p != of_late) continue;
      of_tile[p] = folded;
      waits &= ~(1u << p);
    }
  }
  T val = of_tile[0];
#pragma unroll
  for (int p = 1; p < kPer; ++p) val = F::apply(val, of_tile[p]);
  const T front = wave_fold<T, OP>(val, lane);
  if (lane == 0) s_front[wave] = front;
  __syncthreads();
  T exclusive = s_front[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) exclusive = F::apply(exclusive, s_front[w]);
  return exclusive;
}

// Four waves per SIMD, i.e. 128 registers and two blocks per CU: left to itself
// the compiler takes 180 to 256 registers for the floating-point Max and Min
// kernels, which halves their residency (0.56 -> 0.44 ms at 2^28 float, 0.36 since those
// take three compares: fp_extreme).
// TICKETS: with tiles by tickets; a kernel apart, since with both look-backs in it one over its input took longer
// than before there were two (us, one kernel / two: 10^6 int64 11.65 / 11.15, 2 * 10^6 int32 10.7 / 10.4, 2^22 int64 18.6 / 18.2,
// 10^7 float 21.75 / 20.7; into another view the same).
template <typename T, int OP, bool VECTOR, int VECS, bool TICKETS>
__global__ __launch_bounds__(kBlock, ILGPU_HIP_SCAN_WAVES_PER_EU) void scan_kernel(
    const T* __restrict__ in, T* __restrict__ out, int64_t n,
    int64_t in_stride, int64_t out_stride, int inclusive,
    uint32_t* __restrict__ ticket, TileState<T, status_stride<T, VECS>()> st, uint32_t limit) {
  using F = Functor<T, OP>;
  using V = typename Vec16<T>::type;
  constexpr int VN = Vec16<T>::N;
  constexpr int kTileVecs = VECS;
  constexpr int kTile = kBlock * VECS * VN;
  constexpr int kWaveElems = kTile / kWaves;

  __shared__ int s_tile;
  __shared__ T s_wave_total[kWaves];
  __shared__ T s_front[kWaves];  // of a short tile: what lies in front, a part per wave
  __shared__ T s_prefix;
  constexpr bool kShort = VECS != scan_vecs<T>();

  // An input of one tile comes without status words (and without
  // the launch that clears them): there is nobody to wait for or to tell.
  const bool alone = !TICKETS && gridDim.x == 1;
  if constexpr (TICKETS) {
    if (threadIdx.x == 0) s_tile = (int)atomicAdd(ticket, 1u);
    __syncthreads();
  }
  const int tile = TICKETS ? s_tile : (int)blockIdx.x;
  const int lane = threadIdx.x & (kWaveSize - 1);
  // The wave index and everything derived from it are wave-uniform: kept in
  // scalar registers, so a lane addresses its vectors by one 32-bit offset.
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
  const int64_t tile_base = (int64_t)tile * kTile;
  const int64_t wave_base = tile_base + (int64_t)wave * kWaveElems;
  const bool full = tile_base + kTile <= n;
  // Elements of this wave's chunk that lie inside the view (tail path only).
  const int wave_valid =
      (int)(n - wave_base < kWaveElems ? (n - wave_base < 0 ? 0 : n - wave_base)
                                       : kWaveElems);

  T x[kTileVecs][VN];
  constexpr bool kHalves = ILGPU_HIP_SCAN_LOAD_HALVES && sizeof(T) == 4 && kTileVecs % 2 == 0;
  auto load_rows = [&](int j0, int j1) {
    const V* src = reinterpret_cast<const V*>(in + wave_base);
#pragma unroll
    for (int j = j0; j < j1; ++j) {
      V v = ILGPU_HIP_SCAN_NT_LOAD ? __builtin_nontemporal_load(&src[j * kWaveSize + lane])
                                   : src[j * kWaveSize + lane];
#pragma unroll
      for (int k = 0; k < VN; ++k) x[j][k] = v[k];
    }
  };
  if (VECTOR && full) {
    load_rows(0, kHalves ? kTileVecs / 2 : kTileVecs);
  } else {
    // The last tile, or views that are not aligned or not dense.  Whole vectors of the last tile move as such, and only the
    // lane that holds the view's end goes by elements: by elements everywhere one tile is up to 128 loads and stores
    // of 1 KiB lines each that one compute unit's address unit takes, and the rest of the chip waits for its end
    // (calls, us, before / now: 20000 int32 11.8 / 7.4, 2^23 - 1 int32 20.7 / 14.1, 30000001 49.3 / 43.8).
#pragma unroll
    for (int j = 0; j < kTileVecs; ++j) {
      const int e0 = (j * kWaveSize + lane) * VN;
#pragma unroll
      for (int k = 0; k < VN; ++k) x[j][k] = F::identity();
      if (VECTOR && e0 + VN <= wave_valid) {
        const V v = *reinterpret_cast<const V*>(in + wave_base + e0);
#pragma unroll
        for (int k = 0; k < VN; ++k) x[j][k] = v[k];
      } else if (e0 < wave_valid) {
#pragma unroll
        for (int k = 0; k < VN; ++k)
          if (e0 + k < wave_valid) x[j][k] = in[(wave_base + e0 + k) * in_stride];
      }
    }
  }

  auto fold = [&](int t) -> T { return fold_tile<T, OP, VECTOR, VECS>(in, in_stride, t, lane); };
  auto prefix_of_tile = [&](T block_total) -> T {
    if (alone) return F::identity();
    if constexpr (kShort && !TICKETS && !ILGPU_HIP_SCAN_PROBE_NO_LOOKBACK)
      return resolve_prefix_at_once<T, OP>(st, tile, block_total, wave, lane, s_front, limit, fold);
    if (wave == 0) {
      const T exclusive = ILGPU_HIP_SCAN_PROBE_NO_LOOKBACK
                              ? F::identity()
                              : resolve_prefix<T, OP>(st, tile, block_total, lane, TICKETS ? kNoLimit : limit, fold);
      if (lane == 0) s_prefix = exclusive;
    }
    __syncthreads();
    return s_prefix;
  };

  if constexpr (sizeof(T) == 8) {
    // Register-lean form for 8-byte elements, whose per-row prefixes would
    // take two registers each: the prefix of the lower lanes is folded into
    // the row at once, so no per-row prefix outlives this loop, and the row
    // totals are wave-uniform values in scalar registers (104 registers at 16
    // vectors; 2^27 int64 Add 0.419 -> 0.382 ms against the form below at 10
    // vectors).  For 4-byte elements the two forms measure the same.
    T seg_total[kTileVecs];
#pragma unroll
    for (int j = 0; j < kTileVecs; ++j) {
#pragma unroll
      for (int k = 1; k < VN; ++k) x[j][k] = F::apply(x[j][k - 1], x[j][k]);
      const T inc = wave_inclusive_scan<T, OP>(x[j][VN - 1], lane);
      seg_total[j] = read_lane<T>(inc, kWaveSize - 1);
      const T up = lane_shift_up<T>(F::identity(), inc);
#pragma unroll
      for (int k = 0; k < VN; ++k) {
        x[j][k] = F::apply(up, x[j][k]);
        pin(x[j][k]);
      }
    }
    T wave_total = seg_total[0];
#pragma unroll
    for (int j = 1; j < kTileVecs; ++j) wave_total = F::apply(wave_total, seg_total[j]);
    if (lane == 0) s_wave_total[wave] = wave_total;
    __syncthreads();
    T wave_prefix = F::identity();
    T block_total = s_wave_total[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) {
      if (w == wave) wave_prefix = block_total;
      block_total = F::apply(block_total, s_wave_total[w]);
    }
    T running = F::apply(prefix_of_tile(block_total), wave_prefix);
    V* dst = reinterpret_cast<V*>(out + wave_base);
#pragma unroll
    for (int j = 0; j < kTileVecs; ++j) {
      T r[VN];
      if (inclusive) {
#pragma unroll
        for (int k = 0; k < VN; ++k) r[k] = F::apply(running, x[j][k]);
      } else {
        r[0] = F::apply(running, lane_shift_up<T>(F::identity(), x[j][VN - 1]));
#pragma unroll
        for (int k = 1; k < VN; ++k) r[k] = F::apply(running, x[j][k - 1]);
      }
      const int e0 = (j * kWaveSize + lane) * VN;
      V v;
#pragma unroll
      for (int k = 0; k < VN; ++k) v[k] = r[k];
      if (VECTOR && full) {
        if (ILGPU_HIP_SCAN_NT_STORE) __builtin_nontemporal_store(v, &dst[j * kWaveSize + lane]);
        else dst[j * kWaveSize + lane] = v;
      } else if (VECTOR && e0 + VN <= wave_valid) {
        dst[j * kWaveSize + lane] = v;
      } else if (e0 < wave_valid) {
#pragma unroll
        for (int k = 0; k < VN; ++k)
          if (e0 + k < wave_valid) out[(wave_base + e0 + k) * out_stride] = r[k];
      }
      running = F::apply(running, seg_total[j]);
    }
    return;
  }
  // Lane-local inclusive scan of each vector, then one wave scan per j.
  T lane_excl[kTileVecs];   // fold of the vectors of lower lanes, same j
  T seg_total[kTileVecs];   // fold of the whole 64-lane row j
  auto scan_rows = [&](int j0, int j1) {
#pragma unroll
    for (int j = j0; j < j1; ++j) {
#pragma unroll
      for (int k = 1; k < VN; ++k) x[j][k] = F::apply(x[j][k - 1], x[j][k]);
      const T inc = wave_inclusive_scan<T, OP>(x[j][VN - 1], lane);
      seg_total[j] = shfl(inc, kWaveSize - 1);
      lane_excl[j] = lane_shift_up<T>(F::identity(), inc);
    }
  };
  if (kHalves && VECTOR && full) {
    scan_rows(0, kTileVecs / 2);
    __builtin_amdgcn_sched_barrier(0);
    load_rows(kTileVecs / 2, kTileVecs);
    scan_rows(kTileVecs / 2, kTileVecs);
  } else {
    scan_rows(0, kTileVecs);
  }
  T wave_total = seg_total[0];
#pragma unroll
  for (int j = 1; j < kTileVecs; ++j) wave_total = F::apply(wave_total, seg_total[j]);
  if (lane == 0) s_wave_total[wave] = wave_total;
  __syncthreads();

  T wave_prefix = F::identity();
  T block_total = s_wave_total[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) {
    if (w == wave) wave_prefix = block_total;
    block_total = F::apply(block_total, s_wave_total[w]);
  }

  T running = F::apply(prefix_of_tile(block_total), wave_prefix);  // prefix of row 0 of this wave
  V* dst = reinterpret_cast<V*>(out + wave_base);
#pragma unroll
  for (int j = 0; j < kTileVecs; ++j) {
    const T before = F::apply(running, lane_excl[j]);  // prefix of x[j][0]
    T r[VN];
#pragma unroll
    for (int k = 0; k < VN; ++k) {
      if (inclusive) r[k] = F::apply(before, x[j][k]);
      else r[k] = k == 0 ? before : F::apply(before, x[j][k - 1]);
    }
    const int e0 = (j * kWaveSize + lane) * VN;
    V v;
#pragma unroll
    for (int k = 0; k < VN; ++k) v[k] = r[k];
    if (VECTOR && full) {
      if (ILGPU_HIP_SCAN_NT_STORE) __builtin_nontemporal_store(v, &dst[j * kWaveSize + lane]);
      else dst[j * kWaveSize + lane] = v;
    } else if (VECTOR && e0 + VN <= wave_valid) {
      dst[j * kWaveSize + lane] = v;
    } else if (e0 < wave_valid) {
#pragma unroll
      for (int k = 0; k < VN; ++k)
        if (e0 + k < wave_valid) out[(wave_base + e0 + k) * out_stride] = r[k];
    }
    running = F::apply(running, seg_total[j]);
  }
}

// ---- unique ------------------------------------------------------------------
// Removes consecutive duplicates in place and reports the new length; stands
// in for the Unique delegate of UniqueExtensions.cs:59-209, whose kernel runs
// the groups strictly one after the other (SequentialGroupExecutor) with a
// serial compaction loop per group.  Here it is the same single-pass chain as
// the scan: an element is kept if it differs from its predecessor, a tile
// publishes its number of kept elements, resolves how many were kept in front
// of it, and writes its kept elements to data[kept_before + local rank].
//
// In place is safe without a second buffer: a tile loads all of its elements
// (and the element in front of each vector) before it publishes anything, a
// tile learns its offset only after every earlier tile has published, and it
// writes only at or below the positions it read, so no element is overwritten
// before its owner (or its successor's comparison) has read it.
//
// "Differs" is Comparison<T>.Compare(a, b) != 0 (ComparisonOperations.tt:30-45),
// i.e. CompareTo: all NaNs are equal to each other and -0.0 equals +0.0.
#ifndef ILGPU_HIP_UNIQUE_VECS
#define ILGPU_HIP_UNIQUE_VECS 12
#endif
#ifndef ILGPU_HIP_UNIQUE_NT_STORE
#define ILGPU_HIP_UNIQUE_NT_STORE 1
#endif
#ifndef ILGPU_HIP_UNIQUE_VECS1
#define ILGPU_HIP_UNIQUE_VECS1 4
#endif
#ifndef ILGPU_HIP_UNIQUE_VECS2
#define ILGPU_HIP_UNIQUE_VECS2 8
#endif
// 16-byte vectors per thread and tile, by element size: every element of a
// vector is unpacked into a register of its own, so a vector of bytes costs
// sixteen registers and one of 2-byte elements eight.
constexpr int unique_vecs(int elem_bytes) {
  return elem_bytes == 1 ? ILGPU_HIP_UNIQUE_VECS1
                         : elem_bytes == 2 ? ILGPU_HIP_UNIQUE_VECS2 : ILGPU_HIP_UNIQUE_VECS;
}

template <typename T> struct is_float_like { static constexpr bool value = is_fp<T>::value; };
template <> struct is_float_like<_Float16> { static constexpr bool value = true; };

template <typename T> __device__ __forceinline__ bool differs(T a, T b) {
  if constexpr (is_float_like<T>::value) return !(a == b) && !(a != a && b != b);
  else return a != b;
}

template <typename T, int VECS> constexpr int unique_tile_elems() {
  return kBlock * VECS * Vec16<T>::N;
}
// Of 4-byte elements that fill the chip with such tiles once (two blocks a compute unit): longer ones, as many as fit 128
// registers, for fewer tickets and trips between tiles.  (us with a copy of the keys, 12 vectors / 16: sorted Zipf
// u32 2^27 287 / 273, 2^26 153 / 145, distinct int32 2^27 363 / 354, 3 * 10^7 80.2 / 77.8, but 3 * 10^6, 92 tiles, 18.5 / 21.6.
// 8-byte elements: 2^27 distinct 707 / 714, 14 vectors 702; 3 * 10^7 171.6 / 174.2, 172.5.)
constexpr int unique_long_vecs(int elem_bytes) { return elem_bytes == 4 ? 16 : unique_vecs(elem_bytes); }
constexpr int64_t kUniqueLongTiles = 512;

template <typename T, bool VECTOR, int VECS>
__global__ __launch_bounds__(kBlock) void unique_kernel(
    T* data, int64_t n, int64_t* __restrict__ out_length,
    uint32_t* __restrict__ ticket, TileState<uint32_t> st, int num_tiles) {
  using V = typename Vec16<T>::type;
  constexpr int VN = Vec16<T>::N;
  constexpr int kUniqueVecs = VECS;
  constexpr int kTile = unique_tile_elems<T, VECS>();
  constexpr int kWaveElems = kTile / kWaves;

  __shared__ int s_tile;
  __shared__ uint32_t s_wave_total[kWaves];
  __shared__ uint32_t s_prefix;

  const bool alone = ticket == nullptr;  // one tile: no ticket, no status words
  if (!alone) {
    if (threadIdx.x == 0) s_tile = (int)atomicAdd(ticket, 1u);
    __syncthreads();
  }
  const int tile = alone ? 0 : s_tile;
  const int lane = threadIdx.x & (kWaveSize - 1);
  const int wave = threadIdx.x / kWaveSize;
  const int64_t tile_base = (int64_t)tile * kTile;
  const int64_t wave_base = tile_base + (int64_t)wave * kWaveElems;
  const bool full = tile_base + kTile <= n;

  T x[kUniqueVecs][VN];
  // The element in front of the wave's chunk; every other predecessor is in a
  // register of this wave.
  const T chunk_before = wave_base > 0 && wave_base < n ? data[wave_base - 1] : T();
  // Elements of this wave's chunk that lie inside the view.
  const int64_t inside = n - wave_base;
  const int wave_valid = (int)(inside < kWaveElems ? (inside < 0 ? 0 : inside) : kWaveElems);
  if (VECTOR && full) {
    const V* src = reinterpret_cast<const V*>(data + wave_base);
#pragma unroll
    for (int j = 0; j < kUniqueVecs; ++j) {
      const V v = __builtin_nontemporal_load(&src[j * kWaveSize + lane]);
#pragma unroll
      for (int k = 0; k < VN; ++k) x[j][k] = v[k];
    }
  } else {
#pragma unroll
    for (int j = 0; j < kUniqueVecs; ++j) {
      const int e0 = (j * kWaveSize + lane) * VN;
#pragma unroll
      for (int k = 0; k < VN; ++k) x[j][k] = T();
      if (VECTOR && e0 + VN <= wave_valid) {
        const V v = *reinterpret_cast<const V*>(data + wave_base + e0);
#pragma unroll
        for (int k = 0; k < VN; ++k) x[j][k] = v[k];
      } else if (e0 < wave_valid) {
#pragma unroll
        for (int k = 0; k < VN; ++k)
          if (e0 + k < wave_valid) x[j][k] = data[wave_base + e0 + k];
      }
    }
  }
  T before[kUniqueVecs];  // the element in front of each vector
#pragma unroll
  for (int j = 0; j < kUniqueVecs; ++j) {
    const T from_left = shfl_up(x[j][VN - 1], 1);
    const T row_before = j == 0 ? chunk_before : shfl(x[j > 0 ? j - 1 : 0][VN - 1], kWaveSize - 1);
    before[j] = lane == 0 ? row_before : from_left;
  }

  // keep bit k of vector j; kept elements per vector; wave scan per row.
  // The counts of a few rows, up to 64 * VN each, go through one scan.  (With a scan for each row, element after element
  // asked whether it lies inside the view, and whole rows without a kept element stored lane by lane, 123
  // registers instead of 93 for 12 vectors: sorted Zipf keys, 2^26 u32, 82 -> 72 us, 2^27 of them 302 -> 287 with their copy.)
  constexpr int kRowsAScan = VN <= 8 ? 3 : 2, kRowBits = 32 / kRowsAScan;
  static_assert(kWaveSize * VN < 1 << kRowBits, "a row's total has its bits");
  uint32_t keep[kUniqueVecs], lane_excl[kUniqueVecs], seg_total[kUniqueVecs];
#pragma unroll
  for (int j = 0; j < kUniqueVecs; ++j) {
    uint32_t bits = 0;
#pragma unroll
    for (int k = 0; k < VN; ++k)
      bits |= (differs<T>(x[j][k], k == 0 ? before[j] : x[j][k - 1]) ? 1u : 0u) << k;
    if (j == 0 && wave_base == 0 && lane == 0) bits |= 1u;  // the first element of all
    if (!full) {
      const int left = wave_valid - (j * kWaveSize + lane) * VN;
      bits &= left >= VN ? (1u << VN) - 1u : (left <= 0 ? 0u : (1u << left) - 1u);
    }
    keep[j] = bits;
  }
#pragma unroll
  for (int j0 = 0; j0 < kUniqueVecs; j0 += kRowsAScan) {
    uint32_t cnt = 0;
#pragma unroll
    for (int r = 0; r < kRowsAScan; ++r)
      if (j0 + r < kUniqueVecs) cnt |= (uint32_t)__popc(keep[j0 + r]) << (r * kRowBits);
    const uint32_t inc = wave_inclusive_scan<uint32_t, ILGPU_HIP_OP_ADD>(cnt, lane);
    const uint32_t all = read_lane<uint32_t>(inc, kWaveSize - 1), front = inc - cnt;
#pragma unroll
    for (int r = 0; r < kRowsAScan; ++r)
      if (j0 + r < kUniqueVecs) {
        seg_total[j0 + r] = all >> (r * kRowBits) & ((1u << kRowBits) - 1u);
        lane_excl[j0 + r] = front >> (r * kRowBits) & ((1u << kRowBits) - 1u);
      }
  }
  uint32_t wave_total = 0;
#pragma unroll
  for (int j = 0; j < kUniqueVecs; ++j) wave_total += seg_total[j];
  if (lane == 0) s_wave_total[wave] = wave_total;
  __syncthreads();

  uint32_t wave_prefix = 0, block_total = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    if (w == wave) wave_prefix = block_total;
    block_total += s_wave_total[w];
  }
  if (wave == 0) {
    const uint32_t exclusive =
        alone ? 0u : resolve_prefix<uint32_t, ILGPU_HIP_OP_ADD>(st, tile, block_total, lane, kNoLimit,
                                                                [](int) { return 0u; });
    if (lane == 0) s_prefix = exclusive;
  }
  __syncthreads();

  uint32_t running = s_prefix + wave_prefix;
#pragma unroll
  for (int j = 0; j < kUniqueVecs; ++j) {
    if (seg_total[j] == 0u) continue;  // (wave-uniform)
    uint32_t pos = running + lane_excl[j];
    if (keep[j] == (1u << VN) - 1u) {
      // the whole vector survives: one 16-byte store, aligned like an element
      typedef V UnalignedV __attribute__((aligned(sizeof(T))));
      V v;
#pragma unroll
      for (int k = 0; k < VN; ++k) v[k] = x[j][k];
      if (ILGPU_HIP_UNIQUE_NT_STORE) __builtin_nontemporal_store(v, reinterpret_cast<UnalignedV*>(data + pos));
      else *reinterpret_cast<UnalignedV*>(data + pos) = v;
    } else {
#pragma unroll
      for (int k = 0; k < VN; ++k)
        if (keep[j] >> k & 1u) data[pos++] = x[j][k];
    }
    running += seg_total[j];
  }
  if (tile == num_tiles - 1 && threadIdx.x == 0)
    out_length[0] = (int64_t)s_prefix + (int64_t)block_total;
}

__global__ void zero_words_kernel(uint32_t* words, int64_t count, uint32_t* more,
                                  int64_t more_count) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t first = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (int64_t i = first; i < count; i += stride) words[i] = 0u;
  for (int64_t i = first; i < more_count; i += stride) more[i] = 0u;
}

template <typename T> int64_t num_tiles(int64_t n) {
  return div_up(n, tile_elems<T>());
}

template <typename T, int OP, int VECS>
int32_t launch_tiles(hipStream_t stream, const void* in, int64_t in_stride,
                     void* out, int64_t out_stride, int64_t n, int32_t kind,
                     void* temp, bool apart) {
  const int64_t tiles = div_up(n, (int64_t)kBlock * VECS * Vec16<T>::N);
  char* base = reinterpret_cast<char*>(align_up((int64_t)(uintptr_t)temp, 256));
  uint32_t* ticket = reinterpret_cast<uint32_t*>(base);
  TileState<T, status_stride<T, VECS>()> st;
  st.words = reinterpret_cast<uint64_t*>(base + kHeaderBytes);
  if (tiles > 1) {
    const int64_t zero_words = (kHeaderBytes + tiles * status_stride<T, VECS>() * 8) / 4;
    const int32_t rc = launch_zero_words(stream, reinterpret_cast<uint32_t*>(base), zero_words);
    if (rc != ILGPU_HIP_SUCCESS) return rc;
  }
  // (One tile: one launch.)
  if (tiles == 1 || apart) ticket = nullptr;
  const uint32_t limit = ticket != nullptr ? kNoLimit : lookback_spin_limit();
  // Element strides above one (Stride1D.General) take the scalar path.
  const bool vector = in_stride == 1 && out_stride == 1 &&
                      (reinterpret_cast<uintptr_t>(in) & 15) == 0 &&
                      (reinterpret_cast<uintptr_t>(out) & 15) == 0;
  const int inclusive = kind == ILGPU_HIP_SCAN_INCLUSIVE ? 1 : 0;
  ProfileScope scope(stream, "scan");
  auto* kernel = ticket != nullptr ? (vector ? scan_kernel<T, OP, true, VECS, true> : scan_kernel<T, OP, false, VECS, true>)
                                   : (vector ? scan_kernel<T, OP, true, VECS, false> : scan_kernel<T, OP, false, VECS, false>);
  hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(kBlock), 0, stream, static_cast<const T*>(in),
                     static_cast<T*>(out), n, in_stride, out_stride, inclusive, ticket, st, limit);
  ILGPU_HIP_CHECK(hipGetLastError());
  return ILGPU_HIP_SUCCESS;
}

template <typename T, int OP>
int32_t launch_typed(hipStream_t stream, const void* in, int64_t in_stride,
                     void* out, int64_t out_stride, int64_t n, int32_t kind,
                     void* temp) {
  const int64_t tiles = num_tiles<T>(n);
  // Whether the views, from their first byte to their last, do not meet.
  const auto end = [&](const void* p, int64_t stride) {
    return reinterpret_cast<uintptr_t>(p) + (uintptr_t)((n - 1) * stride + 1) * sizeof(T);
  };
  const bool apart = end(in, in_stride) <= reinterpret_cast<uintptr_t>(out) ||
                     end(out, out_stride) <= reinterpret_cast<uintptr_t>(in);
  constexpr int kShortVecs = scan_vecs<T>() / kShortDivisor;
  const bool one_short = n <= (int64_t)kBlock * kShortVecs * Vec16<T>::N;
  if (one_short || (tiles > 1 && tiles <= (apart ? kShortMaxTiles : kShortMaxTilesTicketed)))
    return launch_tiles<T, OP, kShortVecs>(
        stream, in, in_stride, out, out_stride, n, kind, temp, apart);
  return launch_tiles<T, OP, scan_vecs<T>()>(stream, in, in_stride, out, out_stride, n, kind, temp, apart);
}

template <typename T>
int32_t launch_op(hipStream_t stream, const void* in, int64_t in_stride,
                  void* out, int64_t out_stride, int64_t n, int32_t op,
                  int32_t kind, void* temp) {
  switch (op) {
    case ILGPU_HIP_OP_ADD:
      return launch_typed<T, ILGPU_HIP_OP_ADD>(stream, in, in_stride, out, out_stride, n,
                                               kind, temp);
    case ILGPU_HIP_OP_MAX:
      return launch_typed<T, ILGPU_HIP_OP_MAX>(stream, in, in_stride, out, out_stride, n,
                                               kind, temp);
    case ILGPU_HIP_OP_MIN:
      return launch_typed<T, ILGPU_HIP_OP_MIN>(stream, in, in_stride, out, out_stride, n,
                                               kind, temp);
    default:
      return ILGPU_HIP_ERROR_NOT_SUPPORTED;
  }
}

}  // namespace

int32_t launch_zero_words(hipStream_t stream, uint32_t* words, int64_t count, uint32_t* more,
                          int64_t more_count) {
  if (count <= 0 && more_count <= 0) return ILGPU_HIP_SUCCESS;
  int64_t blocks = div_up(std::max(count, more_count), 256 * 4);
  if (blocks > 2048) blocks = 2048;
  ProfileScope scope(stream, "zero_words");
  hipLaunchKernelGGL(zero_words_kernel, dim3((unsigned)blocks), dim3(256), 0,
                     stream, words, count, more, more_count);
  ILGPU_HIP_CHECK(hipGetLastError());
  return ILGPU_HIP_SUCCESS;
}

int64_t scan_temp_bytes(int64_t n, int elem_bytes) {
  // 256 bytes of alignment slack + header + per-tile state.
  const int64_t tiles =
      elem_bytes == 4 ? num_tiles<uint32_t>(n) : num_tiles<uint64_t>(n);
  return 256 + kHeaderBytes + tiles * kStatusBytes;
}

int32_t launch_scan(hipStream_t stream, const void* in, int64_t in_stride,
                    void* out, int64_t out_stride, int64_t n, int32_t type,
                    int32_t op, int32_t kind, void* temp) {
  switch (type) {
    case ILGPU_HIP_I32: return launch_op<int32_t>(stream, in, in_stride, out, out_stride, n, op, kind, temp);
    case ILGPU_HIP_U32: return launch_op<uint32_t>(stream, in, in_stride, out, out_stride, n, op, kind, temp);
    case ILGPU_HIP_I64: return launch_op<int64_t>(stream, in, in_stride, out, out_stride, n, op, kind, temp);
    case ILGPU_HIP_U64: return launch_op<uint64_t>(stream, in, in_stride, out, out_stride, n, op, kind, temp);
    case ILGPU_HIP_F32: return launch_op<float>(stream, in, in_stride, out, out_stride, n, op, kind, temp);
    case ILGPU_HIP_F64: return launch_op<double>(stream, in, in_stride, out, out_stride, n, op, kind, temp);
    default: return ILGPU_HIP_ERROR_NOT_SUPPORTED;
  }
}

// ---- scan on the library's own scratch ---------------------------------------
// For callers that cannot allocate or carry a temp view: the tile states of one
// scan live in a device array that is part of the library's code object.  It is
// sized for kStaticScanTiles tiles (1 GiB of input); every call on a GPU shares
// that GPU's copy, so calls that overlap in time on one GPU race.
constexpr int64_t kSmallestTileBytes =
    (int64_t)kBlock * 16 * (scan_vecs<uint32_t>() < scan_vecs<uint64_t>() ? scan_vecs<uint32_t>()
                                                                           : scan_vecs<uint64_t>());
constexpr int64_t kStaticScanTiles = ILGPU_HIP_SCAN_STATIC_MAX_BYTES / kSmallestTileBytes;
constexpr int64_t kStaticScratchBytes = kHeaderBytes + kStaticScanTiles * kStatusBytes;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
std::atomic<void*> g_scratch_ptr[kMaxDevices];
}  // namespace

int32_t launch_scan_static(hipStream_t stream, const void* in, int64_t in_stride,
                           void* out, int64_t out_stride, int64_t n, int32_t type,
                           int32_t op, int32_t kind) {
  // The tiles of this call must fit the array: scan_temp_bytes() minus the
  // alignment slack a caller's temp needs (the array is aligned itself).
  if (scan_temp_bytes(n, elem_size(type)) - 256 > kStaticScratchBytes)
    return ILGPU_HIP_ERROR_STATIC_LIMIT;
  int device = -1;
  ILGPU_HIP_CHECK(hipGetDevice(&device));
  if (device < 0 || device >= kMaxDevices) return ILGPU_HIP_ERROR_NOT_SUPPORTED;
  // Every GPU holds its own copy of the array at its own address; the array's
  // name is no device address on the host.  Looked up once per device.
  void* ptr = g_scratch_ptr[device].load(std::memory_order_acquire);
  if (ptr == nullptr) {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    ptr = g_scratch_ptr[device].load(std::memory_order_relaxed);
    if (ptr == nullptr) {
      ILGPU_HIP_CHECK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
      if (ptr == nullptr) return ILGPU_HIP_ERROR_RUNTIME;
      g_scratch_ptr[device].store(ptr, std::memory_order_release);
    }
  }
  // launch_scan clears the ticket and the status lines it will use with a fill
  // kernel (the array keeps the previous call's contents) and hands `ptr` to
  // the scan kernel as it does with a caller's temp.
  return launch_scan(stream, in, in_stride, out, out_stride, n, type, op, kind, ptr);
}

int64_t unique_temp_bytes(int64_t n, int elem_bytes) {
  const int64_t tile = (int64_t)kBlock * unique_vecs(elem_bytes) * (16 / elem_bytes);
  return 256 + kHeaderBytes + div_up(n, tile) * kStatusBytes;
}

namespace {
template <typename T, int VECS>
int32_t launch_unique_tiles(hipStream_t stream, void* data, int64_t n,
                            int64_t* out_length, void* temp) {
  const int64_t tiles = div_up(n, (int64_t)unique_tile_elems<T, VECS>());
  char* base = reinterpret_cast<char*>(align_up((int64_t)(uintptr_t)temp, 256));
  uint32_t* ticket = reinterpret_cast<uint32_t*>(base);
  TileState<uint32_t> st;
  st.words = reinterpret_cast<uint64_t*>(base + kHeaderBytes);
  if (tiles > 1) {
    const int32_t rc = launch_zero_words(stream, reinterpret_cast<uint32_t*>(base),
                                         (kHeaderBytes + tiles * kStatusBytes) / 4);
    if (rc != ILGPU_HIP_SUCCESS) return rc;
  } else {
    ticket = nullptr;  // one tile: one launch
  }
  const bool vector = (reinterpret_cast<uintptr_t>(data) & 15) == 0;
  ProfileScope scope(stream, "unique");
  if (vector)
    hipLaunchKernelGGL((unique_kernel<T, true, VECS>), dim3((unsigned)tiles), dim3(kBlock), 0,
                       stream, static_cast<T*>(data), n, out_length, ticket, st,
                       (int)tiles);
  else
    hipLaunchKernelGGL((unique_kernel<T, false, VECS>), dim3((unsigned)tiles), dim3(kBlock), 0,
                       stream, static_cast<T*>(data), n, out_length, ticket, st,
                       (int)tiles);
  ILGPU_HIP_CHECK(hipGetLastError());
  return ILGPU_HIP_SUCCESS;
}

template <typename T>
int32_t launch_unique_typed(hipStream_t stream, void* data, int64_t n,
                            int64_t* out_length, void* temp) {
  constexpr int kVecs = unique_vecs(sizeof(T)), kLongVecs = unique_long_vecs(sizeof(T));
  static_assert(kLongVecs >= kVecs, "the temp view is sized for the shorter tiles");
  if (kLongVecs != kVecs && n >= kUniqueLongTiles * unique_tile_elems<T, kLongVecs>())
    return launch_unique_tiles<T, kLongVecs>(stream, data, n, out_length, temp);
  return launch_unique_tiles<T, kVecs>(stream, data, n, out_length, temp);
}
}  // namespace

int32_t launch_unique(hipStream_t stream, void* data, int64_t n, int32_t type,
                      int64_t* out_length, void* temp) {
  switch (type) {
    case ILGPU_HIP_I8: return launch_unique_typed<int8_t>(stream, data, n, out_length, temp);
    case ILGPU_HIP_U8: return launch_unique_typed<uint8_t>(stream, data, n, out_length, temp);
    case ILGPU_HIP_I16: return launch_unique_typed<int16_t>(stream, data, n, out_length, temp);
    case ILGPU_HIP_U16: return launch_unique_typed<uint16_t>(stream, data, n, out_length, temp);
    case ILGPU_HIP_I32: return launch_unique_typed<int32_t>(stream, data, n, out_length, temp);
    case ILGPU_HIP_U32: return launch_unique_typed<uint32_t>(stream, data, n, out_length, temp);
    case ILGPU_HIP_I64: return launch_unique_typed<int64_t>(stream, data, n, out_length, temp);
    case ILGPU_HIP_U64: return launch_unique_typed<uint64_t>(stream, data, n, out_length, temp);
    case ILGPU_HIP_F16: return launch_unique_typed<_Float16>(stream, data, n, out_length, temp);
    case ILGPU_HIP_F32: return launch_unique_typed<float>(stream, data, n, out_length, temp);
    case ILGPU_HIP_F64: return launch_unique_typed<double>(stream, data, n, out_length, temp);
    default: return ILGPU_HIP_ERROR_NOT_SUPPORTED;
  }
}

}  // namespace ilgpu_hip
