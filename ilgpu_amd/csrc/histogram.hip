// Histogram: bins[locator(v)] += 1 for every input element.
//
// Stands in for HistogramKernel / HistogramUncheckedKernel and the launchers
// (HistogramExtensions.cs:176-354, HistogramLaunchers.tt:52-101).  The
// reference issues one global atomic per element (HistogramOperations.tt:
// 36-40); here each block counts into a private LDS histogram and adds each
// non-zero bin to the global bins once.
//
// LDS layout: R replicas of every bin, word index = bin * R + (lane % R).
// With R = 32 a wave's 64 LDS atomics land in 32 different banks whatever the
// data (uniform, skewed or constant), so neither bank conflicts nor
// same-address serialisation depend on the input.  R is the largest power of
// two <= 32 for which num_bins * R counters fit in 48 KiB; histograms with
// more than 12288 bins fall through to global atomics per element.
//
// Overflow (checked variant): the reference flags an increment that saw
// old == MaxValue.  A bulk add of c > 0 to a bin holding `old` passes through
// MaxValue exactly when old + c, in wider arithmetic, exceeds it.
//
// Algorithmic HBM traffic: n * sizeof(T) bytes read; bins are negligible.
#include <algorithm>
#include <type_traits>

#include "kernels.hpp"

namespace ilgpu_hip {

namespace {

constexpr int kBlock = 512;
constexpr int kUnroll = 2;
#ifndef ILGPU_HIP_HISTOGRAM_FEW_UNROLL
#define ILGPU_HIP_HISTOGRAM_FEW_UNROLL 4
#endif
#ifndef ILGPU_HIP_HISTOGRAM_FEW_BLOCK
#define ILGPU_HIP_HISTOGRAM_FEW_BLOCK 1024
#endif
constexpr int kFewUnroll = ILGPU_HIP_HISTOGRAM_FEW_UNROLL;  // at most one block per CU
#ifndef ILGPU_HIP_HISTOGRAM_STRIDED_UNROLL
#define ILGPU_HIP_HISTOGRAM_STRIDED_UNROLL 4
#endif
constexpr int kStridedUnroll = ILGPU_HIP_HISTOGRAM_STRIDED_UNROLL;
constexpr int kCrowdedMaxReplicaShift = 2;  // fewer than eight replicas of a bin
constexpr int kLdsBudgetWords = 12288;  // 48 KiB of counters per block
constexpr int kMaxReplicas = 32;
// A block's fixed cost is its flush, one returning global atomic per bin that it
// has counted into; with three blocks per CU whatever the input, 8 M ints into 4096
// bins spent 40 of 50 us on 3.1 M of them.  A block is worth its flush from
// kMinElementsPerBin elements per bin on; half a block per CU is taken anyway, to
// read short inputs.  (4096 bins, initialize and histogram, us with three blocks per
// CU / now: 10^6 ints 30.3 / 16.7, 8 * 10^6 49.5 / 18.8, 2^24 50.1 / 19.9, 2^26
// 71.9 / 54.6, the last by the order of the flush alone.  With 4, 8 and 32 elements
// per bin 2^24 took 31.0, 25.0 and 32.2 where 16 took 23.7, before the loads of
// kFormCrowdedFew.)
#ifndef ILGPU_HIP_HISTOGRAM_ELEMENTS_PER_BIN
#define ILGPU_HIP_HISTOGRAM_ELEMENTS_PER_BIN 16
#endif
#ifndef ILGPU_HIP_HISTOGRAM_MIN_BLOCKS_DIVISOR
#define ILGPU_HIP_HISTOGRAM_MIN_BLOCKS_DIVISOR 2
#endif
constexpr int64_t kMinElementsPerBin = ILGPU_HIP_HISTOGRAM_ELEMENTS_PER_BIN;
constexpr int kMinBlocksDivisor = ILGPU_HIP_HISTOGRAM_MIN_BLOCKS_DIVISOR;

// ---- bin locators ---------------------------------------------------------
// IDENTITY: bin = (int)value.  MODULO: |value % num_bins| with the sign of the
// dividend (C# remainder; HistogramTests.tt:83-94), i.e. |value| mod num_bins;
// floating point uses fmod.
template <typename T, int LOC>
__device__ __forceinline__ int64_t locate(T v, int num_bins) {
  if constexpr (LOC == ILGPU_HIP_LOCATOR_IDENTITY) {
    if constexpr (is_fp<T>::value) {
      // Saturating conversion keeps NaN/inf/huge values out of range.
      if (!(v > (T)-1 && v < (T)2147483648.0)) return -1;
      return (int64_t)(int32_t)v;
    } else if constexpr (sizeof(T) == 8) {
      if constexpr (T(-1) < T(0)) return (int64_t)v;
      else return v > (T)INT64_MAX ? -1 : (int64_t)v;
    } else {
      return (int64_t)v;
    }
  } else {
    if constexpr (is_fp<T>::value) {
      T r = sizeof(T) == 4 ? (T)fmodf((float)v, (float)num_bins)
                           : (T)fmod((double)v, (double)num_bins);
      r = r < 0 ? -r : r;
      if (!(r >= 0)) return -1;  // NaN
      return (int64_t)(int32_t)r;
    } else if constexpr (sizeof(T) == 8) {
      uint64_t mag;
      if constexpr (T(-1) < T(0)) mag = v < 0 ? (uint64_t)0 - (uint64_t)v : (uint64_t)v;
      else mag = (uint64_t)v;
      return (int64_t)(mag % (uint64_t)num_bins);
    } else {
      const int64_t w = (int64_t)v;
      const uint32_t mag = (uint32_t)(w < 0 ? -w : w);
      return (int64_t)(mag % (uint32_t)num_bins);
    }
  }
}

template <typename B> struct BinTraits;
template <> struct BinTraits<int32_t> {
  static __device__ __forceinline__ bool passes_max(int32_t old, uint32_t c) {
    return (int64_t)old + (int64_t)c > (int64_t)INT32_MAX;
  }
};
template <> struct BinTraits<uint32_t> {
  static __device__ __forceinline__ bool passes_max(uint32_t old, uint32_t c) {
    return (uint64_t)old + (uint64_t)c > (uint64_t)UINT32_MAX;
  }
};
template <> struct BinTraits<int64_t> {
  static __device__ __forceinline__ bool passes_max(int64_t old, uint32_t c) {
    return old > INT64_MAX - (int64_t)c;
  }
};
template <> struct BinTraits<uint64_t> {
  static __device__ __forceinline__ bool passes_max(uint64_t old, uint32_t c) {
    return old > UINT64_MAX - (uint64_t)c;
  }
};

// Adds c to bins[b] as bin type B; returns whether the add passed MaxValue.
template <typename B>
__device__ __forceinline__ bool add_to_bin(void* bins, int64_t b, uint32_t c,
                                           bool checked) {
  if constexpr (sizeof(B) == 4) {
    uint32_t* p = static_cast<uint32_t*>(bins) + b;
    if (!checked) {
      __hip_atomic_fetch_add(p, c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
    const uint32_t old = __hip_atomic_fetch_add(p, c, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
    return BinTraits<B>::passes_max((B)old, c);
  } else {
    uint64_t* p = static_cast<uint64_t*>(bins) + b;
    if (!checked) {
      __hip_atomic_fetch_add(p, (uint64_t)c, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
    const uint64_t old = __hip_atomic_fetch_add(p, (uint64_t)c, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
    return BinTraits<B>::passes_max((B)old, c);
  }
}

// ---- floating-point bins ------------------------------------------------------
// The reference adds 1.0 to a float or double bin once per element, each
// addition rounded in the bin's precision (Atomic.Add(ref target, 1),
// HistogramOperations.tt:36-40), so a float bin stops growing at 2^24.  Every
// increment is the same function x -> fl(x + 1), so the value of a bin after c
// of them does not depend on their order, and add_ones gives exactly that
// value without c additions: inside a binade whose spacing is at most one,
// steps of one are exact (x, 1 and x + 1 are multiples of the spacing), so
// whole runs of steps up to the top of the binade (or, for negative values,
// down to magnitude below one) are taken at once; the steps that can round —
// into a coarser binade, across zero, beyond 2^24 or 2^53 — are single
// additions in hardware.
template <typename F>
__device__ __forceinline__ F add_ones(F x, uint32_t c) {
  constexpr int kDigits = sizeof(F) == 4 ? 24 : 53;
  const F limit = (F)(1ull << kDigits);
  if (x != x) return x;  // NaN stays NaN
  while (c > 0) {
    const F y = x + (F)1;
    if (y == x) return x;  // stuck: the spacing has outgrown one (or x is infinite)
    uint32_t k = 1;
    F next = y;
    const F ax = x < (F)0 ? -x : x;
    if (ax >= (F)1 && ax < limit) {
      uint64_t whole;
      if (x > (F)0) {
        int e;
        if constexpr (sizeof(F) == 4) (void)frexpf(x, &e);
        else (void)frexp(x, &e);
        F top;  // 2^e: the first value of the next binade, above x
        if constexpr (sizeof(F) == 4) top = ldexpf(1.0f, e);
        else top = ldexp(1.0, e);
        whole = (uint64_t)(top - x);  // steps that end at or below it
      } else {
        whole = (uint64_t)ax;         // steps that end at or below zero
      }
      if (whole >= 1) {
        k = whole < (uint64_t)c ? (uint32_t)whole : c;
        next = x + (F)k;  // exact
      }
    }
    x = next;
    c -= k;
  }
  return x;
}

// Where a bin stays that ones have taken there: 2^24 (2^53).
template <typename F> constexpr F kOnesEnd = (F)(1ull << (sizeof(F) == 4 ? 24 : 53));
// Whether c ones can be added to a bin that holds x as one c: from a whole number up to
// kOnesEnd on every step of one is exact until it reaches that.
template <typename F>
__device__ __forceinline__ bool ones_are_exact(F x, uint32_t c) {
  const F whole = sizeof(F) == 4 ? (F)truncf((float)x) : (F)trunc((double)x);
  return x == whole && x >= -kOnesEnd<F> && x <= kOnesEnd<F> && (sizeof(F) == 8 || c <= 1u << 24);
}
// What follows an addition of c in one to a bin of which ones_are_exact: `before` is what it held. A bin that
// was taken beyond 2^24 (2^53) is put back to it, the value that the ones would have stopped at.  Whoever
// adds to such a bin in between finds it beyond as well, or puts it back afterwards, so the last to do so leaves
// it there.
template <typename F, typename U>
__device__ __forceinline__ void settle_fp_bin(F* bin, F before, uint32_t c) {
  constexpr F kLimit = kOnesEnd<F>;
  if (before <= kLimit - (F)c) return;
  U* p = reinterpret_cast<U*>(bin);
  U limit_bits, old = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __builtin_memcpy(&limit_bits, &kLimit, sizeof(F));
  while (true) {
    F x;
    __builtin_memcpy(&x, &old, sizeof(F));
    if (x <= kLimit) break;
    if (__hip_atomic_compare_exchange_strong(p, &old, limit_bits, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT))
      break;
  }
}

// Adds c ones to the floating-point bin b; returns whether an increment found
// the bin at MaxValue (only a bin that holds MaxValue already: it is not
// reachable by steps of one).
template <typename F, typename U>
__device__ __forceinline__ bool add_to_fp_bin(void* bins, int64_t b, uint32_t c,
                                              bool checked) {
  const F max_value = sizeof(F) == 4 ? (F)3.402823466e+38f : (F)1.7976931348623157e+308;
  if (c == 1u) {
    // One element: the hardware's floating-point add in L2 is the reference's
    // operation itself (one addition of 1.0, rounded in the bin's precision),
    // and it does not retry: many elements for one bin do not starve each
    // other as compare-and-swap loops would.
    const F before = unsafeAtomicAdd(static_cast<F*>(bins) + b, (F)1);
    return checked && before == max_value;
  }
  U* p = static_cast<U*>(bins) + b;
  U old = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  while (true) {
    F x;
    __builtin_memcpy(&x, &old, sizeof(F));
    const F y = add_ones<F>(x, c);
    U desired;
    __builtin_memcpy(&desired, &y, sizeof(F));
    if (desired == old) break;  // nothing to store
    if (__hip_atomic_compare_exchange_strong(p, &old, desired, __ATOMIC_RELAXED,
                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      break;
  }
  F before;
  __builtin_memcpy(&before, &old, sizeof(F));
  return checked && before == max_value;
}

__device__ __forceinline__ bool add_to_bin_dyn(int bin_type, void* bins,
                                               int64_t b, uint32_t c,
                                               bool checked) {
  switch (bin_type) {
    case ILGPU_HIP_I32: return add_to_bin<int32_t>(bins, b, c, checked);
    case ILGPU_HIP_U32: return add_to_bin<uint32_t>(bins, b, c, checked);
    case ILGPU_HIP_I64: return add_to_bin<int64_t>(bins, b, c, checked);
    case ILGPU_HIP_F32: return add_to_fp_bin<float, uint32_t>(bins, b, c, checked);
    case ILGPU_HIP_F64: return add_to_fp_bin<double, uint64_t>(bins, b, c, checked);
    default: return add_to_bin<uint64_t>(bins, b, c, checked);
  }
}

// A block's counts, a bin per thread and step, into the bins, which are of type B or, for the unsigned
// types, of the signed one of that size if `is_signed`; returns whether one of the adds passed MaxValue.  Their answers are asked for kFlushSteps adds
// at a time: one add after the other, each a round trip to the memory side, the flush of
// 4096 bins was half of the time of 8 M ints.  Floating-point bins are looked at first: most can
// take a block's count at once (a compare-and-swap loop per bin, which all blocks try at
// about the same time: 8 M ints into 4096 float bins 125 us, now 17.6; 2^26 bytes into 256 4238 / 54.6.)
template <typename B, int BLOCK, int kFlushSteps, typename CountOf>
__device__ __forceinline__ bool flush_bins(void* bins, int num_bins, int first_bin, bool checked, bool is_signed,
                                           const CountOf& count_of) {
  using U = std::conditional_t<sizeof(B) == 4, uint32_t, uint64_t>;
  U* target = static_cast<U*>(bins);
  bool passed = false;
  for (int base = threadIdx.x; base < num_bins; base += kFlushSteps * BLOCK) {
    uint32_t c[kFlushSteps];
    U old[kFlushSteps];
    auto bin_of_step = [&](int s) -> int {
      const int i = base + s * BLOCK;
      return i + first_bin < num_bins ? i + first_bin : i + first_bin - num_bins;
    };
#pragma unroll
    for (int s = 0; s < kFlushSteps; ++s) {
      const int b = bin_of_step(s);
      c[s] = base + s * BLOCK < num_bins ? count_of(b) : 0u;
      old[s] = 0;
      if (c[s] == 0u) continue;
      if constexpr (is_fp<B>::value)
        old[s] = __hip_atomic_load(&target[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      else if (checked)
        old[s] = __hip_atomic_fetch_add(&target[b], (U)c[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      else
        __hip_atomic_fetch_add(&target[b], (U)c[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if constexpr (is_fp<B>::value) {
      B before[kFlushSteps];
#pragma unroll
      for (int s = 0; s < kFlushSteps; ++s) {
        if (c[s] == 0u) continue;
        __builtin_memcpy(&before[s], &old[s], sizeof(B));
        if (before[s] == kOnesEnd<B>)
          c[s] = 0u;  // (All blocks would take it beyond and put it back: 8 M ints into 256 such bins 62 us, so 9.3.)
        else if (ones_are_exact<B>(before[s], c[s]))
          before[s] = unsafeAtomicAdd(static_cast<B*>(bins) + bin_of_step(s), (B)c[s]);
        else
          passed |= add_to_fp_bin<B, U>(bins, bin_of_step(s), c[s], checked), c[s] = 0u;
      }
#pragma unroll
      for (int s = 0; s < kFlushSteps; ++s)
        if (c[s] != 0u) settle_fp_bin<B, U>(static_cast<B*>(bins) + bin_of_step(s), before[s], c[s]);
    } else {
#pragma unroll
      for (int s = 0; s < kFlushSteps; ++s)
        passed |= checked && c[s] != 0u &&
                  (is_signed ? BinTraits<std::make_signed_t<B>>::passes_max((std::make_signed_t<B>)old[s], c[s])
                             : BinTraits<B>::passes_max(old[s], c[s]));
    }
  }
  return passed;
}

// RANGE_CHECK = false when every value of T is a valid bin (e.g. u8 into
// >= 256 bins with the identity locator).  FORM: the plain loop stands by itself, so that
// what the others need costs it no registers (2^30 bytes into 256 bins: 3 %).
enum {
  kFormPlain,       // many replicas
  kFormCrowded,     // looks for waves that meet in one bin
  kFormCrowdedFew,  // the same with at most one block per CU: more loads per thread
  kFormStrided,
};
// Threads of a block: where there is at most one per CU, all that it holds (4096 bins, us with 512 / 1024 threads: 2^24
// ints 18.7 / 17.2, 8 M into int64 bins 17.6 / 15.6).
constexpr int form_block(int form) { return form == kFormCrowdedFew ? ILGPU_HIP_HISTOGRAM_FEW_BLOCK : kBlock; }
template <typename T, int LOC, bool RANGE_CHECK, int FORM>
__global__ __launch_bounds__(form_block(FORM)) void histogram_lds_kernel(
    const T* __restrict__ in, int64_t n, int64_t in_stride, void* bins,
    int num_bins, int bin_type, int32_t* overflow, int replica_shift) {
  using V = typename Vec16<T>::type;
  constexpr int VN = Vec16<T>::N;
  constexpr int kBlock = form_block(FORM);
  extern __shared__ uint32_t s_counts[];
  __shared__ int s_overflow;

  const int words = num_bins << replica_shift;
  for (int i = threadIdx.x; i < words; i += kBlock) s_counts[i] = 0u;
  if (threadIdx.x == 0) s_overflow = 0;
  __syncthreads();

  const uint32_t replica = threadIdx.x & ((1u << replica_shift) - 1u);
  auto count = [&](T v) {
    const int64_t b = locate<T, LOC>(v, num_bins);
    if (!RANGE_CHECK || (uint64_t)b < (uint64_t)num_bins)
      atomicAdd(&s_counts[((uint32_t)b << replica_shift) + replica], 1u);
  };
  // Where most lanes of a wave meet in one bin (a constant column, a sorted one)
  // and fewer than eight replicas part them, the LDS would serve them one after
  // the other: the lanes that agree with the first one are added by one of them
  // instead.  Looked for once per round of vectors.  (A constant column of ints, us
  // with three blocks per CU / with the block limit / with the limit and these
  // sums: 8 M into 4096 bins 22.2 / 33.1 / 17.7, 2^26 into 12 000 229 / 331 / 51.)
  auto crowded = [&](T v) -> bool {
    const int64_t b = locate<T, LOC>(v, num_bins);
    const int first = __builtin_amdgcn_readfirstlane((int)b);
    return __popcll(__ballot((int)b == first)) >= kWaveSize / 2;
  };
  auto count_crowded = [&](T v) {
    const int64_t b = locate<T, LOC>(v, num_bins);
    const bool inside = !RANGE_CHECK || (uint64_t)b < (uint64_t)num_bins;
    const int bin = inside ? (int)b : -1;
    const int first = __builtin_amdgcn_readfirstlane(bin);
    const uint64_t same = __ballot(bin == first);
    uint32_t c = 1u;
    if (bin == first)
      c = (threadIdx.x & (kWaveSize - 1)) == (uint32_t)__builtin_ctzll(same) ? (uint32_t)__popcll(same) : 0u;
    if (inside && c != 0u) atomicAdd(&s_counts[((uint32_t)b << replica_shift) + replica], c);
  };

  const uintptr_t addr = reinterpret_cast<uintptr_t>(in);
  int64_t head = (int64_t)(((16 - (addr & 15)) & 15) / sizeof(T));
  if (head > n) head = n;
  const V* body = reinterpret_cast<const V*>(in + head);
  int64_t nvec = (n - head) / VN;
  int64_t tail_start = head + nvec * VN;

  const int64_t stride = (int64_t)gridDim.x * kBlock;
  int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if constexpr (FORM == kFormStrided) {
    // Stride1D.General with an element stride above one: sample i lives at
    // in[i * in_stride]; one scalar load per sample, no vector body.  Several in
    // flight per thread, since the block limit leaves few waves to hide them (8 M
    // ints into 4096 bins, us with three blocks per CU / one load at a time under
    // the limit / four: every second element 52.1 / 46.7 / 25.2, and of 16 values
    // only 22.9 / 43.7 / 22.1; every fourth 55.0 / 48.2 / 27.5, 29.8 / 45.8 / 25.3).
    int64_t e = i;
    for (; e + (kStridedUnroll - 1) * stride < n; e += kStridedUnroll * stride) {
      T v[kStridedUnroll];
#pragma unroll
      for (int u = 0; u < kStridedUnroll; ++u) v[u] = in[(e + u * stride) * in_stride];
      if (replica_shift <= kCrowdedMaxReplicaShift && crowded(v[0])) {
#pragma unroll
        for (int u = 0; u < kStridedUnroll; ++u) count_crowded(v[u]);
      } else {
#pragma unroll
        for (int u = 0; u < kStridedUnroll; ++u) count(v[u]);
      }
    }
    for (; e < n; e += stride) count(in[e * in_stride]);
    nvec = 0;
    head = 0;
    tail_start = n;
  }
  constexpr int kRound = FORM == kFormCrowdedFew ? kFewUnroll : kUnroll;
  for (; i + (kRound - 1) * stride < nvec; i += kRound * stride) {
    V v[kRound];
#pragma unroll
    for (int u = 0; u < kRound; ++u)
      v[u] = __builtin_nontemporal_load(&body[i + u * stride]);
    if constexpr (FORM != kFormPlain) {
      if (crowded(v[0][0])) {
#pragma unroll
        for (int u = 0; u < kRound; ++u)
#pragma unroll
          for (int k = 0; k < VN; ++k) count_crowded(v[u][k]);
        continue;
      }
    }
#pragma unroll
    for (int u = 0; u < kRound; ++u)
#pragma unroll
      for (int k = 0; k < VN; ++k) count(v[u][k]);
  }
  if constexpr (FORM == kFormCrowdedFew) {
    // What is left, less than a round, is half of a short input here: loaded at once and looked at for crowds like a round.
    // (1024 threads a block left 10^6 ints without a round, and a column of one value without these sums: us before there were so
    // many threads / without this / with it, into 4096 bins 6.9 / 7.9 / 5.5, into 12000 11.5 / 12.3 / 6.6; uniform values 8.1 / 6.45 / 6.45
    // and 17.0 / 10.1 / 10.1, 8 M of them into 4096 16.2 / 11.9 / 11.2.)
    V v[kRound - 1];
#pragma unroll
    for (int u = 0; u < kRound - 1; ++u)
      if (i + u * stride < nvec) v[u] = __builtin_nontemporal_load(&body[i + u * stride]);
#pragma unroll
    for (int u = 0; u < kRound - 1; ++u) {
      if (i + u * stride >= nvec) break;
      if (crowded(v[u][0])) {
#pragma unroll
        for (int k = 0; k < VN; ++k) count_crowded(v[u][k]);
      } else {
#pragma unroll
        for (int k = 0; k < VN; ++k) count(v[u][k]);
      }
    }
    i = nvec;
  }
  for (; i < nvec; i += stride) {
    V v = __builtin_nontemporal_load(&body[i]);
#pragma unroll
    for (int k = 0; k < VN; ++k) count(v[k]);
  }
  if (blockIdx.x == 0) {
    const int64_t extra = head + (n - tail_start);
    if ((int64_t)threadIdx.x < extra) {
      const int64_t idx = (int64_t)threadIdx.x < head
                              ? (int64_t)threadIdx.x
                              : tail_start + ((int64_t)threadIdx.x - head);
      count(in[idx]);
    }
  }
  __syncthreads();

  const bool checked = overflow != nullptr;
  bool passed = false;
  const int replicas = 1 << replica_shift;
  // Blocks start their flush at different bins, in steps of a wave's adds: all of
  // them reach it at about the same time, and in one order every bin would take the
  // adds of all blocks at once.  Not where there are few bins: in two or three
  // steps of the block a rotation gains nothing (2^30 bytes into 256 bins lose 0.8 %
  // by it, 2^26 ints into 1000 2 %).
  const int first_bin =
      FORM == kFormPlain ? 0
                         : (int)((uint64_t)blockIdx.x * (uint32_t)num_bins / gridDim.x) & ~(kWaveSize - 1);
  auto count_of = [&](int b) -> uint32_t {
    uint32_t c = 0;
    // Rotate the start so that neighbouring bins read different banks.
    for (int r = 0; r < replicas; ++r)
      c += s_counts[(b << replica_shift) + ((r + b) & (replicas - 1))];
    return c;
  };
  // (Integer bins one step at a time where there are more blocks than compute units, which hide each other's trips: eight at once
  // cost 2000 int64 bins of 12 * 10^6 ints 24.55 us in place of 23.9, 2^24 into 3000 27.0 in place of 26.6.  And where a thread of the
  // strided form has fewer than eight: every second of 16 * 10^6 ints into 256 bins 27.4 in place of 26.7, into 2000 19.7 in place of
  // 19.1, but into 4096 26.35 in place of 26.6 and into 12000 33.8 in place of 34.7.)
  auto flush = [&](auto one) {
    using B = decltype(one);
    constexpr int kFlushSteps = FORM == kFormPlain || (FORM == kFormCrowded && !is_fp<B>::value) ? 1 : 8;
    auto by = [&](auto steps) {
      passed = flush_bins<B, kBlock, decltype(steps)::value>(
          bins, num_bins, first_bin, checked, bin_type == ILGPU_HIP_I32 || bin_type == ILGPU_HIP_I64, count_of);
    };
    if constexpr (FORM == kFormStrided && !is_fp<B>::value) {
      if (num_bins < kFlushSteps * kBlock) return by(std::integral_constant<int, 1>{});
    }
    by(std::integral_constant<int, kFlushSteps>{});
  };
  if (FORM == kFormPlain && bin_type != ILGPU_HIP_F32 && bin_type != ILGPU_HIP_F64) {
    // (Few bins, of which a thread has one to three: steps cost 2 % of 16 MiB of bytes, and their registers a
    // block per CU of 2^30, 181 -> 250 us.)
    for (int b = threadIdx.x; b < num_bins; b += kBlock) {
      const uint32_t c = count_of(b);
      if (c != 0) passed |= add_to_bin_dyn(bin_type, bins, b, c, checked);
    }
  } else {
    switch (bin_type) {
      case ILGPU_HIP_I32: case ILGPU_HIP_U32: flush(uint32_t{}); break;
      case ILGPU_HIP_F32: flush(float{}); break;
      case ILGPU_HIP_F64: flush(double{}); break;
      default: flush(uint64_t{}); break;
    }
  }
  if (checked) {
    if (passed) s_overflow = 1;
    __syncthreads();
    if (threadIdx.x == 0 && s_overflow)
      __hip_atomic_fetch_or(overflow, 1, __ATOMIC_RELAXED,
                            __HIP_MEMORY_SCOPE_AGENT);
  }
}

// More bins than LDS holds: one global atomic per element, as the reference.
template <typename T, int LOC>
__global__ __launch_bounds__(kBlock) void histogram_global_kernel(
    const T* __restrict__ in, int64_t n, int64_t in_stride, void* bins,
    int64_t num_bins, int bin_type, int32_t* overflow) {
  const bool checked = overflow != nullptr;
  bool passed = false;
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += stride) {
    const int64_t b = locate<T, LOC>(in[i * in_stride], (int)num_bins);
    if ((uint64_t)b < (uint64_t)num_bins)
      passed |= add_to_bin_dyn(bin_type, bins, b, 1u, checked);
  }
  if (checked && __ballot(passed) != 0 && (threadIdx.x & (kWaveSize - 1)) == 0)
    __hip_atomic_fetch_or(overflow, 1, __ATOMIC_RELAXED,
                          __HIP_MEMORY_SCOPE_AGENT);
}

template <typename T> constexpr double type_max_as_double();
template <> constexpr double type_max_as_double<int8_t>() { return 127.0; }
template <> constexpr double type_max_as_double<uint8_t>() { return 255.0; }
template <> constexpr double type_max_as_double<int16_t>() { return 32767.0; }
template <> constexpr double type_max_as_double<uint16_t>() { return 65535.0; }
template <> constexpr double type_max_as_double<int32_t>() { return 2147483647.0; }
template <> constexpr double type_max_as_double<uint32_t>() { return 4294967295.0; }
template <> constexpr double type_max_as_double<int64_t>() { return 9.3e18; }
template <> constexpr double type_max_as_double<uint64_t>() { return 1.9e19; }
template <> constexpr double type_max_as_double<float>() { return 3.5e38; }
template <> constexpr double type_max_as_double<double>() { return 1.7e308; }

template <typename T, int LOC>
int32_t launch_typed(hipStream_t stream, const void* in, int64_t n,
                     int64_t in_stride, void* bins, int64_t num_bins,
                     int32_t bin_type, int32_t* overflow) {
  const T* src = static_cast<const T*>(in);
  const int cus = device_cu_count();
  ProfileScope scope(stream, "histogram");
  if (num_bins > kLdsBudgetWords) {
    int64_t blocks = div_up(n, kBlock);
    if (blocks > (int64_t)cus * 4) blocks = (int64_t)cus * 4;
    hipLaunchKernelGGL((histogram_global_kernel<T, LOC>), dim3((unsigned)blocks),
                       dim3(kBlock), 0, stream, src, n, in_stride, bins,
                       num_bins, bin_type, overflow);
    ILGPU_HIP_CHECK(hipGetLastError());
    return ILGPU_HIP_SUCCESS;
  }
  int shift = 0;
  while ((1 << (shift + 1)) <= kMaxReplicas &&
         (num_bins << (shift + 1)) <= kLdsBudgetWords)
    ++shift;
  const size_t lds_bytes = (size_t)(num_bins << shift) * sizeof(uint32_t);
  const int64_t nvec = n / Vec16<T>::N;
  int64_t blocks = div_up(nvec > 0 ? nvec : 1, kBlock);
  // 160 KiB of LDS per CU: as many resident blocks as fit, at most 3 (every
  // block flushes all of its bins with global atomics at the end: measured
  // 0.165 ms at 2 or 3 blocks per CU against 0.186 at 4 for 2^28 keys into
  // 4096 bins, and 0.182 against 0.188 for 2^30 bytes into 256 bins).
  int64_t per_cu = (int64_t)(160 * 1024) / (int64_t)(lds_bytes + 1024);
  if (per_cu > 3) per_cu = 3;
  if (per_cu < 1) per_cu = 1;
  if (blocks > cus * per_cu) blocks = cus * per_cu;
  // Blocks that are worth their flush (kMinElementsPerBin), in whole rounds of the
  // CUs: 349 blocks over 256 of them took as long as 512 (2^26 ints of 16 values into
  // 12 000 bins 64 us, now 51; 50 with three blocks per CU).
  int64_t worth = std::max<int64_t>(n / (num_bins * kMinElementsPerBin), std::max(cus / kMinBlocksDivisor, 1));
  if (worth > cus) worth = div_up(worth, cus) * cus;
  if (blocks > worth) blocks = worth;
  // Values of T that cannot leave [0, num_bins) need no range check.
  const bool unsigned_small =
      LOC == ILGPU_HIP_LOCATOR_IDENTITY && !(T(-1) < T(0)) &&
      !is_fp<T>::value && type_max_as_double<T>() < (double)num_bins;
  const bool no_check = LOC == ILGPU_HIP_LOCATOR_MODULO ? !is_fp<T>::value
                                                        : unsigned_small;
  // One block per CU, or fewer, is bound by the latency of its loads: four vectors per
  // round and thread (8 M ints into 4096 bins 21.0 -> 19.4 us), but two with more
  // blocks (2^26: 53.9 against 59.5).
  const int form = in_stride != 1                      ? kFormStrided
                   : shift > kCrowdedMaxReplicaShift   ? kFormPlain
                   : blocks <= cus                     ? kFormCrowdedFew
                                                       : kFormCrowded;
  auto launch = [&](auto range_check, auto f) {
    hipLaunchKernelGGL(
        (histogram_lds_kernel<T, LOC, decltype(range_check)::value, decltype(f)::value>),
        dim3((unsigned)blocks), dim3(form_block(decltype(f)::value)), lds_bytes, stream, src, n, in_stride, bins,
        (int)num_bins, bin_type, overflow, shift);
  };
  auto launch_form = [&](auto range_check) {
    if (form == kFormPlain) launch(range_check, std::integral_constant<int, kFormPlain>{});
    else if (form == kFormCrowded) launch(range_check, std::integral_constant<int, kFormCrowded>{});
    else if (form == kFormCrowdedFew) launch(range_check, std::integral_constant<int, kFormCrowdedFew>{});
    else launch(range_check, std::integral_constant<int, kFormStrided>{});
  };
  if (no_check) launch_form(std::false_type{});
  else launch_form(std::true_type{});
  ILGPU_HIP_CHECK(hipGetLastError());
  return ILGPU_HIP_SUCCESS;
}

template <typename T>
int32_t launch_locator(hipStream_t stream, const void* in, int64_t n,
                       int64_t in_stride, void* bins, int64_t num_bins,
                       int32_t bin_type, int32_t locator, int32_t* overflow) {
  switch (locator) {
    case ILGPU_HIP_LOCATOR_IDENTITY:
      return launch_typed<T, ILGPU_HIP_LOCATOR_IDENTITY>(
          stream, in, n, in_stride, bins, num_bins, bin_type, overflow);
    case ILGPU_HIP_LOCATOR_MODULO:
      return launch_typed<T, ILGPU_HIP_LOCATOR_MODULO>(
          stream, in, n, in_stride, bins, num_bins, bin_type, overflow);
    default:
      return ILGPU_HIP_ERROR_NOT_SUPPORTED;
  }
}

}  // namespace

int32_t launch_histogram(hipStream_t stream, const void* in, int64_t n,
                         int64_t in_stride, int32_t in_type, void* bins,
                         int64_t num_bins, int32_t bin_type, int32_t locator,
                         int32_t* overflow) {
#define ILGPU_HIP_HIST_CASE(CODE, T)                                      \
  case CODE:                                                              \
    return launch_locator<T>(stream, in, n, in_stride, bins, num_bins,    \
                             bin_type, locator, overflow)
  switch (in_type) {
    ILGPU_HIP_HIST_CASE(ILGPU_HIP_I8, int8_t);
    ILGPU_HIP_HIST_CASE(ILGPU_HIP_I16, int16_t);
    ILGPU_HIP_HIST_CASE(ILGPU_HIP_I32, int32_t);
    ILGPU_HIP_HIST_CASE(ILGPU_HIP_I64, int64_t);
    ILGPU_HIP_HIST_CASE(ILGPU_HIP_U8, uint8_t);
    ILGPU_HIP_HIST_CASE(ILGPU_HIP_U16, uint16_t);
    ILGPU_HIP_HIST_CASE(ILGPU_HIP_U32, uint32_t);
    ILGPU_HIP_HIST_CASE(ILGPU_HIP_U64, uint64_t);
    ILGPU_HIP_HIST_CASE(ILGPU_HIP_F32, float);
    ILGPU_HIP_HIST_CASE(ILGPU_HIP_F64, double);
    default: return ILGPU_HIP_ERROR_NOT_SUPPORTED;
  }
#undef ILGPU_HIP_HIST_CASE
}

}  // namespace ilgpu_hip
