// scatter_nd for gfx950: data[indices[i, 0..k-1], ...] += updates[i, ...] for every index row i
// (duplicates accumulate), fp32 / fp16 / bf16.
//
// Counterpart of ke_scatter_nd and its host launcher (src/kernels/scatter_nd.cu:10-95).  What
// differs: a slice is read and written with consecutive lanes (the reference walks it serially in
// one thread); duplicates inside a workgroup are added up in fp32 registers before they touch
// memory; the strides travel as kernel arguments (the reference cudaMallocs them per call and never
// frees them); index rows that point outside `data` are skipped instead of written out of bounds.
// `data` outside the device's ordinary memory is added to by compare-and-swap.
//
// What bounds it: atomics on one 128-byte line are served one after another, ~20 ns each (the eight
// L2s are not coherent with each other, so a device-wide atomic is done on the memory side).  With
// indices that repeat as word frequencies do, the most frequent row of 8192 updates is hit ~550
// times.  So a workgroup sorts updates by their rows in LDS and issues ONE hardware atomic
// per word and distinct row (16-bit types: packed pairs; a compare-and-swap loop per element, tried
// first, retries for as long as others win).  8192 bf16 updates of 1024 into 32000 rows, log-uniform
// indices: 2200 to 3000 us with compare-and-swap, 41 with a packed atomic per update and word, 20 with every 64
// updates sorted as they come, 17 with workgroups that own rows (scatter_nd_owner_kernel).
// What is left is the rate of the atomics themselves, ~0.9 TB/s with distinct rows as well.
#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace tfk {
namespace {

constexpr int kMaxRank = 8;
struct Strides {
  long long stride[kMaxRank];  // element stride of the first k dimensions of data
  long long dim[kMaxRank];     // their extents
};

constexpr int kScatterThreads = 256;

// How the words of slices lie.  kPairs: every word holds elements of one slice (always so in fp32).  kSplit: 16-bit
// slices of which a word may hold one half (an odd slice length or an odd start).  kSplitShared: as before, and
// the first or the last word of `data` holds 16 bits that are not its own.  (That check in every atomic's
// way costs up to 8%: 676 fp16 updates of 3755 into 82 rows 10.4 us and 11.3.)
enum class Layout { kPairs, kSplit, kSplitShared };

// One 32-bit word of a slice: an fp32 element or an aligned pair of 16-bit ones.
template <typename T>
struct Word {
  static constexpr int kElems = 4 / (int)sizeof(T);
  float v[kElems];
};

// Adds to one element by compare-and-swap on the aligned word that holds it: in any memory that the device can
// reach, and the other half of the word keeps its bits.
TFK_DEVICE void atomic_add_element(float* p, float v) {
  unsigned* const word = reinterpret_cast<unsigned*>(p);
  unsigned old = *word, seen;
  do {
    seen = old;
    old = atomicCAS(word, seen, __builtin_bit_cast(unsigned, __builtin_bit_cast(float, seen) + v));
  } while (old != seen);
}
template <typename T>
TFK_DEVICE void atomic_add_element(T* p, float v) {
  const size_t at = reinterpret_cast<size_t>(p);
  unsigned* const word = reinterpret_cast<unsigned*>(at & ~size_t(3));
  const int shift = at & 2 ? 16 : 0;
  unsigned old = *word, seen;
  do {
    seen = old;
    const float sum = (float)__builtin_bit_cast(T, (unsigned short)(seen >> shift)) + (float)(T)v;
    const unsigned half = __builtin_bit_cast(unsigned short, (T)sum);
    old = atomicCAS(word, seen, (seen & ~(0xffffu << shift)) | (half << shift));
  } while (old != seen);
}

// Adds `w` to the aligned word at `p` with one hardware atomic.  A 16-bit half that has nothing to
// add passes -0.0, which changes no number; a NaN stays one, but loses its signalling bit.
template <typename T>
TFK_DEVICE void atomic_add_word(T* p, const Word<T>& w) {
  if constexpr (sizeof(T) == 4) {
    unsafeAtomicAdd(p, w.v[0]);
  } else {
    typedef T t2 __attribute__((ext_vector_type(2)));
    typedef short s2 __attribute__((ext_vector_type(2)));
    const t2 x = {(T)w.v[0], (T)w.v[1]};
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (std::is_same_v<T, bf16_t>)
      (void)__builtin_amdgcn_global_atomic_fadd_v2bf16((__attribute__((address_space(1))) s2*)p, __builtin_bit_cast(s2, x));
    else
      (void)__builtin_amdgcn_global_atomic_fadd_v2f16((__attribute__((address_space(1))) half2_t*)p, x);
#endif
  }
}

// The words of one slice's sum that a lane holds: loads and adds, and the atomics.
template <typename T, Layout kLayout>
TFK_DEVICE void add_word_of_slice(Word<T>& sum, const T* src, long long e0, long long slice) {
  constexpr int kElems = Word<T>::kElems;
  if constexpr (kElems == 2 && kLayout == Layout::kPairs) {
    typedef T t2 __attribute__((ext_vector_type(2)));
    if (e0 < slice) {
      const t2 x = *reinterpret_cast<const t2*>(src + e0);
      sum.v[0] += (float)x[0];
      sum.v[1] += (float)x[1];
    }
  } else {
#pragma unroll
    for (int e = 0; e < kElems; ++e)
      if (e0 + e >= 0 && e0 + e < slice) sum.v[e] += (float)src[e0 + e];
  }
}
// Adds word `w` at elements e0 .. of the slice at `dst`, the `at`-th element of `data`.  Of a word that the slice shares with memory outside the `total`
// elements of `data` the other half keeps its bits, whatever they stand for: compare-and-swap.  Only the first
// and the last word of `data` can be such; for every word that two slices share it would cost far too
// much (2048 bf16 updates of 33 into 64 rows 8 us and 40, 30000 of 77 into 131072 rows 25 and 1260).
// kAnyMemory: every element by compare-and-swap.
template <typename T, Layout kLayout, bool kAnyMemory>
TFK_DEVICE void add_to_slice(T* dst, const Word<T>& w, long long e0, long long slice, long long at, long long total) {
  T* const word = dst + e0;
  if constexpr (kAnyMemory) {
#pragma unroll
    for (int e = 0; e < Word<T>::kElems; ++e)
      if (e0 + e >= 0 && e0 + e < slice) atomic_add_element(word + e, w.v[e]);
    return;
  }
  if constexpr (kLayout == Layout::kSplitShared) {
    const int outside = at + e0 < 0 ? 0 : at + e0 + 1 >= total ? 1 : -1;   // element of the word that is not data's
    if (outside >= 0) {
      atomic_add_element(word + (1 - outside), outside ? w.v[0] : w.v[1]);
      return;
    }
  }
  atomic_add_word(word, w);
}
// unless kPairs, a slice may start in the upper half of its first word
template <typename T, Layout kLayout>
TFK_DEVICE int first_word_shift(const T* dst) {
  return kLayout != Layout::kPairs ? (int)((reinterpret_cast<size_t>(dst) / sizeof(T)) % Word<T>::kElems) : 0;
}

// Few updates: a group of `lanes` adjacent lanes (a power of two up to 64) per update, one word per
// lane, no sort.  The call is then the latency of a load of the index, one of the update and an atomic.
// kAnyMemory: `data` is not known to be ordinary memory of this device; any number of updates.
template <typename T, Layout kLayout, bool kAnyMemory>
__global__ __launch_bounds__(kScatterThreads) void scatter_nd_direct_kernel(
    const T* __restrict__ updates, T* __restrict__ data, const long long* __restrict__ indices, Strides s, long long n,
    int k, long long slice, long long total, int lanes) {
  constexpr int kElems = Word<T>::kElems;
  const int lane = threadIdx.x & (lanes - 1);
  long long row = blockIdx.x * (long long)(kScatterThreads / lanes) + threadIdx.x / lanes;
  if (row >= n) return;
  do {
    bool inside = true;
    unsigned long long at = 0;
    for (int j = 0; j < k; ++j) {
      const long long ix = indices[row * k + j];
      inside &= ix >= 0 && ix < s.dim[j];
      at += (unsigned long long)ix * (unsigned long long)s.stride[j];
    }
    if (!inside) continue;
    T* const dst = data + at;
    const int shift = first_word_shift<T, kLayout>(dst);
    const long long step = (long long)gridDim.y * lanes * kElems;
    for (long long e0 = ((long long)blockIdx.y * lanes + lane) * kElems - shift; e0 < slice; e0 += step) {
      Word<T> w;
#pragma unroll
      for (int e = 0; e < kElems; ++e) w.v[e] = -0.f;
      add_word_of_slice<T, kLayout>(w, updates + row * slice, e0, slice);
      add_to_slice<T, kLayout, kAnyMemory>(dst, w, e0, slice, at, total);
    }
  } while (kAnyMemory && (row += gridDim.x * (long long)(kScatterThreads / lanes)) < n);
}

// The next kRows updates per workgroup, as they come; a group of `lanes` adjacent lanes (a power of two up to 64) takes one
// distinct row at a time, kWords words per lane.  Unless kPairs, the halves of words are loaded one by one.
// Scalar registers: with more than 80 a SIMD holds fewer than eight wavefronts, and of workgroups of sixteen a CU
// then holds one instead of two (83: 16598 bf16 updates of 627 into 318 rows 53 us, 78: 35).
template <typename T, int kThreads, int kRows, int kWords, Layout kLayout>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_num_sgpr(80))) void scatter_nd_kernel(
    const T* __restrict__ updates, T* __restrict__ data, const long long* __restrict__ indices, Strides s, long long n,
    int k, long long slice, long long total, int lanes) {
  static_assert((kRows % kWaveSize == 0 || kRows < kWaveSize) && kRows <= kThreads,
                "part of one wavefront or whole wavefronts sort the workgroup's rows");
  constexpr int kElems = Word<T>::kElems;
  constexpr int kSortWaves = (kRows + kWaveSize - 1) / kWaveSize;
  constexpr unsigned long long kOutside = ~0ull;
  constexpr float kLargest = std::is_same_v<T, half_t> ? 65504.f : std::is_same_v<T, bf16_t> ? 0x1.FEp127f : 0x1.FFFFFEp127f;
  __shared__ unsigned long long s_base[kRows];   // element offset of an update's slice in data
  __shared__ unsigned long long s_sorted[kRows];
  __shared__ int s_order[kRows];                 // update numbers in the order of their slices
  __shared__ int s_first[kRows + 1];             // first position of every distinct slice
  __shared__ unsigned long long s_firsts[kSortWaves], s_valid[kSortWaves];
  const int tid = threadIdx.x;
  for (long long row0 = blockIdx.x * (long long)kRows; row0 < n; row0 += gridDim.x * (long long)kRows) {
    unsigned long long base = kOutside;
    if (tid < kRows) {
      if (row0 + tid < n) {
        bool inside = true;
        unsigned long long at = 0;
        for (int j = 0; j < k; ++j) {
          const long long ix = indices[(row0 + tid) * k + j];
          inside &= ix >= 0 && ix < s.dim[j];
          at += (unsigned long long)ix * (unsigned long long)s.stride[j];
        }
        if (inside) base = at;
      }
      s_base[tid] = base;
    }
    __syncthreads();
    if (tid < kRows) {
      int rank = 0;
#pragma unroll 16
      for (int j = 0; j < kRows; ++j) {
        const unsigned long long other = s_base[j];
        rank += other < base || (other == base && j < tid);
      }
      s_order[rank] = tid;
      s_sorted[rank] = base;
    }
    __syncthreads();
    const unsigned long long mine = tid < kRows ? s_sorted[tid] : kOutside;
    const bool first = mine != kOutside && (tid == 0 || s_sorted[tid - 1] != mine);
    if (tid < kRows) {
      const unsigned long long f = __ballot(first), v = __ballot(mine != kOutside);
      if (tid % kWaveSize == 0) {
        s_firsts[tid / kWaveSize] = f;
        s_valid[tid / kWaveSize] = v;
      }
    }
    __syncthreads();
    int count = 0, valid = 0, before = 0;
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) {
      if (w == tid / kWaveSize) before = count + __popcll(s_firsts[w] & ((1ull << (tid % kWaveSize)) - 1));
      count += __popcll(s_firsts[w]);
      valid += __popcll(s_valid[w]);
    }
    if (first) s_first[before] = tid;
    if (tid == 0) s_first[count] = valid;
    __syncthreads();

    const int groups = kThreads / lanes, lane = tid & (lanes - 1);
    const long long words = (slice + kElems - 1 + (kLayout != Layout::kPairs ? 1 : 0)) / kElems;
    for (long long word0 = (long long)blockIdx.y * lanes * kWords + lane; word0 - lane < words;
         word0 += (long long)gridDim.y * lanes * kWords) {
      for (int g = tid / lanes; g < count; g += groups) {
        const int begin = s_first[g], end = s_first[g + 1];
        T* const dst = data + s_sorted[begin];
        const int shift = first_word_shift<T, kLayout>(dst);
        Word<T> sum[kWords];
#pragma unroll
        for (int v = 0; v < kWords; ++v)
#pragma unroll
          for (int e = 0; e < kElems; ++e) sum[v].v[e] = -0.f;
#pragma unroll 2
        for (int p = begin; p < end; ++p) {
          const T* src = updates + (row0 + s_order[p]) * slice;
#pragma unroll
          for (int v = 0; v < kWords; ++v) {
            const long long e0 = (word0 + (long long)v * lanes) * kElems - shift;
            add_word_of_slice<T, kLayout>(sum[v], src, e0, slice);
          }
        }
#pragma unroll
        for (int v = 0; v < kWords; ++v) {
          const long long e0 = (word0 + (long long)v * lanes) * kElems - shift;
          if (e0 >= slice) continue;
          // A sum that T does not hold is added as its single updates, which `data` may bring back into range.
          bool held = true;
#pragma unroll
          for (int e = 0; e < kElems; ++e) held &= __builtin_fabsf(sum[v].v[e]) <= kLargest;
          if (!held) {
            for (int p = begin; p < end; ++p) {
              Word<T> w;
#pragma unroll
              for (int e = 0; e < kElems; ++e) w.v[e] = -0.f;
              add_word_of_slice<T, kLayout>(w, updates + (row0 + s_order[p]) * slice, e0, slice);
              add_to_slice<T, kLayout, false>(dst, w, e0, slice, (long long)s_sorted[begin], total);
            }
            continue;
          }
          add_to_slice<T, kLayout, false>(dst, sum[v], e0, slice, (long long)s_sorted[begin], total);
        }
      }
    }
    __syncthreads();   // the next updates are sorted into the same arrays
  }
}

// Many updates: a workgroup owns a share of the TARGETS (a bucket of a hash of their numbers) and 64 or 128 words of
// their slices, looks through a chunk of 1024 * kMine updates for those of its targets, sorts them by target in LDS and adds them up
// window by window of kWindow updates: one atomic per word and target of a chunk, and one more for every window that a
// target's updates run across, where a workgroup that takes the next 64 updates as they come issues one per word and
// distinct row of those 64 (8192 log-uniform updates of 32000 rows: 3252 distinct rows, 6944 over groups of 64).
// A window is the same work however often its targets repeat, and its loads are all in flight.
// What bounds it: the atomics as before where there are many; below ~4 MB the chain of loading indices, sorting (five
// barriers), loading updates and the atomics, ~6 us.  us, before / now: 8192 bf16 updates of 1024 into 32000 rows 20.5 / 17.2,
// 65536 of 1000 into 131072 194 / 90, 16384 of 4096 into 20000 162 / 62, 49954 fp32 of 622 into 77 145 / 52, 4413 fp32 of 65
// into 72 20.3 / 9; all indices distinct: 8192 of 1024 18.7 / 20, 16384 of 4096 110 / 117 (nothing to merge).
// The sort is by hash, not by number: two targets of one slot may lie mixed, which costs them more
// atomics and nothing else.
constexpr int kOwnerThreads = 1024;
template <typename T, int kMine, int kWords, Layout kLayout>
__global__ __launch_bounds__(kOwnerThreads, 8) void scatter_nd_owner_kernel(
    const T* __restrict__ updates, T* __restrict__ data, const long long* __restrict__ indices, Strides s, long long n,
    int k, long long slice, long long total, int lanes, int bucket_bits, int chunk) {
  constexpr int kElems = Word<T>::kElems;
  constexpr int kChunk = kMine * kOwnerThreads, kSlots = 2 * kOwnerThreads, kSlotShift = 32 - 11;
  constexpr int kWindow = kMine > 2 ? 16 : 8;   // longer where more updates of a target meet
  constexpr int kFlight = kWindow / kWords;     // updates whose loads are in flight
  constexpr float kLargest = std::is_same_v<T, half_t> ? 65504.f : std::is_same_v<T, bf16_t> ? 0x1.FEp127f : 0x1.FFFFFEp127f;
  __shared__ unsigned s_target[kChunk];          // target numbers, sorted
  __shared__ unsigned short s_update[kChunk];    // numbers in the chunk of their updates
  __shared__ int s_slot[kSlots];                 // updates of a slot, then the position of its first
  __shared__ int s_wave[kOwnerThreads / kWaveSize];
  const int tid = threadIdx.x;
  const unsigned bucket = blockIdx.x & ((1u << bucket_bits) - 1);
  const long long row0 = (long long)(blockIdx.x >> bucket_bits) * chunk;
  const long long row_end = std::min(row0 + chunk, n);   // (chunk <= kChunk)

  // ---- this bucket's updates ----
  for (int i = tid; i < kSlots; i += kOwnerThreads) s_slot[i] = 0;
  unsigned target[kMine];
  bool inside[kMine];
#pragma unroll
  for (int j = 0; j < kMine; ++j) {
    target[j] = 0;
    inside[j] = row0 + j * kOwnerThreads + tid < row_end;
  }
  for (int d = 0; d < k; ++d) {
    long long ix[kMine];   // all of them in flight
#pragma unroll
    for (int j = 0; j < kMine; ++j) ix[j] = indices[std::min<long long>(row0 + j * kOwnerThreads + tid, row_end - 1) * k + d];
#pragma unroll
    for (int j = 0; j < kMine; ++j) {
      inside[j] &= ix[j] >= 0 && ix[j] < s.dim[d];
      target[j] += (unsigned)ix[j] * (unsigned)s.stride[d];   // (below 2^32 where inside)
    }
  }
  __syncthreads();
  int rank[kMine];
#pragma unroll
  for (int j = 0; j < kMine; ++j) {
    // (bucket_bits + 11 <= 32; a shift by 32 - 0 is not one)
    const unsigned long long hash = (unsigned long long)(target[j] * 0x9E3779B1u) << bucket_bits;
    inside[j] &= (unsigned)(hash >> 32) == bucket;
    target[j] = inside[j] ? target[j] : 0;
    rank[j] = inside[j] ? atomicAdd(&s_slot[(unsigned)hash >> kSlotShift], 1) : 0;
  }
  __syncthreads();
  // ---- positions of the slots: two slots a thread ----
  const int c0 = s_slot[2 * tid], c1 = s_slot[2 * tid + 1];
  int sum = c0 + c1;
#pragma unroll
  for (int d = 1; d < kWaveSize; d *= 2) {
    const int below = __shfl_up(sum, d);
    if (tid % kWaveSize >= d) sum += below;
  }
  if (tid % kWaveSize == kWaveSize - 1) s_wave[tid / kWaveSize] = sum;
  __syncthreads();
  int before = 0, count = 0;
#pragma unroll
  for (int w = 0; w < kOwnerThreads / kWaveSize; ++w) {
    if (w < tid / kWaveSize) before += s_wave[w];
    count += s_wave[w];
  }
  s_slot[2 * tid] = before + sum - c0 - c1;
  s_slot[2 * tid + 1] = before + sum - c1;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kMine; ++j)
    if (inside[j]) {
      const unsigned hash = (unsigned)((unsigned long long)(target[j] * 0x9E3779B1u) << bucket_bits);
      const int at = s_slot[hash >> kSlotShift] + rank[j];
      s_target[at] = target[j];
      s_update[at] = (unsigned short)(j * kOwnerThreads + tid);
    }
  __syncthreads();

  // ---- windows of sorted updates; a group of `lanes` adjacent lanes takes one at a time, kWords words a lane ----
  const int groups = kOwnerThreads / lanes;
  const long long word0 = (long long)blockIdx.y * lanes * kWords + (tid & (lanes - 1));
  auto first_elem = [&](unsigned t, int v) -> long long {   // element of the slice at word v of this lane
    return (word0 + (long long)v * lanes) * kElems - first_word_shift<T, kLayout>(data + (size_t)t * slice);
  };
  auto load = [&](long long row, long long e0) -> unsigned {
    const T* src = updates + row * slice;
    if constexpr (kLayout == Layout::kPairs) {
      return e0 < slice ? *reinterpret_cast<const unsigned*>(src + e0) : 0u;
    } else {
      // (one load of two elements, at any even address, inside the slice; slice > 1)
      typedef unsigned any_u32 __attribute__((aligned(2)));
      const unsigned w = *reinterpret_cast<const any_u32*>(src + std::min(std::max(e0, 0ll), slice - 2));
      // a half that is not the slice's has nothing to add: -0.0
      return e0 < 0 ? w << 16 | 0x8000u : e0 + 1 < slice ? w : w >> 16 | 0x80000000u;
    }
  };
  auto unpack = [](unsigned w) -> Word<T> {
    Word<T> x;
    if constexpr (kElems == 1) {
      x.v[0] = __builtin_bit_cast(float, w);
    } else {
      x.v[0] = (float)__builtin_bit_cast(T, (unsigned short)w);
      x.v[1] = (float)__builtin_bit_cast(T, (unsigned short)(w >> 16));
    }
    return x;
  };
  for (int first = tid / lanes * kWindow; first < count; first += groups * kWindow) {
    const int end = min(first + kWindow, count);
    Word<T> sum[kWords];
    int from = first;   // of the updates that `sum` holds
    auto clear = [&]() {
#pragma unroll
      for (int v = 0; v < kWords; ++v)
#pragma unroll
        for (int e = 0; e < kElems; ++e) sum[v].v[e] = -0.f;
    };
    clear();
    // adds what `sum` holds of updates [from, to), all of one target
    auto flush = [&](int to) {
      const unsigned t = s_target[from];
      T* const dst = data + (size_t)t * slice;
      const long long at = (long long)((size_t)t * slice);
#pragma unroll
      for (int v = 0; v < kWords; ++v) {
        const long long e0 = first_elem(t, v);
        if (e0 >= slice) continue;
        // A sum that T does not hold is added as its single updates, which `data` may bring back into range.
        bool held = true;
#pragma unroll
        for (int e = 0; e < kElems; ++e) held &= __builtin_fabsf(sum[v].v[e]) <= kLargest;
        if (held) {
          add_to_slice<T, kLayout, false>(dst, sum[v], e0, slice, at, total);
        } else {
          for (int p = from; p < to; ++p)
            add_to_slice<T, kLayout, false>(dst, unpack(load(row0 + s_update[p], e0)), e0, slice, at, total);
        }
      }
      from = to;
      clear();
    };
    for (int p0 = first; p0 < end; p0 += kFlight) {
      unsigned raw[kFlight][kWords];
#pragma unroll
      for (int i = 0; i < kFlight; ++i) {
        const int p = min(p0 + i, end - 1);   // (behind the end: the last update again, not added)
        const unsigned t = s_target[p];
#pragma unroll
        for (int v = 0; v < kWords; ++v) raw[i][v] = load(row0 + s_update[p], first_elem(t, v));
      }
#pragma unroll
      for (int i = 0; i < kFlight; ++i) {
        if (p0 + i < end) {
          if (s_target[p0 + i] != s_target[from]) flush(p0 + i);
#pragma unroll
          for (int v = 0; v < kWords; ++v) {
            const Word<T> x = unpack(raw[i][v]);
#pragma unroll
            for (int e = 0; e < kElems; ++e) sum[v].v[e] += x.v[e];
          }
        }
      }
    }
    flush(end);
  }
}

template <typename T, int kThreads, int kRows, int kWords, Layout kLayout>
int launch_shape(const void* updates, void* data, const long long* indices, const Strides& s, long long n, int k,
                 long long slice, long long total, int lanes, long long words, hipStream_t st) {
  const long long per = (long long)lanes * kWords;
  const dim3 grid((unsigned)std::min<long long>((n + kRows - 1) / kRows, 1 << 20),
                  (unsigned)std::min<long long>((words + per - 1) / per, 1024));
  hipLaunchKernelGGL((scatter_nd_kernel<T, kThreads, kRows, kWords, kLayout>), grid, dim3(kThreads), 0, st,
                     static_cast<const T*>(updates), static_cast<T*>(data), indices, s, n, k, slice, total, lanes);
  TFK_HIP_TRY(hipGetLastError());
  return TF_OK;
}

// As many buckets (a power of two, at least two) as bring about 224 workgroups: one a CU.
template <typename T, int kMine, int kWords, Layout kLayout>
int launch_owner(const void* updates, void* data, const long long* indices, const Strides& s, long long n, int k,
                 long long slice, long long total, int lanes, long long words, hipStream_t st) {
  Strides numbers = s;
  for (int d = 0; d < k; ++d) numbers.stride[d] /= slice;   // the number of a target, not its first element
  const long long chunks = (n + kMine * kOwnerThreads - 1) / (kMine * kOwnerThreads);
  const long long columns = (words + lanes * kWords - 1) / (lanes * kWords);
  int bits = 1;
  while (bits < 8 && chunks * columns * 3 << bits <= 2 * 224) ++bits;
  const int chunk = (int)((n + chunks - 1) / chunks);   // (even ones: no nearly empty last chunk)
  const dim3 grid((unsigned)((n + chunk - 1) / chunk) << bits, (unsigned)columns);
  hipLaunchKernelGGL((scatter_nd_owner_kernel<T, kMine, kWords, kLayout>), grid, dim3(kOwnerThreads), 0, st,
                     static_cast<const T*>(updates), static_cast<T*>(data), indices, numbers, n, k, slice, total, lanes, bits,
                     chunk);
  TFK_HIP_TRY(hipGetLastError());
  return TF_OK;
}

template <typename T, Layout kLayout, bool kAnyMemory>
int launch_direct(const void* updates, void* data, const long long* indices, const Strides& s, long long n, int k,
                  long long slice, long long total, int lanes, long long words, hipStream_t st) {
  const int per = kScatterThreads / lanes;
  const dim3 grid((unsigned)std::min<long long>((n + per - 1) / per, 1 << 20),
                  (unsigned)std::min<long long>((words + lanes - 1) / lanes, 1024));
  hipLaunchKernelGGL((scatter_nd_direct_kernel<T, kLayout, kAnyMemory>), grid, dim3(kScatterThreads), 0, st,
                     static_cast<const T*>(updates), static_cast<T*>(data), indices, s, n, k, slice, total, lanes);
  TFK_HIP_TRY(hipGetLastError());
  return TF_OK;
}

// Hardware floating-point atomics are defined for ordinary (coarse-grained) memory of the device that runs the kernel:
// on host, managed or fine-grained memory an update may be lost.
bool is_ordinary_device_memory(const void* p) {
  int device = -1;
  hipPointerAttribute_t a{};
  if (hipGetDevice(&device) != hipSuccess || hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();   // not an error of this call
    return false;
  }
  return a.type == hipMemoryTypeDevice && !a.isManaged && a.device == device && a.allocationFlags == hipDeviceMallocDefault;
}

template <typename T, Layout kLayout>
int launch_rows(const void* updates, void* data, const long long* indices, const Strides& s, long long n, int k,
                long long slice, long long targets, int lanes, long long words, hipStream_t st) {
  if (!is_ordinary_device_memory(data))
    return launch_direct<T, kLayout, true>(updates, data, indices, s, n, k, slice, slice * targets, lanes, words, st);
  // Times in us with log-uniform indices.  Few updates: no sort (806 of 34 fp32: direct 3.3, 16 of 256 threads' updates
  // sorted 5.6).  From 1024 on contention shows (2048 of 64 bf16 into 64 rows: direct 10.8, sorted 6.3).
  if (n <= 1024)
    return launch_direct<T, kLayout, false>(updates, data, indices, s, n, k, slice, slice * targets, lanes, words, st);
  // Beyond, owners of targets, except: a few 16-bit updates (1489 of 1206 bf16 into 1412 rows: 9.4 sorted by 16, 10.4 by
  // owners; 1894 of 3924 21.8 and 14.6; 1077 fp32 of 26 into 95 5.6 and 6.1, 1469 of 68 into 350 8.1 and 6.9), and narrow slices whose targets are hit often, for which the sort of the next 128
  // finds as much to merge (58345 of 55 fp16 into 306 rows: 42 and 54).  (Target numbers are 32 bits there.)
  const bool owners_fit = targets < (1ll << 32) && n < (1ll << 31) && (kLayout == Layout::kPairs || slice > 1) &&
                          words <= 1024ll * lanes;
  if ((n <= 2048 && ((sizeof(T) == 2 && n * words < 2 << 20) || !owners_fit)) || n <= 1280)
    return launch_shape<T, 256, 16, 1, kLayout>(updates, data, indices, s, n, k, slice, slice * targets, lanes, words, st);
  if (!owners_fit || (words <= 32 && n > 8192 && n / 16 >= targets))
    return launch_shape<T, 1024, 128, 2, kLayout>(updates, data, indices, s, n, k, slice, slice * targets, lanes, words, st);
  // Longer chunks find more to merge and cost workgroups (16384 bf16 of 4096 into 20000 rows: 2048 updates a chunk 72,
  // 8192 61; 8192 of 1024 into 32000 17.2 and 19.2); unpaired halves lose by them (45202 bf16 of 365 into 64 rows 49, 92).
  // Two words a lane, likewise, halve the workgroups that look through the same indices, from 256 words on.
  auto owners = [&](auto mine, auto per_lane) -> int {
    return launch_owner<T, decltype(mine)::value, decltype(per_lane)::value, kLayout>(
        updates, data, indices, s, n, k, slice, slice * targets, lanes, words, st);
  };
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  if constexpr (kLayout == Layout::kPairs) {
    using Eight = std::integral_constant<int, 8>;
    if (n >= 20000) return words > 256 ? owners(Eight{}, Two{}) : owners(Eight{}, One{});
    if (words > 256) return owners(Two{}, Two{});
  }
  return owners(Two{}, One{});
}

template <typename T>
int launch(const void* updates, void* data, const long long* indices, const Strides& s, long long n, int k,
           long long slice, long long targets, hipStream_t st) {
  constexpr int kElems = Word<T>::kElems;
  // slices whose words are pairs of one slice in both arrays; otherwise a slice may take one word more
  const bool pairs = kElems == 1 || (slice % 2 == 0 && reinterpret_cast<size_t>(updates) % 4 == 0 &&
                                     reinterpret_cast<size_t>(data) % 4 == 0);
  const long long words = (slice + kElems - 1 + (pairs ? 0 : 1)) / kElems;
  int lanes = 1;
  while (lanes < kWaveSize && lanes < words) lanes *= 2;
  if constexpr (kElems == 2) {
    const size_t first = reinterpret_cast<size_t>(data), behind = first + (size_t)(slice * targets) * sizeof(T);
    if (!pairs && (first % 4 != 0 || behind % 4 != 0))
      return launch_rows<T, Layout::kSplitShared>(updates, data, indices, s, n, k, slice, targets, lanes, words, st);
    if (!pairs) return launch_rows<T, Layout::kSplit>(updates, data, indices, s, n, k, slice, targets, lanes, words, st);
  }
  return launch_rows<T, Layout::kPairs>(updates, data, indices, s, n, k, slice, targets, lanes, words, st);
}

}  // namespace
}  // namespace tfk

extern "C" int tf_scatter_nd(const void* updates, void* data, const int64_t* indices, const int64_t* data_dims,
                             int rank, int64_t num_index_rows, int index_depth, int dtype, void* stream) {
  using namespace tfk;
  TFK_REQUIRE(updates && data && indices && data_dims, TF_ERR_INVALID_ARG, "tf_scatter_nd: null pointer");
  TFK_REQUIRE(rank >= 1 && rank <= kMaxRank, TF_ERR_INVALID_ARG, "tf_scatter_nd: rank %d outside 1..%d", rank,
              kMaxRank);
  TFK_REQUIRE(index_depth >= 1 && index_depth <= rank, TF_ERR_INVALID_ARG,
              "tf_scatter_nd: index depth %d outside 1..rank (%d)", index_depth, rank);
  TFK_REQUIRE(num_index_rows >= 0, TF_ERR_INVALID_ARG, "tf_scatter_nd: negative number of index rows");
  TFK_REQUIRE(dtype >= 0 && dtype <= 2, TF_ERR_UNSUPPORTED, "tf_scatter_nd: dtype %d (0 f32, 1 f16, 2 bf16)", dtype);
  Strides s{};
  long long stride = 1, targets = 1;
  for (int i = rank - 1; i >= 0; --i) {
    TFK_REQUIRE(data_dims[i] > 0, TF_ERR_INVALID_ARG, "tf_scatter_nd: data dimension %d is not positive", i);
    if (i < index_depth) {
      s.stride[i] = stride;
      s.dim[i] = data_dims[i];
      targets *= data_dims[i];
    }
    stride *= data_dims[i];
  }
  long long slice = 1;
  for (int i = index_depth; i < rank; ++i) slice *= data_dims[i];
  if (num_index_rows == 0) return TF_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const long long* idx = reinterpret_cast<const long long*>(indices);
  if (dtype == 0) return launch<float>(updates, data, idx, s, num_index_rows, index_depth, slice, targets, st);
  if (dtype == 1) return launch<half_t>(updates, data, idx, s, num_index_rows, index_depth, slice, targets, st);
  return launch<bf16_t>(updates, data, idx, s, num_index_rows, index_depth, slice, targets, st);
}
