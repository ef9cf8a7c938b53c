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
// indices: 2200 to 3000 us with compare-and-swap, 41 with a packed atomic per update and word, 21 with every 64
// updates sorted as they come, 17 with chunks sorted whole (scatter_nd_owner_kernel).
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

// Many updates: every workgroup of a chunk of 1024 * kMine updates sorts the chunk by target in LDS, into slots of a hash,
// and owns some of them and 64 or 128 words of their slices, which it adds up window by window of kWindow updates: one
// atomic per word and target of a window.  A window is the same work however often its targets repeat, and its loads are
// all in flight.
//
// Who owns what must come out alike in every workgroup: the order of updates within a slot does not (it is that of LDS atomics).
// So a slot belongs whole to the share of the sorted positions in which it begins, and the updates of a hot slot (a
// twelfth of the chunk or more), which would keep its owner busy behind all others, go by their numbers in the chunk.
// Windows of one target that follow each other are added up in LDS before they leave, up to 16 of them, with the updates of it
// that the next window begins with.  That is for speed (atomics on one line are served one after another: 14576 bf16 of 218 into 7
// rows 13.9 and, with those, 11.7 us) and for the sum: a 16-bit target of many updates is rounded with every atomic.  (With a hash to pick the owner and 8 updates an atomic, all of 8192 x 1024 bf16 into
// one row took 50 us and came out at half its value; 12 us and 0.2% as here; every 64 as they come 18.6, 1.2%.)
//
// What bounds it: the atomics where there are many; below ~4 MB the chain of loading indices, sorting (five barriers,
// an LDS atomic per update in every workgroup), loading updates and the atomics, ~6 us.  us, log-uniform indices, sorted
// 64 or 128 as they come / hash owners / as here: 8192 bf16 of 1024 into 32000 rows 20.8 / 16.8 / 14.9, 65536 of 1000 into
// 131072 187 / 90 / 96, 16384 of 4096 into 20000 158 / 74 / 69, 60000 of 40 into 131072 35.9 / 26.6 / 12.8, 49954 fp32 of 622
// into 77 154 / 60 / 44; all indices distinct: 8192 of 1024 20.1 / 22.5 / 21.1, 32768 fp16 of 512 32.9 / 39.7 / 35.4; half
// of them one row: 8192 of 1024 20.5 / 34.5 / 18.2, 60000 of 40 23.2 / 74.9 / 18.6; all: 18.7 / 50.3 / 13.1, 25.4 / 136 / 15.7.
// Two targets of one slot may lie mixed, which costs them more atomics and nothing else.  kSingle: 16-bit slices of one element.
constexpr int kOwnerThreads = 1024;
template <typename T, int kMine, int kWords, Layout kLayout, bool kSingle>
__global__ __launch_bounds__(kOwnerThreads, 8) void scatter_nd_owner_kernel(
    const T* __restrict__ updates, T* __restrict__ data, const long long* __restrict__ indices, Strides s, long long n,
    int k, long long slice, long long total, int lanes, int share_bits, int chunk) {
  constexpr int kElems = Word<T>::kElems;
  constexpr int kChunk = kMine * kOwnerThreads, kSlots = 2 * kOwnerThreads, kSlotShift = 32 - 11;
  constexpr int kWindow = kMine > 2 ? 16 : 8;   // longer where more updates of a target meet
  constexpr int kFlight = kWindow / kWords;     // updates whose loads are in flight
  constexpr int kHotSlots = 12, kHot = kChunk / kHotSlots;   // a hot slot has kHot updates or more
  constexpr int kLinks = 16;                    // windows of one target that are added up before they leave
  constexpr float kLargest = std::is_same_v<T, half_t> ? 65504.f : std::is_same_v<T, bf16_t> ? 0x1.FEp127f : 0x1.FFFFFEp127f;
  __shared__ unsigned s_target[kChunk];          // target numbers of this workgroup's updates, sorted
  __shared__ unsigned short s_update[kChunk];    // numbers in the chunk of these updates
  __shared__ int s_slot[kSlots];                 // updates of a slot; then the position of its first, or -1 - number of a hot slot
  __shared__ int s_hot[kHotSlots];               // this workgroup's updates of a hot slot
  __shared__ int s_wave[kOwnerThreads / kWaveSize];
  __shared__ int s_hots;                         // number of hot slots
  __shared__ bool s_links;                       // windows of one target may follow each other here
  __shared__ int s_front, s_end;                 // positions of the first slot of this workgroup and behind its last one
  __shared__ alignas(16) bool s_linked[kOwnerThreads];
  __shared__ unsigned char s_leading[kOwnerThreads];           // updates of a window that it leaves to the one in front
  __shared__ float s_lead[kWords * kElems * kOwnerThreads];    // their sums
  const int tid = threadIdx.x;
  const int shares = 1 << share_bits, share = blockIdx.x & (shares - 1);
  const long long row0 = (long long)(blockIdx.x >> share_bits) * chunk;
  const long long row_end = std::min(row0 + chunk, n);   // (chunk <= kChunk)

  // ---- updates of every slot ----
  for (int i = tid; i < kSlots; i += kOwnerThreads) s_slot[i] = 0;
  if (tid < kHotSlots) s_hot[tid] = 0;
  if (tid == 0) {
    s_hots = s_front = s_end = 0;
    s_links = false;
  }
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
  auto slot_of = [](unsigned t) { return (t * 0x9E3779B1u) >> kSlotShift; };
  int rank[kMine];   // (in the order of arrival: another one in every workgroup)
#pragma unroll
  for (int j = 0; j < kMine; ++j) rank[j] = inside[j] ? atomicAdd(&s_slot[slot_of(target[j])], 1) : 0;
  __syncthreads();
  // ---- positions of the slots, the hot ones left out: two slots a thread ----
  const int c0 = s_slot[2 * tid], c1 = s_slot[2 * tid + 1];
  const int n0 = c0 < kHot ? c0 : 0, n1 = c1 < kHot ? c1 : 0;
  int sum = n0 + n1;
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
  // this workgroup has the slots that begin at positions [begin, behind)
  const int per_share = (((count + shares - 1) >> share_bits) + kWindow - 1) / kWindow * kWindow;
  const int begin = share * per_share, behind = min(begin + per_share, count);
  auto place = [&](int slot, int c, int n_slot, int pos) {
    s_slot[slot] = c < kHot ? pos : -1 - atomicAdd(&s_hots, 1);
    // (the exchange costs 2 * kWords barriers: below four windows a word, the atomics that it saves cost less)
    if (pos >= begin && pos < behind && n_slot >= 4 * kWords * kWindow) s_links = true;
    if (pos < begin && begin <= pos + n_slot) s_front = pos + n_slot;
    if (pos < behind && behind <= pos + n_slot) s_end = pos + n_slot;
  };
  place(2 * tid, c0, n0, before + sum - n0 - n1);
  place(2 * tid + 1, c1, n1, before + sum - n1);
  __syncthreads();
  const bool links = s_links || s_hots > 0;
  const int hots = s_hots, front = s_front, own = begin < count ? s_end - front : 0;
  // ... and of the hot ones the updates [share * per_hot, (share + 1) * per_hot) of the chunk.  These come first: their runs are
  // cut as seldom as can be, and leave no small rest that a large target would round away.
  int base = 0;
  if (hots > 0) {
    const int per_hot = (((chunk + shares - 1) >> share_bits) + kLinks * kWindow - 1) / (kLinks * kWindow) * (kLinks * kWindow);
#pragma unroll
    for (int j = 0; j < kMine; ++j) {
      const int pos = inside[j] ? s_slot[slot_of(target[j])] : 0;
      if (pos < 0) rank[j] = (j * kOwnerThreads + tid) / per_hot == share ? atomicAdd(&s_hot[-1 - pos], 1) : -1;
    }
    __syncthreads();
    for (int h = 0; h < hots; ++h) base += s_hot[h];
  }
#pragma unroll
  for (int j = 0; j < kMine; ++j) {
    if (!inside[j] || rank[j] < 0) continue;
    const int pos = s_slot[slot_of(target[j])];
    int at = rank[j];
    if (pos >= 0) {
      if (pos < begin || pos >= behind) continue;
      at += base + pos - front;
    } else {
      for (int h = 0; h < -1 - pos; ++h) at += s_hot[h];
    }
    s_target[at] = target[j];
    s_update[at] = (unsigned short)(j * kOwnerThreads + tid);
  }
  __syncthreads();
  const int stop = base + own;

  // ---- windows of sorted updates; a group of `lanes` adjacent lanes takes one at a time, kWords words a lane ----
  const int groups = kOwnerThreads / lanes, group = tid / lanes;
  const int len = (int)slice;   // (at most 65536 words)
  const int word0 = (int)blockIdx.y * lanes * kWords + (tid & (lanes - 1));
  auto first_elem = [&](unsigned t, int v) -> int {   // element of the slice at word v of this lane
    return (word0 + v * lanes) * kElems - first_word_shift<T, kLayout>(data + (size_t)t * slice);
  };
  auto load = [&](long long row, int e0) -> unsigned {
    const T* src = updates + row * slice;
    if constexpr (kLayout == Layout::kPairs) {
      return e0 < len ? *reinterpret_cast<const unsigned*>(src + e0) : 0u;
    } else {
      // a half that is not the slice's has nothing to add: -0.0
      if constexpr (kSingle) {
        const unsigned w = *reinterpret_cast<const unsigned short*>(src);
        return e0 < 0 ? w << 16 | 0x8000u : w | 0x80000000u;
      }
      // (one load of two elements, at any even address, inside the slice)
      typedef unsigned any_u32 __attribute__((aligned(2)));
      const unsigned w = *reinterpret_cast<const any_u32*>(src + std::min(std::max(e0, 0), len - 2));
      return e0 < 0 ? w << 16 | 0x8000u : e0 + 1 < len ? w : w >> 16 | 0x80000000u;
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
  for (int round = 0; round < stop; round += groups * kWindow) {
    const int first = round + group * kWindow, end = min(first + kWindow, stop);
    Word<T> sum[kWords];
    int from = first;   // of the updates that `sum` holds
    auto clear = [&]() {
#pragma unroll
      for (int v = 0; v < kWords; ++v)
#pragma unroll
        for (int e = 0; e < kElems; ++e) sum[v].v[e] = -0.f;
    };
    clear();
    // This window's first target is the last one of the window in front, whose group takes the sums of both.
    const bool led = links && first < end && group % kLinks != 0 && s_target[first - 1] == s_target[first];
    int leading = 0;   // updates of it, where another target follows here
    // adds what `sum` holds of updates [from, to), all of one target
    auto flush = [&](int to) {
      const unsigned t = s_target[from];
      T* const dst = data + (size_t)t * slice;
      const long long at = (long long)((size_t)t * slice);
#pragma unroll
      for (int v = 0; v < kWords; ++v) {
        const int e0 = first_elem(t, v);
        if (e0 >= len) continue;
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
          if (s_target[p0 + i] != s_target[from]) {
            if (led && from == first) {
#pragma unroll
              for (int v = 0; v < kWords; ++v)
#pragma unroll
                for (int e = 0; e < kElems; ++e) s_lead[(v * kElems + e) * kOwnerThreads + tid] = sum[v].v[e];
              from = p0 + i;
              leading = from - first;
              clear();
            } else {
              flush(p0 + i);
            }
          }
#pragma unroll
          for (int v = 0; v < kWords; ++v) {
            const Word<T> x = unpack(raw[i][v]);
#pragma unroll
            for (int e = 0; e < kElems; ++e) sum[v].v[e] += x.v[e];
          }
        }
      }
    }
    const bool linked = led && from == first;   // all of it is of the target in front
    int last = end;
    if (links) {
      if ((tid & (lanes - 1)) == 0) {
        s_linked[group] = linked;
        s_leading[group] = (unsigned char)leading;
      }
      float* const sums = reinterpret_cast<float*>(s_slot) + tid;
      int follow = 0, behind_them = 0;   // linked windows that follow this one, leading updates of the next
#pragma unroll
      for (int v = 0; v < kWords; ++v) {
        if (linked) {
#pragma unroll
          for (int e = 0; e < kElems; ++e) sums[e * kOwnerThreads] = sum[v].v[e];
        }
        __syncthreads();
        if (v == 0) {
          const uint4_t flags = *reinterpret_cast<const uint4_t*>(s_linked + group / kLinks * kLinks);
          unsigned bits = 0;   // of the kLinks windows around this one
#pragma unroll
          for (int w = 0; w < 4; ++w) bits |= ((flags[w] * 0x10204080u) >> 28) << (4 * w);
          follow = linked ? 0 : __builtin_ctz(~(bits >> (group % kLinks + 1)));
          if (!linked && group % kLinks + follow + 1 < kLinks) behind_them = s_leading[group + follow + 1];
          last = min(end + follow * kWindow, stop) + behind_them;
        }
        for (int h0 = 0; h0 < follow; h0 += 4) {
          float more[4][kElems];
#pragma unroll
          for (int h = 0; h < 4; ++h)
#pragma unroll
            for (int e = 0; e < kElems; ++e) more[h][e] = sums[e * kOwnerThreads + min(h0 + h + 1, follow) * lanes];
#pragma unroll
          for (int h = 0; h < 4; ++h)
#pragma unroll
            for (int e = 0; e < kElems; ++e) sum[v].v[e] += h0 + h < follow ? more[h][e] : -0.f;
        }
        if (behind_them > 0) {
#pragma unroll
          for (int e = 0; e < kElems; ++e) sum[v].v[e] += s_lead[(v * kElems + e) * kOwnerThreads + tid + (follow + 1) * lanes];
        }
        __syncthreads();
      }
    }
    if (first < end && !linked) flush(last);
  }
}

template <typename T, int kThreads, int kRows, int kWords, Layout kLayout>
int launch_shape(const void* updates, void* data, const long long* indices, const Strides& s, long long n, int k,
                 long long slice, long long total, int lanes, long long words, hipStream_t st) {
  const long long per = (long long)lanes * kWords;
  const dim3 grid((unsigned)std::min<long long>((n + kRows - 1) / kRows, 1 << 20),
                  (unsigned)std::min<long long>((words + per - 1) / per, 1024));
  return launch_kernel(scatter_nd_kernel<T, kThreads, kRows, kWords, kLayout>, grid, dim3(kThreads), 0, st,
                       static_cast<const T*>(updates), static_cast<T*>(data), indices, s, n, k, slice, total, lanes);
}

// As many shares (a power of two, at least two) as bring about 224 workgroups: one a CU.  Twice as many, two a CU, for chunks of
// 4096 and two words a lane, which have the most loads to wait for: us, one / two, 20837 fp32 of 2166 into 901 rows 75 / 59, 62413 of 994
// into 1447 98 / 82, 27577 fp16 of 1990 into 35292 (uniform) 118 / 116; not beyond 512, which the chip does not hold at once (528: 22339 fp16 of 2710
// 83 / 99), nor with shorter chunks (0-12% behind).
struct OwnerGrid {
  long long chunks, columns;
  int bits;   // of the shares of a chunk
};
OwnerGrid owner_grid(long long n, long long words, int lanes, int mine, int per_lane) {
  OwnerGrid g;
  g.chunks = (n + mine * kOwnerThreads - 1) / (mine * kOwnerThreads);
  g.columns = (words + lanes * per_lane - 1) / (lanes * per_lane);
  g.bits = 1;
  while (g.bits < 8 && g.chunks * g.columns * 3 << g.bits <= 2 * 224) ++g.bits;
  if (mine == 4 && per_lane == 2 && g.bits < 8 && g.chunks * g.columns << g.bits <= 256) ++g.bits;
  return g;
}

template <typename T, int kMine, int kWords, Layout kLayout, bool kSingle>
int launch_owner(const void* updates, void* data, const long long* indices, const Strides& s, long long n, int k,
                 long long slice, long long total, int lanes, long long words, hipStream_t st) {
  Strides numbers = s;
  for (int d = 0; d < k; ++d) numbers.stride[d] /= slice;   // the number of a target, not its first element
  const auto [chunks, columns, bits] = owner_grid(n, words, lanes, kMine, kWords);
  const int chunk = (int)((n + chunks - 1) / chunks);   // (even ones: no nearly empty last chunk)
  const dim3 grid((unsigned)((n + chunk - 1) / chunk) << bits, (unsigned)columns);
  return launch_kernel(scatter_nd_owner_kernel<T, kMine, kWords, kLayout, kSingle>, grid, dim3(kOwnerThreads), 0, st,
                       static_cast<const T*>(updates), static_cast<T*>(data), indices, numbers, n, k, slice, total, lanes, bits,
                       chunk);
}

template <typename T, Layout kLayout, bool kAnyMemory>
int launch_direct(const void* updates, void* data, const long long* indices, const Strides& s, long long n, int k,
                  long long slice, long long total, int lanes, long long words, hipStream_t st) {
  const int per = kScatterThreads / lanes;
  const dim3 grid((unsigned)std::min<long long>((n + per - 1) / per, 1 << 20),
                  (unsigned)std::min<long long>((words + lanes - 1) / lanes, 1024));
  return launch_kernel(scatter_nd_direct_kernel<T, kLayout, kAnyMemory>, grid, dim3(kScatterThreads), 0, st,
                       static_cast<const T*>(updates), static_cast<T*>(data), indices, s, n, k, slice, total, lanes);
}

// What a call whose `data` is ordinary memory runs.  chunk: updates that are sorted together, 0: none, each goes straight to memory.
// owners: by the owners' kernel, otherwise (chunk > 0) by workgroups of `threads`.  per_lane: words of an update that a lane has.
struct ScatterPlan {
  int chunk, threads, per_lane;
  bool owners;
};

// Times in us, log-uniform indices where no others are named.  The host does not see the indices: a form is taken only where none of
// log-uniform, uniform, distinct, evenly repeated and sorted ones, all of them one row or half of them, loses more than 6% by it.
ScatterPlan plan_scatter(int elem_bytes, Layout layout, long long n, long long targets, long long words, int lanes) {
  auto owners = [](int mine, int per_lane) { return ScatterPlan{mine * kOwnerThreads, kOwnerThreads, per_lane, true}; };
  const bool pairs = layout == Layout::kPairs;
  // What the target numbers (32 bits) and columns of sorted chunks do not hold: 2100 bf16 of 140000 into 300 rows 364 sorted by 64, 527 by
  // 128, all to one row 591 and 2010.
  const bool chunks_fit = targets < (1ll << 32) && n < (1ll << 31) && words <= 1024ll * lanes;
  // Few but wide updates, where the atomics are what counts: sorted by the chunk where targets repeat twice on average, from 1.5 Mi words on
  // (3 Mi in place of the sorted 16 below), and from 16 Mi on, where the sort is little beside the rest. The time of the other form / so: 214
  // fp32 of 12266 into 67 rows 16.5 / 10.0, 598 of 5653 into 73 21.9 / 12.6, uniform 19.0 / 10.2, 1138 fp16 of 12030 into 266 32.2 / 20.1; 836
  // fp16 of 41838 into 894 84 / 42, distinct 76 / 74. Over 109 problems 0.51, distinct 0.89, 1.02 at most in any order. Not elsewhere: 407 bf16
  // of 10096 into 3872 12.0 / 10.7, but distinct 10.6 / 12.6; fewer than 128 updates 40 fp32 of 45341 into 3502 9.5 / 19.1.
  const bool few_wide = pairs && chunks_fit && words > 256 && n >= 128 && n <= 1280 &&
                        (n * words >= 16 << 20 || (n / 2 >= targets && n * words >= (n > 1024 ? 3 << 20 : 3 << 19)));
  if (few_wide) return owners(n <= 1024 ? 1 : 2, 1);
  // Few updates: no sort (806 of 34 fp32: direct 3.3, 16 of 256 threads' updates sorted 5.6).  From 1024 on contention shows (2048 of 64
  // bf16 into 64 rows: direct 10.8, sorted 6.3).
  if (n <= 1024) return {0, kScatterThreads, 1, false};
  // Beyond, chunks sorted whole, except a few 16-bit updates: 1894 of 3924 21.8 sorted by 16, 14.6 by the chunk; 1077 fp32 of 26 into 95 5.6 and
  // 6.1, 1469 of 68 into 350 8.1 and 6.9.  (Wide 16-bit ones of less than 2 Mi words: 1791 bf16 of 1264 into 3285 10.0 and 8.1, but
  // distinct 8.1 and 9.4, sorted indices 8.1 and 10.2.)
  if ((n <= 2048 && ((elem_bytes == 2 && n * words < 2 << 20) || !chunks_fit)) || n <= 1280) return {16, 256, 1, false};
  if (!chunks_fit) {
    // Every target hit at least eight times on average: the deeper sort.  A workgroup of eight wavefronts hides its own
    // latencies where there are few of them, enough of four do it better.
    if (n / 8 >= targets) return {128, 1024, 2, false};
    return {64, (n / 64) * ((words + lanes - 1) / lanes) < 1024 ? 512 : 256, 1, false};
  }
  if (!pairs) return owners(2, 1);
  // Longer chunks find more to merge, shorter ones are sorted sooner, in every workgroup.  4096 updates instead of 2048 from
  // 20000 on (40000 bf16 of 1000 into 131072 rows 80 and 67, distinct indices 83 and 85; 8192 a chunk 69 and 88), 1024 where there are
  // few (4096 fp32 of 64 into 8000 rows 7.7 and 7.1).
  if (words <= 256) return owners(n >= 20000 ? 4 : n > 8192 ? 2 : 1, 1);
  // Two words a lane halve the workgroups that sort the same indices, but one wavefront then waits for twice the loads and atomics.  So a word
  // a lane up to 4096 updates (3873 fp16 of 1048 into 2024 12.6 and 13.3 with two), and up to 512 words where that is a workgroup on every CU and
  // eight or more to a chunk: 8192 bf16 of 1024 into 32000 18.2 with two and 14.9, distinct 20.7 and 21.1; over 19 problems 0.81 of the
  // time, uniform 0.92, distinct 0.94, all of them one row 0.81, half of them 0.78, sorted 0.95, 1.06 at most in any order. Elsewhere it
  // loses where rows repeat: 9604 fp32 of 696 into 2760 21.9 and 19.0, all one row 15.5 and 18.6, sorted 21.1 and 24.3. (4096 a
  // chunk and a word a lane: 5032 fp16 of 1162 into 890 14.6 and 14.3, all one row 11.8 and 17.0.)
  if (n >= 20000) return owners(4, 2);
  const OwnerGrid g = owner_grid(n, words, lanes, 2, 1);
  const long long all = g.chunks * g.columns << g.bits;
  return owners(2, n <= 4096 || (words <= 512 && g.bits >= 3 && all >= 224 && all <= 256) ? 1 : 2);
}

template <typename T, Layout kLayout>
int launch_rows(const void* updates, void* data, const long long* indices, const Strides& s, long long n, int k,
                long long slice, long long targets, int lanes, long long words, hipStream_t st) {
  // (floating-point atomics may lose an update elsewhere)
  if (!is_ordinary_device_memory(data))
    return launch_direct<T, kLayout, true>(updates, data, indices, s, n, k, slice, slice * targets, lanes, words, st);
  const ScatterPlan plan = plan_scatter(sizeof(T), kLayout, n, targets, words, lanes);
  if (plan.owners) {
    auto owners = [&](auto mine, auto per_lane, auto single) -> int {
      return launch_owner<T, decltype(mine)::value, decltype(per_lane)::value, kLayout, decltype(single)::value>(
          updates, data, indices, s, n, k, slice, slice * targets, lanes, words, st);
    };
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    if constexpr (kLayout == Layout::kPairs) {
      using Four = std::integral_constant<int, 4>;
      using Many = std::false_type;
      if (plan.chunk == kOwnerThreads) return owners(One{}, One{}, Many{});
      if (plan.chunk == 2 * kOwnerThreads) return plan.per_lane == 1 ? owners(Two{}, One{}, Many{}) : owners(Two{}, Two{}, Many{});
      return plan.per_lane == 1 ? owners(Four{}, One{}, Many{}) : owners(Four{}, Two{}, Many{});
    } else {
      return slice == 1 ? owners(Two{}, One{}, std::true_type{}) : owners(Two{}, One{}, std::false_type{});
    }
  }
  if (plan.chunk == 16)
    return launch_shape<T, 256, 16, 1, kLayout>(updates, data, indices, s, n, k, slice, slice * targets, lanes, words, st);
  if (plan.chunk == 64 && plan.threads == 512)
    return launch_shape<T, 512, 64, 1, kLayout>(updates, data, indices, s, n, k, slice, slice * targets, lanes, words, st);
  if (plan.chunk == 64)
    return launch_shape<T, 256, 64, 1, kLayout>(updates, data, indices, s, n, k, slice, slice * targets, lanes, words, st);
  if (plan.chunk == 128)
    return launch_shape<T, 1024, 128, 2, kLayout>(updates, data, indices, s, n, k, slice, slice * targets, lanes, words, st);
  return launch_direct<T, kLayout, false>(updates, data, indices, s, n, k, slice, slice * targets, lanes, words, st);
}

// Lanes that share an update of `words` words.
int lanes_of(long long words) {
  int lanes = 1;
  while (lanes < kWaveSize && lanes < words) lanes *= 2;
  return lanes;
}

template <typename T>
int launch(const void* updates, void* data, const long long* indices, const Strides& s, long long n, int k,
           long long slice, long long targets, hipStream_t st) {
  constexpr int kElems = Word<T>::kElems;
  // slices whose words are pairs of one slice in both arrays; otherwise a slice may take one word more
  const bool pairs = kElems == 1 || (slice % 2 == 0 && reinterpret_cast<size_t>(updates) % 4 == 0 &&
                                     reinterpret_cast<size_t>(data) % 4 == 0);
  const long long words = (slice + kElems - 1 + (pairs ? 0 : 1)) / kElems;
  const int lanes = lanes_of(words);
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

extern "C" int tf_scatter_nd_plan(int64_t num_index_rows, int64_t targets, int64_t slice, int dtype, int* words_a_lane) {
  using namespace tfk;
  if (num_index_rows <= 0 || targets <= 0 || slice <= 0 || dtype < 0 || dtype > 2 || !words_a_lane) return -1;
  const bool split = dtype != 0 && slice % 2 != 0;
  const long long words = dtype == 0 ? slice : (slice + 1 + (split ? 1 : 0)) / 2;
  const ScatterPlan plan = plan_scatter(dtype == 0 ? 4 : 2, split ? Layout::kSplit : Layout::kPairs, num_index_rows, targets, words,
                                        lanes_of(words));
  *words_a_lane = plan.per_lane;
  return plan.chunk;
}
