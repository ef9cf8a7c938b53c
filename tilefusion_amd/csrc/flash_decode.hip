// Split-KV flash-decoding for gfx950: single-query attention per (batch x head) slice with the
// key/value range cut into up to `num_splits` chunks, followed by a log-sum-exp combine (or, where one
// workgroup per slice is done sooner, not cut and finished in one kernel).
//
// No counterpart in the reference (it has no decoding kernel); the per-chunk algebra is the
// online softmax of include/kernels/flash_attention_device.cuh:257-301 with one query row.
// Both kernels are HBM-bound streaming kernels, MFMA is irrelevant (1 flop per byte):
//   * split kernel: grid (splits, batch_heads), 4 or 8 wavefronts.  One key row of 128 16-bit
//     elements is 256 bytes = 16 lanes x 16 bytes (head dimension 64: 8 lanes), so a wavefront
//     load instruction fetches 4 (8) whole rows fully coalesced; every group of 16 (8) lanes keeps
//     its own running (max, sum, o[D]) over the rows it sees; the groups of a wavefront are merged with
//     lane swaps, the wavefronts through LDS.  The dot product is v_dot2 (fp16 or bf16) +
//     a DPP reduction inside the lane group;
//     two batches of 4 or 6 rows per group are in flight (16 or 24 KiB per wavefront), the next one
//     requested before the current one is consumed; the partials leave through streaming
//     stores (ordinary stores in the middle of the read stream cost 7% of its bandwidth);
//   * the partials of a slice are merged by the workgroup of it that is done last, where the workspace has room for a word of
//     arrivals a slice and fewer than 1024 workgroups run (32 slices of 1999 x 64, bf16: 9.6 us with a second kernel, 6.3 as
//     this; 9 of 5829 x 128 11.4 and 8.4);
//   * otherwise by the combine kernel, grid batch_heads: with many workgroups every one holds its place on a CU
//     until its partials and its arrival are acknowledged (60 slices of 38872 x 64: 95 us, merged in one kernel 112).
// The kernels are templates of the element type (fp16 / bf16, the reference's 16-bit types,
// include/kernels/dispatch_macros.hpp:6-23) and of the head dimension (128 / 64).
// All offsets are 64-bit.
#include <algorithm>
#include <cmath>
#include <mutex>
#include <type_traits>

#include "common.hpp"

namespace tfk {
namespace {

// Rows per lane group in one batch of loads, of which up to two are in flight.  More cost registers and with them
// wavefronts; six pay where a CU often has one workgroup only (fp16, four / six / eight rows: 157 slices of 6530 x 128
// 84.1 / 79.9 / 79.9 us, 186 of 11138 x 128 160.9 / 152.1 / 151.6, 33 of 662 x 64 5.5 / 5.8 / 7.2).
__host__ __device__ constexpr int batch_rows(int waves, bool whole) { return whole && waves == 8 ? 6 : 4; }
using float2_t = float __attribute__((ext_vector_type(2)));

constexpr int kD = 128;   // head dimension of the benchmark configuration (and of the static entry point)

template <int CTRL>
TFK_DEVICE float dpp_f32(float x) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, false));
}
// Sum over a group of kLanes (16 or 8) adjacent lanes; every lane ends up with the total.
template <int kLanes>
TFK_DEVICE float group_sum(float x) {
  if constexpr (kLanes == 16) {
    x += dpp_f32<0x128>(x);  // row_ror:8
    x += dpp_f32<0x124>(x);  // row_ror:4
    x += dpp_f32<0x122>(x);  // row_ror:2
    x += dpp_f32<0x121>(x);  // row_ror:1
  } else {
    static_assert(kLanes == 8, "a key row is 16 or 8 lanes wide");
    x += dpp_f32<0x141>(x);  // row_half_mirror: lane i <-> 7 - i inside each half row
    x += dpp_f32<0xB1>(x);   // quad_perm [1, 0, 3, 2]
    x += dpp_f32<0x4E>(x);   // quad_perm [2, 3, 0, 1]
  }
  return x;
}

// op(x of this lane, x of the lane kXor away), kXor = 8, 16 or 32
template <int kXor, typename Op>
TFK_DEVICE float xor_combine(float x, Op op) {
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (kXor == 8) {
    return op(x, dpp_f32<0x128>(x));  // row_ror:8
  } else {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    // with both operands x, the swap leaves the even rows (halves) in one and the odd ones in the other
    const auto sw = kXor == 16 ? __builtin_amdgcn_permlane16_swap(u, u, false, false)
                               : __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const unsigned a = sw[0], b = sw[1];
    return op(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
  }
#else
  return x;
#endif
}
// op over the lanes that hold the same vector of different rows; every lane ends up with the result
template <int kLanesPerRow, typename Op>
TFK_DEVICE float across_rows(float x, Op op) {
  if constexpr (kLanesPerRow == 8) x = xor_combine<8>(x, op);
  return xor_combine<32>(xor_combine<16>(x, op), op);
}

template <typename T>
struct Vec8 {
  using type = T __attribute__((ext_vector_type(8)));
};
template <typename T>
TFK_DEVICE float dot8(typename Vec8<T>::type k, typename Vec8<T>::type q) {
  float acc = 0.f;
#define TFK_DOT2(i)                                                                                         \
  if constexpr (std::is_same_v<T, bf16_t>)                                                                  \
    acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(k, k, i, i + 1), __builtin_shufflevector(q, q, i, i + 1), acc, false); \
  else                                                                                                      \
    acc = __builtin_amdgcn_fdot2(__builtin_shufflevector(k, k, i, i + 1), __builtin_shufflevector(q, q, i, i + 1), acc, false);
  TFK_DOT2(0) TFK_DOT2(2) TFK_DOT2(4) TFK_DOT2(6)
#undef TFK_DOT2
  return acc;
}

// 16 bytes at base + offset, zeros where that is not within `bytes`; `base` and `bytes` are wavefront-uniform.
template <typename V>
TFK_DEVICE V load_below(const char* base, unsigned bytes, unsigned offset) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int kRaw32Bit = 0x00020000, kStreaming = 2;
  const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, bytes, kRaw32Bit);
  return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(rsrc, offset, 0, kStreaming));
#else
  return V{};
#endif
}

// The partials of one slice put together; the first kCombThreads threads of a workgroup, behind which all of it meets at the barrier.  Groups
// of D / 4 lanes take every kGroups-th split with its loads in flight at once, then the groups are added up in LDS.  (One thread per column
// that walks the splits one after another is a chain of loads: 9.5 us for 64 splits of 32 slices, 2.4 as here.)
// kShared: the partials come from other workgroups of the same launch.
constexpr int kCombThreads = 256;
template <typename T, int D, bool kShared>
TFK_DEVICE void combine_slice(const float* o_part, const float* ml_part, T* __restrict__ O, int num_splits) {
  constexpr int kLanes = D / 4, kGroups = kCombThreads / kLanes, kUnroll = 8;
  __shared__ float4_t s_o[kGroups][kLanes];
  __shared__ float s_l[kGroups];
  const int lane = threadIdx.x % kLanes, grp = threadIdx.x / kLanes;
  if (threadIdx.x < kCombThreads) {
    float4_t o[kUnroll];
    float m[kUnroll], sum[kUnroll];
    auto load = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        const int s = min(s0 + u * kGroups, num_splits - 1);
        if constexpr (kShared) {
          o[u] = load_shared_16B<float4_t>(o_part, (unsigned)(s * kLanes + lane) * 16u);
          m[u] = load_shared(ml_part + 2 * s);
          sum[u] = load_shared(ml_part + 2 * s + 1);
        } else {
          o[u] = reinterpret_cast<const float4_t*>(o_part)[s * kLanes + lane];
          const float2_t x = reinterpret_cast<const float2_t*>(ml_part)[s];
          m[u] = x[0];
          sum[u] = x[1];
        }
      }
    };
    load(grp);   // in flight while the maximum is found
    float big = -INFINITY;
    for (int s = threadIdx.x % kWaveSize; s < num_splits; s += kWaveSize)
      big = fmaxf(big, kShared ? load_shared(ml_part + 2 * s) : ml_part[2 * s]);
#pragma unroll
    for (int x = 1; x < kWaveSize; x *= 2) big = fmaxf(big, __shfl_xor(big, x));
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
    float l = 0.f;
    for (int s0 = grp; s0 < num_splits; s0 += kGroups * kUnroll) {
      if (s0 != grp) load(s0);
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        if (s0 + u * kGroups >= num_splits) break;   // (the last split again, which may hold infinities)
        const float w = __builtin_amdgcn_exp2f(m[u] - big);
        acc += w * o[u];
        l += w * sum[u];
      }
    }
    s_o[grp][lane] = acc;
    if (lane == 0) s_l[grp] = l;
  }
  __syncthreads();
  if (threadIdx.x < D) {
    float sum = 0.f, total = 0.f;
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
      sum += s_o[g][threadIdx.x / 4][threadIdx.x % 4];
      total += s_l[g];
    }
    O[threadIdx.x] = (T)(sum / total);
  }
}

// workspace: o_part [batch_heads][num_splits][D] fp32, then ml_part [batch_heads][num_splits][2], then (kMerged) a word of
// arrivals a slice.
// kWhole: one workgroup per slice, which writes O itself (num_splits == 1, chunk == Lkv).
// kMerged: the workgroup of a slice that is done last puts the parts together; kParts leaves that to a second kernel.
enum DecodeEnd { kWhole, kMerged, kParts };
// `chunk` is a multiple of the rows of one load step.
// kDecWaves wavefronts per workgroup.
template <typename T, int D, int kDecWaves, DecodeEnd kEnd>
__global__ __launch_bounds__(kDecWaves * kWaveSize) void flash_decode_split_kernel(
    const T* __restrict__ Q, const T* __restrict__ K, const T* __restrict__ V, T* __restrict__ O,
    float* o_part, float* ml_part, int64_t Lkv, int num_splits,
    int64_t chunk, float scale_log2, arrivals_t* arrivals, arrivals_t tag) {
  using V8 = typename Vec8<T>::type;
  constexpr int kLanesPerRow = D / 8;                   // 16-byte vectors per row
  constexpr int kRowsPerWave = kWaveSize / kLanesPerRow;  // rows one wavefront load instruction covers
  constexpr int kRowsPerStep = kDecWaves * kRowsPerWave;  // ... and one workgroup load step
  constexpr int kBatchRows = batch_rows(kDecWaves, kEnd == kWhole);
  __shared__ float s_o[kDecWaves][D];
  __shared__ float s_m[kDecWaves], s_l[kDecWaves];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lv = lane % kLanesPerRow, gw = lane / kLanesPerRow;   // vector of the row, row of the wavefront's load
  const int split = blockIdx.x;
  const int64_t bh = blockIdx.y;
  const int64_t row_begin = (int64_t)split * chunk;
  const int64_t row_end = min(row_begin + chunk, Lkv);

  const V8 q8 = *reinterpret_cast<const V8*>(Q + bh * D + 8 * lv);

  float m_run = -INFINITY, l_run = 0.f;
  float o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = 0.f;

  // Two register sets of kBatchRows rows per group: the loads of batch b+1 are issued before
  // batch b is consumed, so a wavefront always has loads on their way (a load-all / wait-all /
  // compute loop leaves the memory pipe of that wavefront empty while it computes).
  // The loop asks past the end of the range as well: the bounds check of a buffer load returns zeros there and
  // fetches nothing.  (With a branch around the loads of a short batch the compiler waits for all loads
  // in flight where its two ways meet.  Zeros, because the weight of such a row is zero, and zero
  // times another row's infinity would be NaN.)
  constexpr int kBatchSpan = kBatchRows * kRowsPerStep;
  constexpr int kRowBytes = D * 2;
  const int lane_row = wave * kRowsPerWave + gw;
  unsigned lane_off[kBatchRows];   // bytes inside a batch
#pragma unroll
  for (int u = 0; u < kBatchRows; ++u) lane_off[u] = (unsigned)((lane_row + u * kRowsPerStep) * kRowBytes + 16 * lv);
  const char* k_slice = reinterpret_cast<const char*>(K + bh * Lkv * D);
  const char* v_slice = reinterpret_cast<const char*>(V + bh * Lkv * D);
  auto rows_left = [&](int64_t base) __attribute__((always_inline)) {   // of a batch
    return (int)max((int64_t)0, min((int64_t)kBatchSpan, row_end - base));
  };
  auto load_batch = [&](V8* kd, V8* vd, int64_t base) __attribute__((always_inline)) {
    const unsigned bytes = (unsigned)rows_left(base) * kRowBytes;
#pragma unroll
    for (int u = 0; u < kBatchRows; ++u) kd[u] = load_below<V8>(k_slice + base * kRowBytes, bytes, lane_off[u]);
#pragma unroll
    for (int u = 0; u < kBatchRows; ++u) vd[u] = load_below<V8>(v_slice + base * kRowBytes, bytes, lane_off[u]);
    __builtin_amdgcn_sched_barrier(0);   // the requests leave before the other batch is consumed
  };
  auto consume = [&](const V8* kd, const V8* vd, int64_t base) __attribute__((always_inline)) {
    const int left = rows_left(base) - lane_row;
    float s[kBatchRows];
    float mx = -INFINITY;
#pragma unroll
    for (int u = 0; u < kBatchRows; ++u) {
      const float d = group_sum<kLanesPerRow>(dot8<T>(kd[u], q8)) * scale_log2;
      s[u] = u * kRowsPerStep < left ? d : -INFINITY;
      mx = fmaxf(mx, s[u]);
    }
    const float m_new = fmaxf(m_run, mx);
    const float m_safe = (m_new == -INFINITY) ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_safe);
    m_run = m_new;
    l_run *= alpha;
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] *= alpha;
#pragma unroll
    for (int u = 0; u < kBatchRows; ++u) {
      const float p = __builtin_amdgcn_exp2f(s[u] - m_safe);
      l_run += p;
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] += p * (float)vd[u][i];
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  V8 k_a[kBatchRows], v_a[kBatchRows], k_b[kBatchRows], v_b[kBatchRows];
  load_batch(k_a, v_a, row_begin);
  if (kEnd == kMerged && tid == 0 && split == 0) open_arrivals(arrivals + bh * kArrivalsPitch, tag);
  int64_t base = row_begin;
  for (; base + kBatchSpan < row_end; base += 2 * kBatchSpan) {
    load_batch(k_b, v_b, base + kBatchSpan);
    consume(k_a, v_a, base);
    load_batch(k_a, v_a, base + 2 * kBatchSpan);
    consume(k_b, v_b, base + kBatchSpan);
  }
  if (base < row_end) consume(k_a, v_a, base);

  // merge the lane groups of the wavefront, then the wavefronts
  const auto add = [](float a, float b) { return a + b; };
  float big = across_rows<kLanesPerRow>(m_run, [](float a, float b) { return fmaxf(a, b); });
  const float scale = __builtin_amdgcn_exp2f(m_run - ((big == -INFINITY) ? 0.f : big));
  l_run = across_rows<kLanesPerRow>(l_run * scale, add);
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = across_rows<kLanesPerRow>(o[i] * scale, add);
  if (gw == 0) {
#pragma unroll
    for (int i = 0; i < 8; ++i) s_o[wave][8 * lv + i] = o[i];
  }
  if (lane == 0) {
    s_m[wave] = big;
    s_l[wave] = l_run;
  }
  __syncthreads();
  if (tid < D) {
    big = -INFINITY;
#pragma unroll
    for (int w = 0; w < kDecWaves; ++w) big = fmaxf(big, s_m[w]);
    const float big_safe = (big == -INFINITY) ? 0.f : big;
    float acc = 0.f, l = 0.f;
#pragma unroll
    for (int w = 0; w < kDecWaves; ++w) {
      const float f = __builtin_amdgcn_exp2f(s_m[w] - big_safe);
      acc += f * s_o[w][tid];
      l += f * s_l[w];
    }
    if constexpr (kEnd == kWhole) {
      O[bh * D + tid] = (T)(acc / l);
      return;
    }
    const int64_t idx = bh * num_splits + split;
    if constexpr (kEnd == kMerged) {
      store_shared(o_part + idx * D + tid, acc);
      if (tid == 0) {
        store_shared(ml_part + idx * 2, big);
        store_shared(ml_part + idx * 2 + 1, l);
      }
    } else {
      // Streaming stores: an ordinary store of these few hundred bytes per workgroup, issued in
      // the middle of an 8 GiB read stream, costs 7% of the read bandwidth (6.6 against 7.15
      // TB/s in a plain two-stream read kernel with and without such a store; 7.05 with this one).
      __builtin_nontemporal_store(acc, o_part + idx * D + tid);
      if (tid == 0) {
        __builtin_nontemporal_store(big, ml_part + idx * 2);
        __builtin_nontemporal_store(l, ml_part + idx * 2 + 1);
      }
    }
  }
  if constexpr (kEnd == kMerged) {
    __shared__ bool s_last;
    wait_vmem_all();
    if constexpr (D > kWaveSize) __syncthreads();   // (otherwise the first wavefront has written all of it)
    if (tid == 0) s_last = arrive(arrivals + bh * kArrivalsPitch, tag, (unsigned)num_splits);
    __syncthreads();
    if (!s_last) return;
    combine_slice<T, D, true>(o_part + bh * num_splits * D, ml_part + bh * num_splits * 2, O + bh * D, num_splits);
  }
}

// One workgroup per slice.
template <typename T, int D>
__global__ __launch_bounds__(kCombThreads) void flash_decode_combine_kernel(
    const float* __restrict__ o_part, const float* __restrict__ ml_part, T* __restrict__ O,
    int num_splits) {
  const int64_t bh = blockIdx.x;
  combine_slice<T, D, false>(o_part + bh * num_splits * D, ml_part + bh * num_splits * 2, O + bh * D, num_splits);
}

}  // namespace
}  // namespace tfk

extern "C" size_t tf_flash_decode_workspace_bytes(int64_t batch_heads, int64_t D, int num_splits) {
  if (batch_heads <= 0 || D <= 0 || num_splits <= 0) return 0;
  return (size_t)batch_heads * (size_t)num_splits * (size_t)(D + 2) * sizeof(float);
}

namespace tfk {
namespace {

// Argument checks shared by both entry points.
int check_decode_args(const char* who, const void* Q, const void* K, const void* V, const void* O,
                      int64_t batch_heads, int64_t Lkv, int64_t D, int num_splits,
                      double softmax_scale) {
  TFK_REQUIRE(Q && K && V && O, TF_ERR_INVALID_ARG, "%s: null pointer", who);
  TFK_REQUIRE(batch_heads > 0 && Lkv > 0 && num_splits > 0, TF_ERR_INVALID_ARG,
              "%s: sizes must be positive", who);
  TFK_REQUIRE(batch_heads < 65536 && num_splits <= 65536, TF_ERR_INVALID_ARG,
              "%s: batch_heads / num_splits too large", who);
  TFK_REQUIRE(D == 128 || D == 64, TF_ERR_UNSUPPORTED, "%s: head dim must be 128 or 64 (got %lld)", who, (long long)D);
  TFK_REQUIRE(softmax_scale == softmax_scale && softmax_scale - softmax_scale == 0.0,
              TF_ERR_INVALID_ARG, "%s: softmax_scale must be finite", who);
  return TF_OK;
}

// How a problem is cut.  `splits` ranges of `chunk` keys per slice; 1: one workgroup per slice, no partials
// and no second kernel.  `waves` wavefronts per workgroup.
struct DecodePlan {
  int splits;
  int64_t chunk;
  int waves;
};
// One workgroup takes in ~45 GB/s when few run, all of them together 6.7 TB/s; the second kernel and its
// launch, or the arrivals and the merge, cost ~4 or ~2 us.  Measured (fp16, us, one workgroup per slice / best split): 33 slices of 662 x 64
// 6.5 / 8.1, 964 of 913 x 128 68 / 73, 11 of 825 x 128 10.4 / 8.5, 64 of 8192 x 128 85 / 44.  Slices that the
// CUs cannot share evenly cost about a third of the unevenness (802 of 2574 x 128: 180 / 165).
// Where the slices are large and many, one workgroup in each means hundreds of streams, megabytes apart, and a first
// pass over memory whose translations no cache holds yet pays for each (512 of 32768 x 128: 1460-1500 us, in 8
// ranges 1320-1370; 155 of 36332 x 128 636 / 569, 180 of 50000 x 128 886 / 807).  Passes after that take as long
// either way (512 of 32768 x 128 1237 / 1235, over ten caches in turn too).  So slices of more than 4 MiB, of
// more than 2.75 GB together, come in ranges of at most 2 MiB.  (Below neither was ahead at first: 512 of 8192 x 128 375 whole
// and 384 cut, 512 of 10000 x 128 484 and 491, 200 of 12000 x 128 246 and 242 - then 190 and 196.)
// Up to 128 slices, of 600 MB together, are cut so that every CU has one workgroup at most: eight wavefronts take in what a
// CU's share is, more workgroups are a second round and more arrivals (us, 256 workgroups at most / 1024: 24 of 4301 x 128 11.9 /
// 13.7, 19 of 2620 x 128 8.0 / 10.5, 102 of 1952 x 128 18.9 / 20.9, 66 of 2934 x 64 11.8 / 14.0, 128 of 8192 x 128 84 / 87).  Beyond,
// long ranges cost a first pass more than they gain (32 of 55533 x 128: first 144-160 us in 4 MiB, 151-181; repeated 139 both).
// Otherwise the cut aims at 1024 workgroups, and at no more than 256 KiB of keys and values in each: they
// come in rounds, and the last one fills the chip badly (584 of 16256 x 64: 4 splits 411, 16 364; 136 of
// 36053 x 64: 8 splits 201, 32 192).  In any case 32 KiB at least (with the second kernel, 32 of 1999 x 64: 16 splits 10.2,
// 64 12.8; for few slices, 3 of 1001 x 64, it is what limits the cut), all within the caller's num_splits.
template <int D>
DecodePlan plan_decode(int64_t batch_heads, int64_t Lkv, int num_splits) {
  const double slice_bytes = 4.0 * D * Lkv, stream_us = slice_bytes * batch_heads / 6.7e6, alone_us = slice_bytes / 45e3;
  const double per_cu = batch_heads / 256.0;
  const double uneven = per_cu > 1.0 ? 1.0 + 0.35 * (std::ceil(per_cu) / per_cu - 1.0) : 1.0;
  // one workgroup per slice: eight wavefronts take it in faster, four share a full chip better (512 slices of
  // 32768 x 128: 1254 and 1203 us; 33 of 662 x 64: 6.5 and 8.1)
  const DecodePlan whole = {1, Lkv, batch_heads >= 512 ? 4 : 8};
  const bool shared_evenly = 2.5 + std::max(alone_us, stream_us * uneven) <= 6.5 + stream_us;
  if (num_splits == 1 || (shared_evenly && (slice_bytes <= 4194304.0 || slice_bytes * batch_heads <= 2.75e9))) return whole;
  constexpr int64_t kStep = 8 * (kWaveSize / (D / 8));   // rows of one load step of the larger workgroup
  const bool one_round = batch_heads <= 128 && slice_bytes * batch_heads <= 6e8;
  const int64_t fill = one_round ? 256 / batch_heads : (1024 + batch_heads - 1) / batch_heads;
  const int64_t least = one_round       ? 1
                        : shared_evenly ? (int64_t)std::ceil(slice_bytes / 2097152.0)
                                        : (int64_t)(slice_bytes / 262144.0) + 1;
  const int64_t most = (int64_t)(slice_bytes / 32768.0) + 1;
  const int64_t want = std::min<int64_t>(num_splits, std::min(std::max(fill, least), most));
  const int64_t chunk = ((Lkv + want - 1) / want + kStep - 1) / kStep * kStep;
  const int64_t splits = (Lkv + chunk - 1) / chunk;
  // few workgroups: eight wavefronts each (8 slices of 65536 x 128 in 16 splits: 76 us with four, 54 with
  // eight; 802 of 2574 x 128 in 4: 165 and 173)
  return splits > 1 ? DecodePlan{(int)splits, chunk, batch_heads * splits < 1024 ? 8 : 4} : whole;
}

template <typename T, int D, int kDecWaves, DecodeEnd kEnd>
int launch_split(const void* Q, const void* K, const void* V, void* O, float* o_part, float* ml_part,
                 int64_t batch_heads, int64_t Lkv, DecodePlan plan, double softmax_scale, hipStream_t st, arrivals_t* arrivals = nullptr) {
  const float scale_log2 = (float)(softmax_scale * 1.4426950408889634);
  return launch_kernel(flash_decode_split_kernel<T, D, kDecWaves, kEnd>, dim3(plan.splits, (unsigned)batch_heads),
                       dim3(kDecWaves * kWaveSize), 0, st, static_cast<const T*>(Q), static_cast<const T*>(K),
                       static_cast<const T*>(V), static_cast<T*>(O), o_part, ml_part, Lkv, plan.splits, plan.chunk,
                       scale_log2, arrivals, kEnd == kMerged ? next_arrivals_tag() : 0);
}

// The kernels on `st`; `partials` holds o_part then ml_part and, where there is `room` (bytes) for them, the words in which the
// workgroups of a slice arrive, and is at a 16-byte boundary.  The arrivals are atomics: a caller's workspace elsewhere than in the
// device's ordinary memory holds partials only.  own: it is the library's, which is.
template <typename T, int D>
int launch_decode_t(const void* Q, const void* K, const void* V, void* O, float* partials, size_t room, bool own,
                    int64_t batch_heads, int64_t Lkv, int num_splits, double softmax_scale,
                    hipStream_t st) {
  const DecodePlan plan = plan_decode<D>(batch_heads, Lkv, num_splits);
  if (plan.splits == 1) {
    if (plan.waves == 4)
      return launch_split<T, D, 4, kWhole>(Q, K, V, O, nullptr, nullptr, batch_heads, Lkv, plan, softmax_scale, st);
    return launch_split<T, D, 8, kWhole>(Q, K, V, O, nullptr, nullptr, batch_heads, Lkv, plan, softmax_scale, st);
  }
  float* o_part = partials;
  float* ml_part = o_part + (size_t)batch_heads * plan.splits * D;
  const size_t part_floats = (size_t)batch_heads * plan.splits * (D + 2);   // (even: the words behind it are at 8-byte boundaries)
  if (part_floats * sizeof(float) + (size_t)batch_heads * kArrivalsPitch * sizeof(arrivals_t) <= room && plan.waves == 8 &&
      (own || is_ordinary_device_memory(partials))) {
    arrivals_t* arrivals = reinterpret_cast<arrivals_t*>(partials + part_floats);
    return launch_split<T, D, 8, kMerged>(Q, K, V, O, o_part, ml_part, batch_heads, Lkv, plan, softmax_scale, st, arrivals);
  }
  const int rc = plan.waves == 8
      ? launch_split<T, D, 8, kParts>(Q, K, V, O, o_part, ml_part, batch_heads, Lkv, plan, softmax_scale, st)
      : launch_split<T, D, 4, kParts>(Q, K, V, O, o_part, ml_part, batch_heads, Lkv, plan, softmax_scale, st);
  if (rc != TF_OK) return rc;
  return launch_kernel(flash_decode_combine_kernel<T, D>, dim3((unsigned)batch_heads), dim3(kCombThreads), 0, st,
                       o_part, ml_part, static_cast<T*>(O), plan.splits);
}
int launch_decode(const void* Q, const void* K, const void* V, void* O, float* partials, size_t room, bool own, int dtype,
                  int64_t batch_heads, int64_t Lkv, int64_t D, int num_splits, double softmax_scale,
                  hipStream_t st) {
  if (dtype == TF_DTYPE_BF16) {
    if (D == 128) return launch_decode_t<bf16_t, 128>(Q, K, V, O, partials, room, own, batch_heads, Lkv, num_splits, softmax_scale, st);
    return launch_decode_t<bf16_t, 64>(Q, K, V, O, partials, room, own, batch_heads, Lkv, num_splits, softmax_scale, st);
  }
  if (D == 128) return launch_decode_t<half_t, 128>(Q, K, V, O, partials, room, own, batch_heads, Lkv, num_splits, softmax_scale, st);
  return launch_decode_t<half_t, 64>(Q, K, V, O, partials, room, own, batch_heads, Lkv, num_splits, softmax_scale, st);
}

int decode_with_workspace(const char* who, const void* Q, const void* K, const void* V, void* O, int dtype,
                          void* workspace, size_t workspace_bytes, int64_t batch_heads, int64_t Lkv, int64_t D,
                          int num_splits, double softmax_scale, void* stream) {
  TFK_REQUIRE(workspace, TF_ERR_INVALID_ARG, "%s: null pointer", who);
  if (int rc = check_decode_args(who, Q, K, V, O, batch_heads, Lkv, D, num_splits, softmax_scale)) return rc;
  const size_t need = tf_flash_decode_workspace_bytes(batch_heads, D, num_splits);
  TFK_REQUIRE(workspace_bytes >= need, TF_ERR_INVALID_ARG, "%s: workspace holds %zu bytes, %zu needed", who,
              workspace_bytes, need);
  TFK_REQUIRE(((uintptr_t)workspace & 15) == 0, TF_ERR_INVALID_ARG, "%s: workspace must be 16-byte aligned", who);
  return launch_decode(Q, K, V, O, static_cast<float*>(workspace), workspace_bytes, false, dtype, batch_heads, Lkv, D, num_splits,
                       softmax_scale, static_cast<hipStream_t>(stream));
}

}  // namespace
}  // namespace tfk

extern "C" int tf_flash_decode_plan(int64_t batch_heads, int64_t Lkv, int64_t D, int num_splits, int* wavefronts) {
  using namespace tfk;
  if (batch_heads <= 0 || Lkv <= 0 || num_splits <= 0 || !wavefronts || (D != 128 && D != 64)) return 0;
  const DecodePlan plan = D == 128 ? plan_decode<128>(batch_heads, Lkv, num_splits) : plan_decode<64>(batch_heads, Lkv, num_splits);
  *wavefronts = plan.waves;
  return plan.splits;
}

extern "C" int tf_flash_decode_f16(const void* Q, const void* K, const void* V, void* O,
                                   void* workspace, size_t workspace_bytes, int64_t batch_heads,
                                   int64_t Lkv, int64_t D, int num_splits, double softmax_scale,
                                   void* stream) {
  return tfk::decode_with_workspace("tf_flash_decode_f16", Q, K, V, O, TF_DTYPE_F16, workspace, workspace_bytes,
                                    batch_heads, Lkv, D, num_splits, softmax_scale, stream);
}

extern "C" int tf_flash_decode(const void* Q, const void* K, const void* V, void* O, int dtype,
                               void* workspace, size_t workspace_bytes, int64_t batch_heads,
                               int64_t Lkv, int64_t D, int num_splits, double softmax_scale,
                               void* stream) {
  using namespace tfk;
  TFK_REQUIRE(dtype == TF_DTYPE_F16 || dtype == TF_DTYPE_BF16, TF_ERR_UNSUPPORTED,
              "tf_flash_decode: dtype must be TF_DTYPE_F16 or TF_DTYPE_BF16");
  return decode_with_workspace("tf_flash_decode", Q, K, V, O, dtype, workspace, workspace_bytes, batch_heads, Lkv, D,
                               num_splits, softmax_scale, stream);
}

extern "C" int tf_flash_decode_uncut(const void* Q, const void* K, const void* V, void* O, int dtype, int64_t batch_heads,
                                     int64_t Lkv, int64_t D, int num_splits, double softmax_scale, void* stream) {
  using namespace tfk;
  // (no message for what is cut or not taken: tf_flash_decode has one)
  if (dtype != TF_DTYPE_F16 && dtype != TF_DTYPE_BF16) return TF_ERR_UNSUPPORTED;
  int waves = 0;
  if (tf_flash_decode_plan(batch_heads, Lkv, D, num_splits, &waves) != 1) return TF_ERR_UNSUPPORTED;
  if (int rc = check_decode_args("tf_flash_decode_uncut", Q, K, V, O, batch_heads, Lkv, D, num_splits, softmax_scale)) return rc;
  return launch_decode(Q, K, V, O, nullptr, 0, false, dtype, batch_heads, Lkv, D, num_splits, softmax_scale,
                       static_cast<hipStream_t>(stream));
}

// ---- the same kernels with the partials in a static device array -------------------
//
// For callers that cannot allocate device memory (code under HIP graph capture, tight serving
// loops, harnesses that forbid hipMalloc): no workspace argument, nothing allocated.  Every GPU
// the library runs on holds its own copy of `scratch` until the process ends.  The name
// `scratch` is only a host-side handle of the symbol, not a device address: the address on each
// device comes from hipGetSymbolAddress, once, with that device current, and only that pointer
// is ever handed to a kernel.
namespace tfk {
namespace {

constexpr size_t kScratchFloats = (size_t)TF_FLASH_DECODE_STATIC_MAX_PARTIALS * (kD + 2);
static __device__ __align__(256) float scratch[kScratchFloats];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
float* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device (looked up on the first call per device).
int scratch_on_current_device(float** out) {
  int dev = -1;
  TFK_HIP_TRY(hipGetDevice(&dev));
  TFK_REQUIRE(dev >= 0 && dev < kMaxDevices, TF_ERR_UNSUPPORTED,
              "tf_flash_decode_static_f16: device ordinal %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    TFK_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    TFK_REQUIRE(p != nullptr, TF_ERR_HIP, "tf_flash_decode_static_f16: null symbol address");
    g_scratch_ptr[dev] = static_cast<float*>(p);
  }
  *out = g_scratch_ptr[dev];
  return TF_OK;
}

}  // namespace
}  // namespace tfk

extern "C" size_t tf_flash_decode_static_max_partials(void) {
  return (size_t)TF_FLASH_DECODE_STATIC_MAX_PARTIALS;
}

extern "C" int tf_flash_decode_static_prepare(void) {
  float* unused = nullptr;
  return tfk::scratch_on_current_device(&unused);
}

extern "C" int tf_flash_decode_static_f16(const void* Q, const void* K, const void* V, void* O,
                                          int64_t batch_heads, int64_t Lkv, int64_t D,
                                          int num_splits, double softmax_scale, void* stream) {
  using namespace tfk;
  if (int rc = check_decode_args("tf_flash_decode_static_f16", Q, K, V, O, batch_heads, Lkv, D,
                                 num_splits, softmax_scale))
    return rc;
  TFK_REQUIRE(D == kD, TF_ERR_UNSUPPORTED, "tf_flash_decode_static_f16: head dim must be 128 (got %lld)", (long long)D);
  TFK_REQUIRE((uint64_t)batch_heads * (uint64_t)num_splits <= TF_FLASH_DECODE_STATIC_MAX_PARTIALS,
              TF_ERR_INVALID_ARG,
              "tf_flash_decode_static_f16: batch_heads * num_splits = %llu exceeds the static "
              "scratch array (%llu partials); use tf_flash_decode_f16 with a workspace",
              (unsigned long long)((uint64_t)batch_heads * (uint64_t)num_splits),
              (unsigned long long)TF_FLASH_DECODE_STATIC_MAX_PARTIALS);
  float* partials = nullptr;
  if (int rc = scratch_on_current_device(&partials)) return rc;
  // Nothing has to start at zero: the split kernel writes every (slice, split) partial before it is
  // read, and a word of arrivals may hold anything (arrivals_t).
  return launch_decode(Q, K, V, O, partials, kScratchFloats * sizeof(float), true, TF_DTYPE_F16, batch_heads, Lkv, D, num_splits,
                       softmax_scale, static_cast<hipStream_t>(stream));
}
