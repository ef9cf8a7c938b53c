// Flash-attention forward for gfx950: O = softmax(scale * Q K^T (+ causal mask)) V per
// (batch x head) slice, fp16 or bf16 in/out, fp32 scores and fp32 running max / sum.
//
// Counterpart of ke_flash_attention (include/kernels/flash_attention_device.cuh:130-312, mask
// include/cell/mask.hpp:75-82) and its host launcher (src/kernels/flash_attn.cu:58-152).
// CDNA4 design (FA-2 style, un-normalised O with one divide at the end):
//   * one workgroup = 256 queries (8 wavefronts x 32), or 128 (8 x 16) or 64 (4 x 16) where 256
//     would leave CUs idle; key/value tiles of 64 rows, v_mfma_f32_16x16x32_f16 throughout (the most
//     power-efficient fp16 MFMA shape: the kernel runs at the power limit, so energy per
//     flop sets its speed);
//   * Q stays in registers for the whole workgroup (the reference reloads it per KV tile);
//   * scores are computed transposed, S^T = K Q^T, so a lane owns one query row per 16-query
//     block: its score values are plain registers, the running max is an in-lane
//     reduction (the 4 lanes that share a query only talk when the reference max moves),
//     and exp2(S^T) converted to fp16 is already the B-operand fragment of the second MFMA
//     O^T = V^T P^T;
//   * K and V tiles go global -> LDS directly (global_load_lds_dwordx4) into a ring of 5 tiles
//     (4 for the 4-wavefront workgroup, 2 with head dimensions above 128);
//     V is kept [key][dim] in LDS and transposed on the way to registers with
//     ds_read_b64_tr_b16; both tiles are XOR-swizzled against bank conflicts;
//   * causal: tiles right of the diagonal are skipped, only tiles crossing it are masked.
#pragma once

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "flash_attention_runs.hpp"

namespace tfk {
namespace {

// Keys per tile.  Above a head dimension of 128 a tile of 64 keys is 64 KiB, of which the LDS holds two; of 32 keys it
// holds the five of the 8-wavefront ring, and the two of either 4-wavefront workgroup of a CU.
__host__ __device__ constexpr int key_tile(int d) { return d <= 128 ? 64 : 32; }
// LDS ring depth: the 8-wavefront kernel keeps two tiles live (its two wavefront sets are half a
// tile apart) and three in flight; the 4-wavefront kernel one live and three in flight, or, with head dimensions above
// 128, one live and one in flight, so that two workgroups share a CU.
__host__ __device__ constexpr int ring_stages(int waves, int d) { return waves == 8 ? 5 : d > 128 ? 2 : 4; }
// Row pitch (in elements) of a [key][dim] tile in LDS: the next power of two.  The swizzles XOR
// chunk indices, which needs a power-of-two chunk count, and a 1 KiB request must cover whole
// rows.  A head dimension of 96 is kept in 128-element rows whose last quarter is never read (160 and
// 192 likewise in 256-element rows).
__host__ __device__ constexpr int lds_pitch(int d) { return d <= 64 ? 64 : d <= 128 ? 128 : 256; }

// K tile [kBN][D] (and a transposed V tile [DV][kBN]): 16 consecutive rows reading one logical
// 16-byte chunk hit 16 different bank groups.  The pattern repeats every 16 rows at the latest, so that
// the fragments of different 16-row blocks differ by a constant.
template <int CH>
__host__ __device__ constexpr int swz_k(int row, int c) {
  constexpr int kRowsPer256B = CH >= 16 ? 1 : 16 / CH;
  return c ^ ((row / kRowsPer256B) % (CH > 16 ? 16 : CH));
}
// V tile [kBN][DV] read by transposing 4-row x 16-column blocks: a half wavefront touches 8
// rows x 32 bytes at the same column, which must land in 8 different 32-byte bank windows.
template <int CH>
__host__ __device__ constexpr int swz_v(int row, int c) {
  if constexpr (CH >= 16) return c ^ ((row & 7) << 1);
  return c ^ (((row >> 1) & 3) << 1);
}
// K^T tile [D][64] read the same way, where the half wavefront's 8 rows are 0-3 and 8-11 (or 4-7 and 12-15) of 16.
__host__ __device__ constexpr int swz_kt(int row, int c) {
  return c ^ ((((row >> 1) & 1) | ((row >> 2) & 2)) << 1);
}

// Workgroups of this kernel share a CU in pairs (its LDS and registers hold two).
__host__ __device__ constexpr bool two_on_cu(int waves, int qb, int D, bool kt) {
  return ring_stages(waves, D) == 2 || (D == 64 && (waves == 4 || (qb == 1 && !kt)));
}
// What a workgroup's number stands for (causal; see the kernel).
enum : int { kSingle = 0, kPairs = 1, kByXcd = 2, kFolded = 3 };
constexpr int kCUs = 256;

typedef float float2_t __attribute__((ext_vector_type(2)));
typedef __fp16 fp16x4_t __attribute__((__vector_size__(4 * sizeof(__fp16))));

// The kernel moves 16-bit elements without looking at them; the element type T (half_t or bf16_t)
// only selects the MFMA and the float -> T conversion.
template <typename T>
struct Vec {
  using v2 = T __attribute__((ext_vector_type(2)));
  using v4 = T __attribute__((ext_vector_type(4)));
  using v8 = T __attribute__((ext_vector_type(8)));
};
template <typename T>
TFK_DEVICE float4_t mfma_t(typename Vec<T>::v8 a, typename Vec<T>::v8 b, float4_t c) {
  if constexpr (std::is_same_v<T, bf16_t>) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  else return mfma_16x16x32(a, b, c);
}
// fp16 saturates at its largest finite value (an absurd |Q * scale| must not become inf); bf16
// has the range of fp32.
template <typename T>
TFK_DEVICE T to_elem_saturating(float x) {
  if constexpr (std::is_same_v<T, bf16_t>) return (T)x;
  else return (T)__builtin_amdgcn_fmed3f(x, -65504.f, 65504.f);
}

// `addr` is a 32-bit LDS byte address: integer arithmetic on it (base register + constant)
// folds into the instruction's offset field, pointer arithmetic through a generic pointer
// does not.
template <typename V4>
TFK_DEVICE V4 lds_read_tr4(unsigned addr) {
  fp16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4f16(
      (__attribute__((address_space(3))) fp16x4_t*)(size_t)addr);
  return __builtin_bit_cast(V4, v);
}
template <typename V4>
TFK_DEVICE V4 lds_read_b64(unsigned addr) {
  return *(__attribute__((address_space(3))) const V4*)(size_t)addr;
}
template <typename V8>
TFK_DEVICE V8 lds_read_b128(unsigned addr) {
  return *(__attribute__((address_space(3))) const V8*)(size_t)addr;
}
// Hides how `x` was computed from the optimiser.  Without it the loop-invariant part of
// (stage base + lane offset + constant) is hoisted as one register per read and the constant
// never reaches the offset field.
TFK_DEVICE unsigned opaque(unsigned x) {
  asm volatile("" : "+v"(x));
  return x;
}
// Reduction over the 4 lanes l, l^16, l^32, l^48 that share a query (rare path).
TFK_DEVICE float quad_max(float x) {
  x = fmaxf(x, __shfl_xor(x, 16));
  return fmaxf(x, __shfl_xor(x, 32));
}

// A weight p >= 0 as a 16-bit number cut off behind its last bit and a 16-bit remainder.  The remainder of a
// weight that the 16-bit number holds exactly is the smallest number instead of zero, so that
// both have the weight's sign and an infinite value stays that infinity (zero or a negative remainder
// would make it NaN).
template <typename T>
struct SplitWeight {
  T whole, rest;
};
template <typename T>
TFK_DEVICE SplitWeight<T> split_weight(float p) {
  SplitWeight<T> w;
  float smallest;
  if constexpr (std::is_same_v<T, bf16_t>) {
    w.whole = __builtin_bit_cast(T, (unsigned short)(__builtin_bit_cast(unsigned, p) >> 16));
    smallest = 0x1p-126f;
  } else {
    w.whole = __builtin_bit_cast(T, (unsigned short)__builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_pkrtz(p, 0.f)));
    smallest = 0x1p-24f;
  }
  // p where p is below `smallest` (0 for 0), else the remainder, `smallest` at least
  w.rest = (T)__builtin_amdgcn_fmed3f(p, p - (float)w.whole, smallest);
  return w;
}

// kWavesT wavefronts x 16 * kQB queries per workgroup.  8 x 32 (256 queries) read K and V fragments
// least often per query and put two wavefronts on every SIMD, so one wavefront's softmax
// (VALU) overlaps the other's MFMAs; 8 x 16 and 4 x 16 take less time for a key tile (D = 128: 0.9 and 0.77 us
// against 1.3) but more for a query, and serve problems that do not fill the chip with 256, and head dimensions above 128.
//
// Above 128 (kWide) two 4-wavefront workgroups share a CU, each with a ring of two tiles, so that one's softmax runs
// beside the other's MFMAs: what bounds them then is the LDS reads, 128 KiB a key tile of a workgroup (1024 cycles; its MFMAs
// take 800 on each SIMD).  64 slices of 512 x 4096 x 256, bf16: 290 us with one workgroup a CU, 64 or 128 queries, and a ring
// of four tiles, 256 with two, 203 without the wait of q_is_there; causal, 32 of 1024 x 1024 x 256: 53, 51 and 39.
// The weights enter the second product as a 16-bit number and a 16-bit remainder (pb_rest): rounded to 16
// bits once, against a reference that is raised lazily, they made the result 5% worse (relative error of
// 4 slices of 1024 x 1024 x 256, bf16, against 64 bits: 2.33e-3, against the true running maximum, whose
// weight of 1 has no error, 2.22e-3, with the remainder 1.66e-3).  Raising the reference to every larger
// score instead, which gives 2.22e-3, multiplies all accumulators in most tiles and is slower: causal, 32 slices
// of 1024 x 1024 x 256: 45 us without either, 51 with the remainder, 57 with the true maximum.
// The scale is applied to the fp32 scores there: Q stays as it came, a second rounding of Q
// would make a 16-bit result measurably worse.
//
// kKT: K comes as [D][Lkv].  Its tile keeps that layout in LDS ([D][kBN], 128-byte rows, as the V^T tile) and the
// K fragments are transposed on their way to registers as those of V are: two ds_read_b64_tr_b16 for a
// ds_read_b128, the same bytes.  Bound as the other instances are; the extra read instructions and their
// addresses cost 0-12%, a transposed copy of K in front of the kernel costs more at every size (fp16, us, K
// as [Lkv][D] / as [D][Lkv] / copied first: 64 slices of 4096 x 4096 x 128 444 / 449 / 534, causal 241 / 254 / 340; 16 of
// 1024 x 1024 x 128 29 / 31 / 40; 32 of 100 x 8192 x 128 157 / 176 / 266; 64 of 1336 x 1336 x 64 causal 30 / 31 / 45).
//
// kTail: rows of Q, K, V and O have d < D elements (a multiple of 8, more than D - 32): they are read and written
// as they are, the last reduction step takes zeros for what is missing of Q and K, columns of V beyond d are those of its
// last chunk and are not stored.  The same bits as on operands padded with zeros, without the three padded copies and the
// copy of the result (bf16, us, padded / as they are: 40 slices of 500 x 500 x 80 46 / 13.5, 16 of 4096 x 4096 x 80 125 / 89,
// 32 of 100 x 2048 x 80 68 / 27, 64 of 1024 x 1024 x 80 causal 67 / 25, 32 of 1024 x 1024 x 112 causal 58 / 22; the kernel
// alone on padded operands is 0-5% ahead of the one on rows as they are).  With K as [D][Lkv] such instances were at most 15%
// ahead of a transposed copy in front (none in the largest case), and are left out.
//
// kSplit: a workgroup takes `chunk` keys (whole tiles; the last of a slice's `splits` parts may be shorter) and leaves its
// un-normalised fp32 rows, minus their reference and their weights' sum in `part` (V as it comes, all head dimensions); merge_parts_kernel puts them together.
template <typename T, int D, int DV, bool kKT, bool kVT, bool kCausal, int kWavesT, int kQB, bool kTail, bool kSplit>
__global__ __launch_bounds__(kWavesT * 64, ring_stages(kWavesT, D) == 2 ? 2 : 1) void flash_attention_fwd_kernel(
    const T* __restrict__ Q, const T* __restrict__ K, const T* __restrict__ V,
    T* __restrict__ O, int Lq, int Lkv, float scale_log2, int q_tiles, int total_items, int order, int d, int end, float* __restrict__ part, int splits, int chunk) {
  using V2 = typename Vec<T>::v2;
  using V4 = typename Vec<T>::v4;
  using V8 = typename Vec<T>::v8;
  constexpr bool kWide = D > 128;
  constexpr int kBN = key_tile(D);
  constexpr int kStages = ring_stages(kWavesT, D);
  constexpr bool kPairOnCU = kStages == 2;
  constexpr bool kTwoOnCU = two_on_cu(kWavesT, kQB, D, kKT);
  constexpr int kRowsPerWave = 16 * kQB;  // kQB 16-query blocks per wavefront
  constexpr int kBMq = kWavesT * kRowsPerWave;
  constexpr int DP = lds_pitch(D), DVP = lds_pitch(DV);   // LDS row pitch of the K / natural V tile
  constexpr bool kEnds = kCausal && kBMq > 64;   // (tiles of 64 rows end where the queries end as they are)
  static_assert(!kKT || !kWide, "K^T tiles are 64 keys wide");
  static_assert(!kTail || (D == DV && !kWide && !kKT && !kVT), "");
  static_assert(!kSplit || (!kCausal && !kVT && kWavesT == 4 && kQB == 1), "");
  // A row's reference is set by its first tile with a score above -inf, whichever that is; else by the first tile.
  constexpr bool kLateReference = kWide || kSplit;
  const int d_row = kTail ? d : D, dv_row = kTail ? d : DV;   // elements of a row in memory
  constexpr int kKChunks = kKT ? kBN / 8 : DP / 8;
  constexpr int kVChunks = kVT ? kBN / 8 : DVP / 8;
  constexpr int kKBytes = kKT ? D * kBN * 2 : kBN * DP * 2;
  constexpr int kVBytes = kVT ? DV * kBN * 2 : kBN * DVP * 2;
  constexpr int kStageBytes = kKBytes + kVBytes;
  constexpr int kKB = kBN / 16;   // 16-key blocks per tile (rows of S^T)
  constexpr int kKK = D / 32;     // reduction steps of S^T = K Q^T
  constexpr int kDB = DV / 16;    // 16-wide blocks of the head dimension (rows of O^T)
  constexpr int kJ = kBN / 32;    // reduction steps of O^T += V^T P^T
  constexpr int kKInstr = kKBytes / 1024;            // 1 KiB wavefront loads per K tile
  constexpr int kVInstr = kVBytes / 1024;
  constexpr int kKPerWave = (kKInstr + kWavesT - 1) / kWavesT;
  constexpr int kVPerWave = (kVInstr + kWavesT - 1) / kWavesT;
  constexpr int kLoadsPerTile = kKPerWave + kVPerWave;  // per wavefront (idle slots re-load)
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  // Workgroup ids are dealt round-robin to the 8 XCDs, each with its own L2: id % 8 is the XCD,
  // id / 8 the position in that XCD's queue.  Work is arranged so that the query tiles of a
  // slice stream the same K/V through ONE L2 instead of eight.
  //   non-causal: items in slice-major order, cut into 8 contiguous chunks (the last one may
  //               be short; its surplus workgroups exit at once);
  //   causal:     work per query tile grows with its position, so a workgroup takes query
  //               tile q_tiles-1-p and then tile p of the same slice: every workgroup does the
  //               same amount of work, no sorting by weight is needed and the slice-major
  //               order (with its L2 locality) is kept.  Where that is done sooner (the
  //               caller tells) and with an odd number of query tiles, one tile per workgroup,
  //               heaviest first over all slices (kSingle) or over those of an XCD (kByXcd).
  //               Where two share a CU (the p-th and the (p + 256)-th, by a probe) and few are left for a third, the second 256 come
  //               lightest first (kFolded), or the heaviest would share their CUs with ones half as heavy and all others
  //               wait: 32 slices of 1024 x 1024 x 256 37.2 / 35.9 us, 18 of 1600 51.1 / 48.2, 9 of 3584 x 160 78 / 75, 33 of 2048 x 64 33.1 /
  //               30.2, 28 of 2176 x 64 29.7 / 27.8; 77 of D = 64 with 257 to 576 workgroups 0.985. With more than 576 those of the
  //               third round find the light CUs by themselves.
  int qt_of_pass[2] = {0, 0};
  int num_passes = 1;
  size_t bh;
  int split = 0;
  if (!kCausal || order == kPairs) {
    const int per_slice = kCausal ? q_tiles / 2 : q_tiles;
    const int per_xcd = (total_items + 7) / 8;
    const int item = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
    if (item >= total_items) return;
    const int p = item % per_slice;
    bh = item / per_slice;
    if constexpr (kSplit) {
      split = (int)(bh % splits);
      bh /= splits;
    }
    if (kCausal) {
      qt_of_pass[0] = q_tiles - 1 - p;
      qt_of_pass[1] = p;
      num_passes = 2;
    } else {
      qt_of_pass[0] = p;
    }
  } else {
    const int slices = total_items / q_tiles;
    if (order == kByXcd) {
      const int xcd = (int)blockIdx.x % 8, p = (int)blockIdx.x / 8;
      const int own = (slices - xcd + 7) / 8;   // slices of this XCD
      if (p >= own * q_tiles) return;
      qt_of_pass[0] = q_tiles - 1 - p / own;
      bh = xcd + 8 * (p % own);
    } else {
      int i = (int)blockIdx.x;
      if (i >= total_items) return;
      if constexpr (kTwoOnCU) {
        // the second 256 in the opposite order (by eights: a slice's stay on one XCD)
        const int j = i - kCUs, count = min(total_items - kCUs, kCUs) & ~7;
        if (order == kFolded && (unsigned)j < (unsigned)count) i = kCUs + (count - 8) - (j & ~7) + (j & 7);
      }
      qt_of_pass[0] = q_tiles - 1 - i / slices;
      bh = i % slices;
    }
  }
  Q += bh * (size_t)Lq * d_row;
  K += bh * (size_t)Lkv * d_row;
  V += bh * (size_t)Lkv * dv_row;
  O += bh * (size_t)Lq * dv_row;

  const int kv_pitch = Lkv;   // row length of a transposed K or V
  if constexpr (kSplit) {
    K += (size_t)split * chunk * (kKT ? 1 : d_row);
    V += (size_t)split * chunk * dv_row;
    Lkv = min(chunk, Lkv - split * chunk);
  }

  for (int pass = 0; pass < num_passes; ++pass) {
  const int qt = qt_of_pass[pass];
  const int tile_row0 = kEnds ? 64 * end - (q_tiles - qt) * kBMq : qt * kBMq;   // (below 0 where the caller says so)
  const int q_row0 = tile_row0 + wave * kRowsPerWave;  // first query row of this wavefront
  // this lane's query rows: block qb holds row q_row0 + 16*qb + lr

  // The softmax scale (times log2 e) is folded into Q once: Q' = fp16(Q * scale_log2), so the
  // MFMA result is already in log2 units; and each score accumulator starts at minus the
  // row's reference maximum instead of zero, so the MFMA result IS the exp2 argument - no
  // per-score multiply or subtract is left in the tile loop.
  // Q^T fragments (B operand): lane holds Q'[row][32*kk + 8*lg .. +7]
  V8 qf[kKK][kQB];
#pragma unroll
  for (int qb = 0; qb < kQB; ++qb) {
    const int m = q_row0 + 16 * qb + lr, m_ld = kEnds ? (int)min((unsigned)m, (unsigned)Lq - 1u) : min(m, Lq - 1);   // (m < 0, too)
#pragma unroll
    for (int kk = 0; kk < kKK; ++kk) {
      const int col = kk * 32 + lg * 8;
      V8 raw = *reinterpret_cast<const V8*>(Q + (size_t)m_ld * d_row + (kTail ? min(col, d_row - 8) : col));
      if (kTail && col >= d_row) raw = V8{};
      if constexpr (kWide) {
        qf[kk][qb] = raw;
      } else {
#pragma unroll
        for (int t = 0; t < 8; ++t) qf[kk][qb][t] = to_elem_saturating<T>((float)raw[t] * scale_log2);
      }
    }
  }

  int n_end = Lkv;
  if (kCausal) n_end = min(Lkv, tile_row0 + kBMq);
  const int num_tiles = (n_end + kBN - 1) / kBN;

  // ---- global -> LDS plan: wavefront instruction i of a tile covers 1 KiB of it ------------
  // Request r of a wavefront (r < kKPerWave: K tile, else V tile) is one instruction: scalar
  // base (start of the tile in global memory) + a per-lane 32-bit offset computed once here.
  // Only a tile that crosses the end of the keys takes the slow form with clamped addresses.
  const unsigned smem_base = lds_address(smem);
  const int k_last = d_row / 8 - 1, v_last = dv_row / 8 - 1;   // last 16-byte chunk of a row
  unsigned req_off[kLoadsPerTile];   // per-lane byte offset inside the tile (global side)
  unsigned req_lds[kLoadsPerTile];   // wave-uniform byte offset inside the stage (LDS side)
#pragma unroll
  for (int t = 0; t < kKPerWave; ++t) {
    const int i = (wave + kWavesT * t) % kKInstr;
    constexpr int kRowsPerInstr = 64 / kKChunks;
    const int row = i * kRowsPerInstr + lane / kKChunks;
    if constexpr (kKT)  // K^T tile: [D][kBN] out of a [D][Lkv] matrix
      req_off[t] = ((unsigned)row * (unsigned)kv_pitch + swz_kt(row, lane % kKChunks) * 8) * 2u;
    else                // K tile: [kBN][D]
      // (a physical chunk whose logical chunk lies beyond the row is never read: it re-fetches the last one)
      req_off[t] = (unsigned)(row * d_row + min(swz_k<kKChunks>(row, lane % kKChunks), k_last) * 8) * 2u;
    req_lds[t] = i * 1024;
  }
#pragma unroll
  for (int t = 0; t < kVPerWave; ++t) {
    const int i = (wave + kWavesT * t) % kVInstr;
    constexpr int kRowsPerInstr = 64 / kVChunks;
    const int row = i * kRowsPerInstr + lane / kVChunks;
    if constexpr (!kVT)  // V tile: [kBN][DV]
      req_off[kKPerWave + t] = (unsigned)(row * dv_row + min(swz_v<kVChunks>(row, lane % kVChunks), v_last) * 8) * 2u;
    else                 // V^T tile: [DV][kBN] out of a [DV][Lkv] matrix
      req_off[kKPerWave + t] = ((unsigned)row * (unsigned)kv_pitch + swz_k<kVChunks>(row, lane % kVChunks) * 8) * 2u;
    req_lds[kKPerWave + t] = kKBytes + i * 1024;
  }
  auto issue_request = [&](int tile, int r) __attribute__((always_inline)) {
    const int n0 = min(tile, num_tiles - 1) * kBN;  // clamped past the end (never read)
    const unsigned dst = smem_base + (tile % kStages) * kStageBytes + req_lds[r];
    if (n0 + kBN <= Lkv) {
      const char* base = r < kKPerWave ? reinterpret_cast<const char*>(K + (size_t)n0 * (kKT ? 1 : d_row))
                         : kVT         ? reinterpret_cast<const char*>(V + n0)
                                       : reinterpret_cast<const char*>(V + (size_t)n0 * dv_row);
      // the LDS destination is an M0 INPUT of the statement: the compiler writes M0 itself and
      // cannot use the register for anything else between that write and the request; the
      // s_nop is the wait state an M0 write needs in front of an LDS-direct load
      asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                   :
                   : "v"(req_off[r]), "s"(base), "{m0}"(dst)
                   : "memory");
      return;
    }
    if (r < kKPerWave) {
      const int i = (wave + kWavesT * r) % kKInstr;
      constexpr int kRowsPerInstr = 64 / kKChunks;
      const int row = i * kRowsPerInstr + lane / kKChunks;
      if constexpr (kKT) {
        const int gc = min(n0 + swz_kt(row, lane % kKChunks) * 8, Lkv - 8);
        lds_dma_16B(K + (size_t)row * kv_pitch + gc, dst);
      } else {
        const int cc = min(swz_k<kKChunks>(row, lane % kKChunks), k_last);
        const int gr = min(n0 + row, Lkv - 1);
        lds_dma_16B(K + (size_t)gr * d_row + cc * 8, dst);
      }
    } else {
      const int i = (wave + kWavesT * (r - kKPerWave)) % kVInstr;
      constexpr int kRowsPerInstr = 64 / kVChunks;
      const int row = i * kRowsPerInstr + lane / kVChunks;
      if constexpr (!kVT) {
        const int cc = min(swz_v<kVChunks>(row, lane % kVChunks), v_last);
        const int gr = min(n0 + row, Lkv - 1);
        lds_dma_16B(V + (size_t)gr * dv_row + cc * 8, dst);
      } else {
        const int cc = swz_k<kVChunks>(row, lane % kVChunks);
        const int gc = min(n0 + cc * 8, Lkv - 8);
        lds_dma_16B(V + (size_t)row * kv_pitch + gc, dst);
      }
    }
  };
  // The same request for a tile known to lie wholly inside the key range: no clamping, no
  // branch.  The tile loop uses this form wherever it can, because the bookkeeping of the
  // general form (~30 scalar instructions and two branches per request) is issued between
  // MFMAs of a wavefront that has the matrix pipe to itself at that moment: it cost ~100
  // cycles per request with the pipe idle.
  auto issue_request_lean = [&](int tile, int r) __attribute__((always_inline)) {
    const unsigned dst = smem_base + (tile % kStages) * kStageBytes + req_lds[r];
    const char* base = r < kKPerWave ? reinterpret_cast<const char*>(K) + (size_t)tile * (kBN * (kKT ? 1 : d_row) * 2)
                       : kVT         ? reinterpret_cast<const char*>(V) + (size_t)tile * (kBN * 2)
                                     : reinterpret_cast<const char*>(V) + (size_t)tile * (kBN * dv_row * 2);
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(req_off[r]), "s"(base), "{m0}"(dst)
                 : "memory");
  };
  auto issue_tile_loads = [&](int tile) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < kLoadsPerTile; ++r) issue_request(tile, r);
  };

  // ---- LDS -> register plan -----------------------------------------------------------------
  // Every fragment read is (stage base) + (per-lane offset) + (compile-time immediate): the
  // swizzles only XOR lane-dependent bits into the chunk index, so the lane part is computed
  // once here and the tile loop spends no VALU on addresses beyond adding the stage base.
  //   K fragment (kb, kk) - A operand, 16 keys x 32 dims: row 16*kb + lr, logical chunk 4*kk + lg.
  //     K kept [dim][key]: rows 32*kk + 8*lg (+4) .. +3, columns 16*kb .. +15, transposed by the read; lane r of
  //     a 16-lane group addresses row r/4, columns 4*(r%4) .. +3 of that block.  The lane part is kept per kb.
  //     (256-element rows: the swizzles reach the low 16 of 32 chunks, so that steps and blocks half a row apart
  //     differ by a constant and share an offset)
  constexpr int kKOffs = kKT ? kKB : kKChunks > 16 ? 4 : kKK;
  unsigned k_off[kKOffs];
  if constexpr (kKT) {
    const int row_l = 8 * lg + (lr >> 2);
#pragma unroll
    for (int kb = 0; kb < kKB; ++kb) {
      const int col = kb * 16 + 4 * (lr & 3);
      k_off[kb] = row_l * kBN * 2 + swz_kt(row_l, col / 8) * 16 + (col % 8) * 2;
    }
  } else {
#pragma unroll
    for (int kk = 0; kk < kKOffs; ++kk) k_off[kk] = lr * DP * 2 + swz_k<kKChunks>(lr, 4 * kk + lg) * 16;
  }
  //   Reduction step j of the second product covers keys 32*j .. +31; slot t of lane group lg
  //   is key 32*j + 4*lg + t (t < 4) or 32*j + 16 + 4*lg + (t - 4): exactly the keys whose
  //   scores the lane already holds in its accumulators of key blocks 2*j and 2*j + 1.
  //   V fragment (db, j) - A operand, 16 dims x 32 keys.
  //     V kept [key][dim]: each 16-lane group transposes the 4 x 16 block of rows
  //     32*j + 4*lg (+16) .. +3, columns 16*db .. +15; lane r of the group addresses row r/4,
  //     columns 4*(r%4) .. +3 of that block.  One offset per (db & 1, db / 2 via XOR) would not
  //     be constant, so the lane part is kept per db.
  //     V kept [dim][key]: row 16*db + lr, keys 32*j + 4*lg (+16) .. +3 (8 bytes each).
  constexpr int kVOffs = kVT ? 2 * kJ : kVChunks > 16 ? 8 : kDB;
  unsigned v_off[kVOffs];
  if constexpr (!kVT) {
    const int row_l = 4 * lg + (lr >> 2);
#pragma unroll
    for (int db = 0; db < kVOffs; ++db) {
      const int col = db * 16 + 4 * (lr & 3);
      v_off[db] = row_l * DVP * 2 + swz_v<kVChunks>(row_l, col / 8) * 16 + (col % 8) * 2;
    }
  } else {
#pragma unroll
    for (int x = 0; x < 2 * kJ; ++x) {  // x = 2*j + half: keys 32*j + 16*half + 4*lg .. +3
      const int key = 16 * x + 4 * lg;
      v_off[x] = lr * kBN * 2 + swz_k<kVChunks>(lr, key / 8) * 16 + (key % 8) * 2;
    }
  }

  float4_t o_acc[kDB][kQB];
#pragma unroll
  for (int db = 0; db < kDB; ++db)
#pragma unroll
    for (int qb = 0; qb < kQB; ++qb) o_acc[db][qb] = float4_t{0.f, 0.f, 0.f, 0.f};
  // neg_m: minus the reference maximum of a row's scaled scores (the accumulator start value);
  // l_acc: the running sum of a row's weights, kept as one more accumulator block of the second
  // product (a block of V^T whose 16 rows are all ones): the matrix pipe adds up the 16-bit
  // weights that actually multiply V.  Every register of l_acc[qb] holds the sum of row lr.
  // (A v_dot2 per pair of weights, the obvious VALU form, takes ~20 cycles per instruction while
  // another wavefront of the SIMD streams MFMAs - against 8 for an ordinary VALU instruction.)
  float neg_m[kQB];
  float4_t l_acc[kQB];
  bool unset[kQB];    // kLateReference: no finite score seen yet (the row's reference is not set)
#pragma unroll
  for (int qb = 0; qb < kQB; ++qb) {
    unset[qb] = true;
    neg_m[qb] = 0.f;  // reference 0 until the first tile raises it
    l_acc[qb] = float4_t{0.f, 0.f, 0.f, 0.f};
  }
  V8 ones_frag;
#pragma unroll
  for (int t = 0; t < 8; ++t) ones_frag[t] = (T)1.f;

  float4_t s[kKB][kQB];  // scores of the tile in flight
  // Operand fragments are requested from LDS one step ahead of the MFMAs that use them, into
  // ping-pong registers, so that LDS latency is covered by the previous step's MFMAs (or by
  // the softmax arithmetic) instead of stalling the wavefront in front of every MFMA group.
  // kWide: few MFMAs a step, so K fragments are requested two steps ahead where the registers hold them, and the V
  // fragments during the QK product, behind whose MFMAs they arrive (causal, D = 256, with one wavefront a SIMD and before the
  // weights had a remainder: 32 slices of 1024 x 1024 52.5 -> 47.0 us, 8 of 4096 173 -> 157; D = 160: 46.2 -> 44.8).
  constexpr int kKAhead = kWide && D <= 192 && kWavesT == 4 ? 2 : 1;
  V8 kf[kKAhead + 1][kKB];   // K fragments of reduction step kk (buffer kk % (kKAhead + 1))
  // kTail: all ones where this lane's dims of the last reduction step exist (K may hold infinities there)
  const int tail_mask = kTail && (kKK - 1) * 32 + lg * 8 >= d_row ? 0 : -1;
  auto k_frag = [&](int buf, int kk, int kb) __attribute__((always_inline)) {
    if constexpr (kTail) {
      typedef int int4v_t __attribute__((ext_vector_type(4)));
      if (kk == kKK - 1) return __builtin_bit_cast(V8, __builtin_bit_cast(int4v_t, kf[buf][kb]) & tail_mask);
    }
    return kf[buf][kb];
  };
  V8 vf[kJ > 1 ? 2 : 1][kDB];   // V fragments of reduction step j (buffer j & 1)
  // lane address of the fragments of step kk (kKT: recomputed per fragment)
  auto k_addr = [&](int it, int kk) __attribute__((always_inline)) {
    const unsigned stage_base = smem_base + (it % kStages) * kStageBytes;
    return kKT ? stage_base : opaque(stage_base + k_off[kk % kKOffs]) + kk / kKOffs * 256;
  };
  auto k_read = [&](int buf, unsigned ka, int kk, int kb) __attribute__((always_inline)) {
    if constexpr (kKT) {
      const unsigned a = opaque(ka + k_off[kb]) + 32 * kk * kBN * 2;
      const V4 lo = lds_read_tr4<V4>(a), hi = lds_read_tr4<V4>(a + 4 * kBN * 2);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        kf[buf][kb][t] = lo[t];
        kf[buf][kb][4 + t] = hi[t];
      }
    } else {
      kf[buf][kb] = lds_read_b128<V8>(ka + kb * 16 * DP * 2);
    }
  };
  auto k_reads = [&](int buf, int it, int kk) __attribute__((always_inline)) {
    const unsigned ka = k_addr(it, kk);
#pragma unroll
    for (int kb = 0; kb < kKB; ++kb) k_read(buf, ka, kk, kb);
  };
  auto first_k_reads = [&](int it) __attribute__((always_inline)) {
#pragma unroll
    for (int kk = 0; kk < kKAhead; ++kk) k_reads(kk, it, kk);
  };
  auto v_read = [&](int buf, int it, int j, int db) __attribute__((always_inline)) {
    const unsigned stage_base = smem_base + (it % kStages) * kStageBytes;
    {
      V4 lo, hi;
      if constexpr (!kVT) {
        const unsigned va = opaque(stage_base + v_off[db % kVOffs]) + db / kVOffs * 256 + kKBytes;
        lo = lds_read_tr4<V4>(va + (32 * j) * DVP * 2);
        hi = lds_read_tr4<V4>(va + (32 * j + 16) * DVP * 2);
      } else {
        lo = lds_read_b64<V4>(opaque(stage_base + v_off[2 * j]) + kKBytes + db * 16 * kBN * 2);
        hi = lds_read_b64<V4>(opaque(stage_base + v_off[2 * j + 1]) + kKBytes + db * 16 * kBN * 2);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        vf[buf][db][t] = lo[t];
        vf[buf][db][4 + t] = hi[t];
      }
    }
  };
  auto v_reads = [&](int buf, int it, int j) __attribute__((always_inline)) {
#pragma unroll
    for (int db = 0; db < kDB; ++db) v_read(buf, it, j, db);
  };
  // ---- S^T = K Q'^T - m: s[kb][qb][r] = log2-scaled score of key kBN*it + 16*kb + 4*lg + r
  //      against row lr of query block qb, minus that row's reference maximum.  Expects the
  //      fragments of step kk = 0 to be on their way into kf[0]. ---------------------------
  //      req_tile >= 0: that tile's requests are issued between the reduction steps.
  //      lean_c: the requested tile is a whole tile inside the key range (lean request form).
  //      The fragment reads of the next reduction step and the requests sit BETWEEN the MFMAs
  //      (one piece behind each pair): a wavefront issues in order, so anything clustered
  //      between two reduction steps runs with the matrix pipe drained.
  auto qk_tile = [&](int it, int req_tile, auto lean_c) __attribute__((always_inline)) {
    constexpr bool kLean = decltype(lean_c)::value;
#pragma unroll
    for (int kb = 0; kb < kKB; ++kb)
#pragma unroll
      for (int qb = 0; qb < kQB; ++qb) {
        const float start = kWide ? 0.f : neg_m[qb];
        s[kb][qb] = float4_t{start, start, start, start};
      }
#pragma unroll
    for (int kk = 0; kk < kKK; ++kk) {
      const int next = kk + kKAhead;
      const unsigned ka = next < kKK ? k_addr(it, next < kKK ? next : 0) : 0u;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kb = 0; kb < kKB; ++kb) {
        const V8 k_now = k_frag(kk % (kKAhead + 1), kk, kb);
#pragma unroll
        for (int qb = 0; qb < kQB; ++qb) s[kb][qb] = mfma_t<T>(k_now, qf[kk][qb], s[kb][qb]);
        if (next < kKK) k_read(next % (kKAhead + 1), ka, next, kb);
        if constexpr (kWide) {
#pragma unroll
          for (int db = 0; db < kDB; ++db)
            if ((db * kKK * kKB) / kDB == kk * kKB + kb) v_read(0, it, 0, db);
        }
        if (req_tile >= 0) {
#pragma unroll
          for (int r = 0; r < kLoadsPerTile; ++r)
            if ((r * kKK * kKB) / kLoadsPerTile == kk * kKB + kb) {
              if constexpr (kLean) issue_request_lean(req_tile, r);
              else issue_request(req_tile, r);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  V8 pb[kJ][kQB];  // 16-bit weights, B operand of the second product
  V8 pb_rest[kJ][kQB];   // kWide: what their rounding left out, rounded in turn
  // ---- mask, online softmax, fp16 weights.  Requests the V fragments of step j = 0 (unless kWide). -------
  auto softmax_tile = [&](int it, auto mask_c) __attribute__((always_inline)) {
    constexpr bool kMask = decltype(mask_c)::value;
    const int n0 = it * kBN;
    if constexpr (!kWide) v_reads(0, it, 0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kWide) {
#pragma unroll
      for (int kb = 0; kb < kKB; ++kb)
#pragma unroll
        for (int qb = 0; qb < kQB; ++qb)
#pragma unroll
          for (int r = 0; r < 4; ++r) s[kb][qb][r] = fmaf(s[kb][qb][r], scale_log2, neg_m[qb]);
    }
    // ---- mask -------------------------------------------------------------------------
    if constexpr (kMask) {
#pragma unroll
      for (int kb = 0; kb < kKB; ++kb)
#pragma unroll
        for (int qb = 0; qb < kQB; ++qb)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int n = n0 + kb * 16 + 4 * lg + r;
            if (n >= Lkv || (kCausal && n > q_row0 + 16 * qb + lr)) s[kb][qb][r] = -INFINITY;
          }
    }

    // ---- online softmax: p = exp2(s) ---------------------------------------------------
    // Lazy reference: the reference maximum is only raised when some lane sees a score more
    // than kLazy (log2 units) above it.  Until then p may reach 2^kLazy, which fp16 P and the
    // fp32 sums hold easily, and the final O / l is unchanged because O and l share the
    // reference.  The check needs no cross-lane traffic: it looks at each lane's own 16 keys;
    // only when it fires are the 4 lanes that share a query reduced, every O accumulator
    // multiplied and this tile's scores re-based.
    // kWide, fp16: weights are taken 2^7 times as large (up to 2^15), which leaves the smallest remainder
    // at 2^-31 of the largest weight.
    constexpr float kUp = kWide && !std::is_same_v<T, bf16_t> ? 7.f : 0.f;
    constexpr float kLazy = kUp + 8.f;
    float mx[kQB];
    bool grow = false;
#pragma unroll
    for (int qb = 0; qb < kQB; ++qb) {
      mx[qb] = s[0][qb][0];
#pragma unroll
      for (int kb = 0; kb < kKB; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx[qb] = fmaxf(mx[qb], s[kb][qb][r]);
      grow |= mx[qb] > kLazy;
      if constexpr (kLateReference) grow |= unset[qb];
    }
    // The first tile sets the reference to the row's true maximum, whichever way that is from
    // the initial 0 (every row has at least key 0 unmasked there; nothing is accumulated yet).
    // kLateReference: a row whose scores were all -inf so far takes its reference from the first tile that has another.
    const bool first = !kLateReference && it == 0;
    if (first || __builtin_amdgcn_ballot_w64(grow) != 0) {
#pragma unroll
      for (int qb = 0; qb < kQB; ++qb) {
        const float qmax = quad_max(mx[qb]) - kUp;
        const bool set = kLateReference ? unset[qb] : first;
        float shift = set ? qmax : fmaxf(0.f, qmax);  // afterwards the reference only rises
        const float alpha = set ? 1.f : __builtin_amdgcn_exp2f(-shift);
        if constexpr (kLateReference) {
          if (set && qmax == -INFINITY) shift = 0.f;
          unset[qb] = set && qmax == -INFINITY;
        }
        l_acc[qb] *= alpha;
#pragma unroll
        for (int db = 0; db < kDB; ++db) o_acc[db][qb] *= alpha;
#pragma unroll
        for (int kb = 0; kb < kKB; ++kb) s[kb][qb] -= shift;
        neg_m[qb] -= shift;
      }
    }
#pragma unroll
    for (int qb = 0; qb < kQB; ++qb)
#pragma unroll
      for (int kb = 0; kb < kKB; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) s[kb][qb][r] = __builtin_amdgcn_exp2f(s[kb][qb][r]);

#pragma unroll
    for (int j = 0; j < kJ; ++j)
#pragma unroll
      for (int qb = 0; qb < kQB; ++qb) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          if constexpr (kWide) {
            const SplitWeight<T> lo = split_weight<T>(s[2 * j][qb][t]), hi = split_weight<T>(s[2 * j + 1][qb][t]);
            pb[j][qb][t] = lo.whole;
            pb_rest[j][qb][t] = lo.rest;
            pb[j][qb][4 + t] = hi.whole;
            pb_rest[j][qb][4 + t] = hi.rest;
          } else {
            pb[j][qb][t] = (T)s[2 * j][qb][t];
            pb[j][qb][4 + t] = (T)s[2 * j + 1][qb][t];
          }
        }
      }
    __builtin_amdgcn_sched_barrier(0);
  };
  // ---- O^T += V^T P^T; during its last step the K fragments (kk = 0) of tile `it_next`
  //      are requested for the QK phase that follows ------------------------------------------
  auto pv_tile = [&](int it, int it_next) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < kJ; ++j) {
      if (j + 1 < kJ) v_reads((j + 1) & 1, it, j + 1);
      else if (!kPairOnCU) first_k_reads(it_next);
#pragma unroll
      for (int db = 0; db < kDB; ++db)
#pragma unroll
        for (int qb = 0; qb < kQB; ++qb) o_acc[db][qb] = mfma_t<T>(vf[j & 1][db], pb[j][qb], o_acc[db][qb]);
#pragma unroll
      for (int qb = 0; qb < kQB; ++qb) l_acc[qb] = mfma_t<T>(ones_frag, pb[j][qb], l_acc[qb]);
      if constexpr (kWide) {
#pragma unroll
        for (int db = 0; db < kDB; ++db)
#pragma unroll
          for (int qb = 0; qb < kQB; ++qb) o_acc[db][qb] = mfma_t<T>(vf[j & 1][db], pb_rest[j][qb], o_acc[db][qb]);
#pragma unroll
        for (int qb = 0; qb < kQB; ++qb) l_acc[qb] = mfma_t<T>(ones_frag, pb_rest[j][qb], l_acc[qb]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // kWide: Q comes into its registers as it is, and the compiler would wait for it at its first use, in the tile loop
  // and in every iteration: a wait for vmcnt(0), which there drains the requests of the tiles ahead (64 slices of
  // 512 x 4096 x 256: 256 us with it, 203 without).  This is a use in front of the loop.
  auto q_is_there = [&]() __attribute__((always_inline)) {
    if constexpr (kWide) {
#pragma unroll
      for (int kk = 0; kk < kKK; ++kk)
#pragma unroll
        for (int qb = 0; qb < kQB; ++qb) asm volatile("" : "+v"(qf[kk][qb]));
    }
  };
  // Tiles [0, n_plain) need no mask for this wavefront's rows, [n_plain, n_compute) cross
  // the diagonal or the end of the keys, and [n_compute, num_tiles) lie above the diagonal:
  // the wavefront only keeps the ring (barrier + loads) going for its workgroup.
  int n_plain = min(num_tiles, Lkv / kBN);
  int n_compute = num_tiles;
  if (kCausal) {
    n_plain = max(0, min(n_plain, (q_row0 + 1) / kBN));
    n_compute = min(num_tiles, (q_row0 + kRowsPerWave - 1) / kBN + 1);
    if ((unsigned)q_row0 >= (unsigned)Lq) n_plain = n_compute = 0;   // (all rows in front of the first query or behind the last)
  }
  const int n_fast = min(num_tiles, Lkv / kBN);  // whole tiles of this pass (lean request form)
  if constexpr (kWavesT == 8) {
    // Two wavefronts share a SIMD (w and w + 4) and a SIMD has one matrix pipe and one VALU, so
    // the two SETS of wavefronts (0-3, 4-7) run the same loop half a tile apart, in time slots
    // fenced by two workgroup barriers per tile:
    //     slot 2t   : set 0: PV(t-1), QK(t)  [MFMA]      set 1: softmax(t-1)     [VALU]
    //     slot 2t+1 : set 0: softmax(t)      [VALU]      set 1: PV(t-1), QK(t)   [MFMA]
    // While one wavefront of a SIMD streams its 64 MFMAs the other one does its exp2 / convert
    // work, and neither pipe waits for the other: measured per tile, a wavefront's MFMA block
    // takes ~1100-1200 cycles and its softmax ~1000 while the partner's MFMAs run (VALU
    // instructions issue at half rate then), against ~3500 for an arrangement that lets the
    // phases of the two wavefronts drift (QK, softmax and PV of both then run one after another).
    // Without the second barrier the sets do drift: the hardware issues from the older wavefront
    // first and whichever set gets ahead keeps the matrix pipe.
    // Ring of 5 tiles: tile t is read from slot 2t (QK by set 0) to slot 2t+3 (PV by set 1), so
    // two tiles are live and three are in flight.  QK(t) carries the requests of tile t+3, which
    // go into the stage of tile t-2 (last read in slot 2t-1).  The barrier behind an MFMA block
    // (after QK(t+1) has requested tile t+4) waits until only tiles t+3, t+4 are in flight: tile
    // t+2 has then landed, one slot before the first wavefront reads it.
#pragma unroll
    for (int t = 0; t < 3; ++t) issue_tile_loads(t);
    barrier_keep_vmem<2 * kLoadsPerTile>();  // tile 0 has landed
    q_is_there();
    const bool second_set = wave >= 4;
    if (second_set) barrier_only();  // slot 0: set 0 alone
    first_k_reads(0);
    if (n_compute > 0) qk_tile(0, 3, std::false_type{});
    else issue_tile_loads(3);
    auto tile_step = [&](int t, auto mask_c, auto lean_c) __attribute__((always_inline)) {
      barrier_keep_vmem<2 * kLoadsPerTile>();  // tile t+1 has landed (own loads; then everyone's)
      softmax_tile(t, mask_c);
      barrier_only();  // the V fragments requested by softmax_tile stay in flight across it
      // Raised issue priority for the MFMA block: the arbiter serves the older wavefront first, so
      // without it the MFMA blocks of set 1 lose issue slots to the softmax of set 0 (~1700 against
      // ~1480 cycles per block).  It buys 7% in cycles and 1-2% in time: the kernel runs at the
      // power limit, and the shader clock gives back most of what a denser schedule saves.
      __builtin_amdgcn_s_setprio(2);
      pv_tile(t, t + 1);
      if (t + 1 < n_compute) qk_tile(t + 1, t + 4, lean_c);
      else issue_tile_loads(t + 4);
      __builtin_amdgcn_s_setprio(0);
    };
    // [0, n_lean): unmasked tile, a QK product follows and its requests (tile t+4) are whole tiles
    const int n_lean = min(min(n_plain, n_compute - 1), n_fast - 4);
    int t = 0;
    for (; t < n_lean; ++t) tile_step(t, std::false_type{}, std::true_type{});
    for (; t < n_plain; ++t) tile_step(t, std::false_type{}, std::false_type{});
    for (; t < n_compute; ++t) tile_step(t, std::true_type{}, std::false_type{});
    for (; t < num_tiles; ++t) {  // above the diagonal: keep the ring and the barriers going
      barrier_keep_vmem<2 * kLoadsPerTile>();
      barrier_only();
      issue_tile_loads(t + 4);
    }
    if (!second_set) barrier_only();  // the slot in which set 1 finishes its last tile
  } else {
    // One wavefront of the workgroup per SIMD.  Ring of 4 tiles: iteration `it` starts with the ring barrier (tiles
    // it and it+1 have landed, the stage of tile it-1 is free) and QK(it) carries the requests of tile it+3.
    // Two stages (kPairOnCU): tile it has landed, and QK(it) carries the requests of tile it+1.
#pragma unroll
    for (int t = 0; t < kStages - 1; ++t) issue_tile_loads(t);
    barrier_keep_vmem<(kStages - 2) * kLoadsPerTile>();  // tile 0 has landed
    q_is_there();
    auto ring_barrier = [&](int it) __attribute__((always_inline)) {
      barrier_keep_vmem<kPairOnCU ? 0 : (kStages - 3) * kLoadsPerTile>();
      if (kPairOnCU) first_k_reads(it);
    };
    const int n_lean = min(n_plain, n_fast - (kStages - 1));
    int it = 0;
    if (!kPairOnCU) first_k_reads(0);
    for (; it < n_lean; ++it) {
      ring_barrier(it);
      qk_tile(it, it + kStages - 1, std::true_type{});
      softmax_tile(it, std::false_type{});
      pv_tile(it, it + 1);
    }
    for (; it < n_plain; ++it) {
      ring_barrier(it);
      qk_tile(it, it + kStages - 1, std::false_type{});
      softmax_tile(it, std::false_type{});
      pv_tile(it, it + 1);
    }
    for (; it < n_compute; ++it) {
      ring_barrier(it);
      qk_tile(it, it + kStages - 1, std::false_type{});
      softmax_tile(it, std::true_type{});
      pv_tile(it, it + 1);
    }
    for (; it < num_tiles; ++it) {
      ring_barrier(it);
      issue_tile_loads(it + kStages - 1);
    }
  }
  wait_vmem_all();  // the clamped tail loads must not outlive the workgroup's LDS

  // ---- epilogue: O[m][16*db + 4*lg + r] = O^T / l ------------------------------------------
  // A lane holds 4 consecutive head dims of row lr for every 16-wide block db.  Stored as they
  // are, a store instruction writes 16 rows x 32 bytes with the four lanes of a row 16 lane
  // ids apart, and the address unit only merges ADJACENT lanes: 64 accesses per instruction.
  // The data is therefore re-dealt first, a pair of blocks (db, db+1) at a time: the 16-lane
  // groups g and g^1 trade halves (v_permlane16_swap), after which groups 0/2 hold dims 0-7 /
  // 8-15 of block db and groups 1/3 the same of block db+1, 16 bytes per lane; ds_bpermute then
  // moves the 16 bytes of (row r, segment s) to lane 4*r + s, and four adjacent lanes store 64
  // contiguous bytes of a row.
  if constexpr (kSplit) {
    // (fp32: the 64 bytes that four lanes of a row hold are stored as they are)
    const size_t rows = (size_t)(total_items / q_tiles / splits) * Lq;
    const int m_row = q_row0 + lr;
    if (m_row < Lq) {
      const size_t row = split * rows + bh * Lq + m_row;
#pragma unroll
      for (int db = 0; db < kDB; ++db) *reinterpret_cast<float4_t*>(part + row * DV + 16 * db + 4 * lg) = o_acc[db][0];
      if (lg == 0) {
        float* stats = part + splits * rows * DV + 2 * row;
        stats[0] = neg_m[0];
        stats[1] = l_acc[0][0];
      }
    }
  } else {
    const int st_row = lane >> 2, st_seg = lane & 3;
    // segment s of a row lives in group {0, 2, 1, 3}[s] after the swap
    const int src_lane = st_row + 16 * (((st_seg & 1) << 1) | (st_seg >> 1));
#pragma unroll
    for (int qb = 0; qb < kQB; ++qb) {
      const float inv = 1.f / l_acc[qb][0];   // of this lane's own row lr
      const int m_row = q_row0 + 16 * qb + st_row;   // the row this lane stores
      T* o_lane = O + (size_t)m_row * dv_row + 8 * st_seg;
#pragma unroll
      for (int db = 0; db < kDB; db += 2) {
        unsigned x[2], y[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const V2 hx = {(T)(o_acc[db][qb][2 * h] * inv), (T)(o_acc[db][qb][2 * h + 1] * inv)};
          const V2 hy = {(T)(o_acc[db + 1][qb][2 * h] * inv), (T)(o_acc[db + 1][qb][2 * h + 1] * inv)};
          x[h] = __builtin_bit_cast(unsigned, hx);
          y[h] = __builtin_bit_cast(unsigned, hy);
#if defined(__HIP_DEVICE_COMPILE__)
          // x of the odd groups <-> y of the even groups
          auto sw = __builtin_amdgcn_permlane16_swap(x[h], y[h], false, false);
          x[h] = sw[0];
          y[h] = sw[1];
#endif
        }
        uint4_t v;
        v[0] = (unsigned)__builtin_amdgcn_ds_bpermute(4 * src_lane, (int)x[0]);
        v[1] = (unsigned)__builtin_amdgcn_ds_bpermute(4 * src_lane, (int)x[1]);
        v[2] = (unsigned)__builtin_amdgcn_ds_bpermute(4 * src_lane, (int)y[0]);
        v[3] = (unsigned)__builtin_amdgcn_ds_bpermute(4 * src_lane, (int)y[1]);
        if (m_row < Lq && (!kEnds || m_row >= 0) && (!kTail || 16 * db + 8 * st_seg < dv_row)) *reinterpret_cast<uint4_t*>(o_lane + 16 * db) = v;
      }
    }
  }
  // the next pass re-fills the ring: nobody may still be reading the last tiles
  if (pass + 1 < num_passes) __syncthreads();
  }  // pass
}

// O = sum over parts of 2^(m_part - m) rows / the same of their sums, m the largest reference; a part without a score
// above -inf (sum 0) has none.  A thread takes 8 elements of a row.  Bound by its launch and the
// latency of two dependent reads: the rows (33 MB at most) come from eight L2s that are not coherent with each other, through
// the memory side.  The rule that asks for it counts 3.5 us and their way there and back.
template <typename T, int D>
__global__ __launch_bounds__(256) void merge_parts_kernel(const float* __restrict__ part, T* __restrict__ O, size_t rows, int d,
                                                          int splits) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  const int per_row = d / 8;
  const size_t row = i / per_row;
  const int col = (int)(i % per_row) * 8;
  if (row >= rows) return;
  const float2_t* stats = reinterpret_cast<const float2_t*>(part + splits * rows * D);
  float m = -INFINITY;
#pragma unroll 8
  for (int s = 0; s < splits; ++s) {
    const float2_t x = stats[s * rows + row];
    if (x[1] != 0.f) m = fmaxf(m, -x[0]);
  }
  float sum = 0.f;
  float4_t acc[2] = {};
#pragma unroll 4
  for (int s = 0; s < splits; ++s) {
    const float2_t x = stats[s * rows + row];
    const float4_t* src = reinterpret_cast<const float4_t*>(part + (s * rows + row) * D + col);
    const float w = x[1] != 0.f ? __builtin_amdgcn_exp2f(-x[0] - m) : 0.f;
    sum = fmaf(w, x[1], sum);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[h][e] = fmaf(w, src[h][e], acc[h][e]);
  }
  typename Vec<T>::v8 out;
  const float inv = 1.f / sum;
#pragma unroll
  for (int e = 0; e < 8; ++e) out[e] = (T)(acc[e / 4][e % 4] * inv);
  *reinterpret_cast<typename Vec<T>::v8*>(O + row * d + col) = out;
}

template <typename T, int D, int DV, bool kKT, bool kVT, bool kCausal, int kWavesT, int kQB, bool kTail, bool kSplit = false>
int launch_w(const AttentionCall& c) {
  auto kern = flash_attention_fwd_kernel<T, D, DV, kKT, kVT, kCausal, kWavesT, kQB, kTail, kSplit>;
  constexpr int kBN = key_tile(D);
  constexpr int lds = ring_stages(kWavesT, D) * (kBN * (kKT ? D : lds_pitch(D)) * 2 + (kVT ? DV * kBN * 2 : kBN * lds_pitch(DV) * 2));
  static_assert(lds <= kMaxLdsBytes, "tiles do not fit in LDS");
  TFK_LDS_OPT_IN(kern, lds);
  constexpr int bm = kWavesT * 16 * kQB;
  const int q_tiles = (c.Lq + bm - 1) / bm;
  const bool paired = kCausal && c.paired;
  const int total_items = paired ? (q_tiles / 2) * c.batch : q_tiles * c.batch * (kSplit ? c.splits : 1);
  // Single causal tiles: a slice's stay on one XCD by themselves where 8 divides the slices, and where it does not if
  // that leaves the XCDs within 4% of each other (bf16, 150 slices of 384 x 384 x 256: 39.4 / 31.4 us).
  const int per_xcd = (c.batch + 7) / 8;
  const bool by_xcd = kCausal && !paired && c.batch % 8 != 0 && 8 * per_xcd * 100 <= c.batch * 104;
  const bool folded = kCausal && two_on_cu(kWavesT, kQB, D, kKT) && !paired && !by_xcd && total_items > kCUs && total_items <= (D == 64 ? kCUs * 9 / 4 : 2 * kCUs);
  // Where causal tiles end, in 64 rows: where the queries end where CUs get several, so that the tile that is not full is the lightest instead of
  // the heaviest: up to a tile's keys less for every slice.  (64 slices of 1337 x 1337 x 64 27.0 / 25.8 us, 66 of 1560 x 128 71 / 61, 114 of 704 x
  // 128 36.0 / 32.6.  Ends at multiples of 16 leave more to the lightest, but then wavefronts of one set meet their masked tiles
  // at different times: 9 of 1364 x 64, which one workgroup's chain bounds, 14.8 / 15.5.)  Rows in front of the first query are none then.
  // With single tiles for no more than the CUs the heaviest is what counts, and it is done sooner if it is the one that is not full: 95 of
  // 320 x 128 16.2 / 14.6, 0.94 of the time over 114 problems of up to 8 tiles a slice, 1.015 at most; longer slices are 2% behind so (6
  // of 10 to 32 tiles, 8 of 3992 x 96 50.8 / 53.3).  The same rows share a wavefront either way, and their results are the same bits.
  const bool from_front = !paired && total_items <= kCUs && q_tiles <= 8;
  const int end = from_front ? q_tiles * (bm / 64) : (c.Lq + 63) / 64;
  const dim3 grid(by_xcd ? 8 * per_xcd * q_tiles : 8 * ((total_items + 7) / 8));
  return launch_kernel(kern, grid, dim3(kWavesT * 64), lds, c.stream,
                       static_cast<const T*>(c.Q), static_cast<const T*>(c.K),
                       static_cast<const T*>(c.V), static_cast<T*>(c.O), c.Lq, c.Lkv, c.scale_log2,
                       q_tiles, total_items, paired ? kPairs : by_xcd ? kByXcd : folded ? kFolded : kSingle, c.d, end, c.part, c.splits, c.chunk);
}

template <typename T, int D, bool kKT, bool kVT, bool kCausal, bool kTail>
int launch_rows(const AttentionCall& c) {
  if (c.rows == 256) return launch_w<T, D, D, kKT, kVT, kCausal, 8, 2, kTail>(c);
  if (c.rows == 128) return launch_w<T, D, D, kKT, kVT, kCausal, 8, 1, kTail>(c);
  return launch_w<T, D, D, kKT, kVT, kCausal, 4, 1, kTail>(c);
}
template <typename T, int D, bool kKT, bool kVT, bool kTail = false>
int launch_causal(const AttentionCall& c) {
  return c.causal ? launch_rows<T, D, kKT, kVT, true, kTail>(c) : launch_rows<T, D, kKT, kVT, false, kTail>(c);
}
template <typename T, int D>
int launch_layout(const AttentionCall& c) {
  if (c.k_transposed) return launch_causal<T, D, true, false>(c);
  if (c.v_transposed) return launch_causal<T, D, false, true>(c);
  return launch_causal<T, D, false, false>(c);
}
template <typename T, int D, bool kTail>
int launch_split(const AttentionCall& c) {
  int rc;
  if constexpr (kTail) rc = launch_w<T, D, D, false, false, false, 4, 1, true, true>(c);
  else if constexpr (D > 128) rc = launch_w<T, D, D, false, false, false, 4, 1, false, true>(c);
  else rc = c.k_transposed ? launch_w<T, D, D, true, false, false, 4, 1, false, true>(c)
                           : launch_w<T, D, D, false, false, false, 4, 1, false, true>(c);
  if (rc != TF_OK) return rc;
  const size_t rows = (size_t)c.batch * c.Lq, threads = rows * (c.d / 8);
  return launch_kernel(merge_parts_kernel<T, D>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, c.stream, c.part,
                       static_cast<T*>(c.O), rows, c.d, c.splits);
}
template <int D>
int launch(const AttentionCall& c) {
  if (c.splits > 1) return c.bf16 ? launch_split<bf16_t, D, false>(c) : launch_split<half_t, D, false>(c);
  return c.bf16 ? launch_layout<bf16_t, D>(c) : launch_layout<half_t, D>(c);
}
// rows of c.d < D elements (K and V as they come)
template <int D>
int launch_tail(const AttentionCall& c) {
  if (c.splits > 1) return c.bf16 ? launch_split<bf16_t, D, true>(c) : launch_split<half_t, D, true>(c);
  return c.bf16 ? launch_causal<bf16_t, D, false, false, true>(c) : launch_causal<half_t, D, false, false, true>(c);
}

}  // namespace
}  // namespace tfk
