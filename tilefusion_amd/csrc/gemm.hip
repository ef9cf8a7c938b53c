// GEMM macro kernel for gfx950: C[M,N] = A[M,K] * B[K,N] with A row-major and B handed over
// as its [N,K] buffer (column-major K x N), fp16 in, fp32 accumulate, fp32 or fp16 out.
//
// Counterpart of the reference's ke_gemm / ke_gemm_level1_pipeline / ke_gemm_level2_pipeline
// (include/kernels/gemm_device.cuh:110-419) and its host launcher (src/kernels/gemm.cu:63-142),
// re-designed for CDNA4:
//   * 64-lane wavefronts, v_mfma_f32_16x16x32_f16 base tiles, accumulators in the unified
//     512-entry register file (one wavefront per SIMD, 128x128 per wavefront at the big tile);
//   * both operands are K-contiguous, so an MFMA operand fragment is one 16-byte LDS read;
//   * tiles go global -> LDS without passing through VGPRs (global_load_lds_dwordx4) into an
//     XOR-swizzled LDS ring: a wavefront instruction always writes 1 KiB of consecutive LDS,
//     so the swizzle is applied on the global (source) side;
//   * the main kernel (gemm_ring64_kernel) uses 64-deep k-tiles so that every request fetches
//     whole 128-byte lines, keeps the ring in units of one operand, and issues its MFMAs from
//     assembly with a hand-placed instruction order (a lone wavefront issues one instruction
//     per 4 cycles: at most three others fit behind a 16-cycle MFMA); it comes with tiles from
//     128 x 128 to 256 x 256, for any M and N from one tile on and any K % 8 == 0 from 64 on;
//   * problems of few rows, columns or tiles run gemm_split_k_kernel, whose wavefronts share one small
//     tile and split K; a measured cost model picks the kernel and the tile;
//   * workgroup -> tile map keeps the workgroups of one XCD (one L2) on a compact block of
//     output tiles.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.hpp"

namespace tfk {
namespace {

template <int BM_, int BN_, int BK_, int WAVES_M_, int WAVES_N_>
struct GemmShape {
  static constexpr int BM = BM_, BN = BN_, BK = BK_;
  static constexpr int WAVES_M = WAVES_M_, WAVES_N = WAVES_N_;
  static constexpr int kWaves = WAVES_M * WAVES_N;
  static constexpr int kThreads = kWaves * kWaveSize;
  static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;  // tile of one wavefront
  static constexpr int TM = WM / 32, TN = WN / 32;            // 32x32 MFMA tiles per wavefront
  static constexpr int kKSteps = BK / 16;
  static constexpr int kChunks = BK / 8;              // 16-byte chunks per tile row
  static constexpr int kRowsPer256B = 16 / kChunks;   // rows that share one pass over all banks
  static constexpr int kABytes = BM * BK * 2;
  static constexpr int kBBytes = BN * BK * 2;
  static_assert(WM % 32 == 0 && WN % 32 == 0 && BK % 16 == 0, "wavefront tile must be MFMA-sized");

  // Physical 16-byte chunk of logical chunk `c` in tile row `row`.  Sixteen consecutive rows
  // reading the same logical chunk land in sixteen different 16-byte bank groups.
  __host__ __device__ static constexpr int swizzle(int row, int c) {
    return c ^ ((row / kRowsPer256B) % kChunks);
  }
};

// Workgroup ids are dealt round-robin to the 8 XCDs, so ids that are equal mod 8 share an L2.  This
// gives each XCD a run of consecutive positions out of 0 .. nblocks-1.
TFK_DEVICE int xcd_major(int bid, int nblocks) {
  const int xcd = bid & 7;
  return xcd * (nblocks >> 3) + min(xcd, nblocks & 7) + (bid >> 3);
}
// XCD-aware tile order: a grouped (4 tile-rows at a time) walk of the output, so that the workgroups
// of an XCD re-use A and B panels.
TFK_DEVICE void tile_of_block(int bid, int nblocks, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int pid = xcd_major(bid, nblocks);
  constexpr int kGroup = 4;
  const int group_size = kGroup * tiles_n;
  const int gid = pid / group_size;
  const int first_m = gid * kGroup;
  const int rows = min(tiles_m - first_m, kGroup);
  const int in_group = pid - gid * group_size;
  tm = first_m + in_group % rows;
  tn = in_group / rows;
}

template <typename OutT>
TFK_DEVICE void store_out(OutT* p, float v) {
  if constexpr (sizeof(OutT) == 2) {
    *p = (OutT)v;
  } else {
    *p = v;
  }
}

// MFMAs by operand type (half_t or bf16_t) for the kernels that issue them through builtins
template <typename InT> using in8_t = InT __attribute__((ext_vector_type(8)));
template <typename InT>
TFK_DEVICE float4_t mfma16_t(in8_t<InT> a, in8_t<InT> b, float4_t c) {
  if constexpr (std::is_same_v<InT, bf16_t>) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  else return mfma_16x16x32(a, b, c);
}
template <typename InT>
TFK_DEVICE float16_t mfma32_t(in8_t<InT> a, in8_t<InT> b, float16_t c) {
  if constexpr (std::is_same_v<InT, bf16_t>) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  else return mfma_32x32x16(a, b, c);
}

// ------------------------------------------------------------------------------------------
// 256 x 256 x 64 path: same 2 x 2 wavefronts of 128 x 128, but k-tiles of 64 so that every
// global->LDS instruction fetches whole 128-byte lines (8 rows x 128 bytes).  The vector L1
// moves full lines, so the 64-byte row segments of a 32-deep tile spend half of the L2->L1
// bandwidth on bytes that are dropped and requested again one k-tile later.
//
// A 64-deep tile is 64 KiB and only 160 KiB of LDS exist, so the ring is kept in UNITS of one
// operand of one tile (32 KiB, five of them): unit u lives in ring slot u % 5, A of tile t is
// unit 2t and B of tile t unit 2t+1.  Iteration t:
//   k-step 0: multiplies fragments (t, 0), reads fragments (t, 1), requests A of tile t+2 into
//             the slot B of tile t-1 left;
//   barrier:  tile t is read out (both its units are free) and tile t+1 has landed
//             (vmcnt leaves only the 8 requests of k-step 0 outstanding);
//   k-step 1: multiplies (t, 1), reads fragments (t+1, 0), requests B of tile t+2 into the
//             slot A of tile t left.
// Every request has at least 8 MFMA slots (1024 MFMA cycles) to land.
// ------------------------------------------------------------------------------------------
//
// The same kernel serves smaller tiles (2 x 2 wavefronts of half a tile each way), for grids that 256 x 256
// tiles would leave CUs idle on: 3333 x 2288 x 1944 takes 45.5 us with 126 tiles of 256 x 256, 36.7 with
// 216 of 192 x 192 and 36.4 with 252 of 256 x 128; 2999 x 1544 x 1032 27.6 and, with 192 x 128, 18.7 (the bounds-checked kernel that ran
// these shapes before: 37.8; whole lines, below, 17.3, and with 160 x 128 16.6).  Units then have the size of the larger operand.  128 x 128 tiles have k-steps
// four times shorter; where a workgroup has its CU to itself their requests run kAhead = 4 tiles
// ahead (a ring of 2 * kAhead + 1 = 9 units).
//
// K that is no multiple of 64 (kLines): rows start anywhere in a 128-byte line, and k-tiles that start where a row starts
// would fetch every line twice, for two tiles (8 rows x 128 bytes are 16 lines instead of 8: 0.13 to 0.27 us more a k-tile).
// So what is fetched are SEGMENTS of whole lines: segment u of a row is its u-th line, and in it k-tile t of the row takes
// the end of segment t and the front of segment t + 1, by an amount that only depends on the row. Rows 8 apart start at
// the same place in a line, so a lane's fragments all are shifted alike, and what a lane pays is the choice between
// the two segments (one v_and and one v_add3 an address). The ring is kept in whole tiles then, kLines of them: two are
// read, the others in flight. 2999 x 1544 x 1032 18.7 -> 17.3 us (K = 1024: 14.7).
template <int BM_, int BN_, int AHEAD_, int LINES_ = 0>
struct Ring64Shape {
  static constexpr int BM = BM_, BN = BN_, BK = 64;
  static constexpr int WAVES_M = 2, WAVES_N = 2;
  static constexpr int kWaves = WAVES_M * WAVES_N, kThreads = kWaves * kWaveSize;
  static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
  static constexpr int TM = WM / 16, TN = WN / 16;          // 16x16 MFMA tiles per wavefront
  static constexpr int kRowBytes = BK * 2;                  // 128
  static constexpr int kUnitBytes = (BM > BN ? BM : BN) * kRowBytes;   // one operand of one tile
  static constexpr int kAhead = AHEAD_;                     // tiles between a request and its use
  static constexpr int kUnits = 2 * kAhead + 1;
  static constexpr int kLoadsA = BM / 8 / kWaves, kLoadsB = BN / 8 / kWaves;   // 1 KiB requests per wavefront and unit
  static constexpr int kLoadsMax = kLoadsA > kLoadsB ? kLoadsA : kLoadsB;
  static constexpr int kLoads = kLoadsA + kLoadsB;
  static constexpr int kLines = LINES_;                     // segments in the ring, 0: k-tiles start where rows start
  static constexpr int kTileBytes = (BM + BN) * kRowBytes;
  static constexpr int kLdsBytes = kLines ? kLines * kTileBytes : kUnits * kUnitBytes;
  // slot schedule of a k-step (TM slots of TN MFMAs): the TM + TN fragment reads of the next
  // k-step are dealt to the first kReadSlots slots; the scalar bookkeeping runs in the gaps
  // without a read from slot kPrepSlot on
  static constexpr int kReads = TM + TN;
  static constexpr int kReadSlots = TM == 8 ? 6 : TM - 1;
  static constexpr int kPrepSlot = TM == 8 ? 6 : 0;
  static constexpr int reads_first(int i) { return i < kReadSlots ? (i * kReads) / kReadSlots : kReads; }
  static constexpr int reads_in(int i) { return reads_first(i + 1) - reads_first(i); }
  // read number d of a slot follows MFMA (d * TN) / n of that slot (gap j = that + 1)
  static constexpr bool gap_has_read(int i, int j) {
    const int n = reads_in(i);
    for (int d = 0; d < n; ++d)
      if (j == (d * TN) / n + 1) return true;
    return false;
  }
  // which bookkeeping piece runs in gap j of slot i (-1: none); a table, so that the unrolled
  // slots index it with constants
  struct PrepTable {
    int piece[TM * TN];
  };
  static constexpr PrepTable make_prep_table() {
    PrepTable t{};
    int rank = 0;
    for (int i = 0; i < TM; ++i)
      for (int j = 0; j < TN; ++j) t.piece[i * TN + j] = (i < kPrepSlot || gap_has_read(i, j)) ? -1 : rank++;
    return t;
  }
  static constexpr PrepTable kPrep = make_prep_table();
  static constexpr int free_gaps() { return kPrep.piece[TM * TN - 1] + 1; }
  static constexpr bool reads_fit() {
    for (int i = 0; i < TM; ++i) {
      if (reads_in(i) > TN - 1) return false;
      for (int d = 1; d < reads_in(i); ++d)   // two reads never share a gap
        if ((d * TN) / reads_in(i) == ((d - 1) * TN) / reads_in(i)) return false;
    }
    return true;
  }
  static_assert(BM % 32 == 0 && BN % 64 == 0, "whole MFMA tile pairs; an even request count of B (see the swizzle of g_off)");
  static constexpr bool kOwnOffsetsB = kLines > 0 || kLoadsA % 2 != 0;   // requests of B do not lie as those of A
  static_assert(reads_fit() && free_gaps() >= 7,
                "slot schedule: every read and bookkeeping piece needs its own gap");
  // requests in flight behind the barrier in the middle of a tile: A of tile t+kAhead, all of the
  // tiles t+2 .. t+kAhead-1
  // (kLines: the segments t+3 .. t+kLines-1)
  static constexpr int kInFlight = kLines ? (kLines - 3) * kLoads : kLoadsA + (kAhead - 2) * kLoads;
  static_assert((kAhead - 1) * kLoads < 64 && (kLines - 2) * kLoads < 64, "vmcnt is a 6-bit counter");
  static_assert(kLines == 0 || (kLines >= 3 && free_gaps() >= 8), "two segments are read, one is in flight; a gap for every piece");
  // 128-byte rows: two rows per pass over the banks; chunk ^ (row / 2) % 8 keeps every
  // ds_read_b128 lane pass on 16 different bank groups
  __host__ __device__ static constexpr int swizzle(int row, int c) { return c ^ ((row / 2) % 8); }
};

__device__ const uint4_t kZeros[1] = {};   // what the chunks in front of a row are fetched from

// M >= BM, N >= BN, and K >= BK (kLines: K > 64 * kLines): requests past the last k-tile ask for that tile again, which must not
// be the one completed with zeros.
// InT is half_t or bf16_t: the two differ in the MFMA mnemonic and in the conversion of the
// result, everything else moves 16-bit elements without looking at them.
template <typename S, typename InT, typename OutT>
__global__ __launch_bounds__(S::kThreads) void gemm_ring64_kernel(
    const InT* __restrict__ A, const InT* __restrict__ B, OutT* __restrict__ C, int M,
    int N, int K, int tiles_m, int tiles_n) {
  constexpr bool kBf16 = std::is_same_v<InT, bf16_t>;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int tile_m, tile_n;
  tile_of_block(blockIdx.x, gridDim.x, tiles_m, tiles_n, tile_m, tile_n);
  // The last tile of a row or column of tiles ends where C ends: it overlaps its neighbour, and the rows
  // and columns both compute are written twice with the same bits.  No request, product or store has
  // to know about edges.
  const int m0 = min(tile_m * S::BM, M - S::BM), n0 = min(tile_n * S::BN, N - S::BN);
  const int wm = wave / S::WAVES_N, wn = wave % S::WAVES_N;

  // global -> LDS plan: request n of a wavefront covers rows (wave * kLoads + n) * 8 .. +7 of a
  // unit (consecutive 1 KiB blocks of LDS, so four requests share one M0 base and differ in the
  // instruction's immediate offset); lane l fills physical chunk l % 8 of row l / 8 and fetches the logical chunk the
  // swizzle maps there.  A and B share the per-lane offsets (same row stride K); the address
  // is a scalar base (tile origin + k offset) plus this 32-bit per-lane offset, so a request
  // needs no vector arithmetic.
  const int ld_row = lane / 8, ld_c = lane % 8;
  // K is completed to whole k-tiles at its FRONT: k-tile t starts at element 64 * t - k_pad of a row, and
  // the chunks of tile 0 that lie in front of the row are fetched from a block of zeros.  Only the
  // prologue knows about it.
  const int num_k_tiles = (K + S::BK - 1) / S::BK;
  const int k_pad = num_k_tiles * S::BK - K;
  // kLines: chunk c of row r, counted from the completed front, is chunk (c + shift(r)) % 8 of segment (c + shift(r)) / 8,
  // shift(r) = 1 .. 8. In LDS it lies where it would without a shift, so that reads see the same banks.
  constexpr bool kShift = S::kLines > 0;
  constexpr int kLead = kShift ? 256 : 0;   // (keeps lane offsets positive: up to 15 chunks in front of a row)
  const int pad_chunks = k_pad / 8;
  auto shift_of = [&](const InT* X, int row) __attribute__((always_inline)) {
    const unsigned in_line = (unsigned)(reinterpret_cast<uintptr_t>(X) >> 4) + (unsigned)row * (unsigned)(K / 8);
    return (int)((in_line - (unsigned)pad_chunks - 1u) & 7u) + 1;
  };
  const int a_shift = shift_of(A, m0 + ld_row), b_shift = shift_of(B, n0 + ld_row);   // of the rows that this lane fetches
  const char* a_tile = reinterpret_cast<const char*>(A + (size_t)(m0 + wave * 8 * S::kLoadsA) * K) - (kShift ? kLead : 2 * k_pad);
  const char* b_tile = reinterpret_cast<const char*>(B + (size_t)(n0 + wave * 8 * S::kLoadsB) * K) - (kShift ? kLead : 2 * k_pad);
  unsigned g_off[S::kLoadsMax];
  unsigned g_off_b[S::kOwnOffsetsB ? S::kLoadsB : 1];
  // (an odd number of requests: every other wavefront's rows begin in the middle of the swizzle's sixteen)
  const int a_odd = S::kLoadsA % 2 ? wave & 1 : 0;
  // the chunk of a segment that this lane fetches with request n
  auto segment_chunk = [&](int n, int shift) __attribute__((always_inline)) { return (S::swizzle(ld_row + 8 * n, ld_c) + shift) & 7; };
  auto segment_off = [&](int n, int odd, int shift) __attribute__((always_inline)) {
    return (unsigned)(ld_row + 8 * n) * (unsigned)K * 2u + (unsigned)(kLead + 16 * (segment_chunk(n + odd, shift) - shift - pad_chunks)) -
           1024u * (n % 4);
  };
  auto tile_off = [&](int n, int odd) __attribute__((always_inline)) {
    return (unsigned)(ld_row + 8 * n) * (unsigned)K * 2u + (unsigned)S::swizzle(ld_row + 8 * (n + odd), ld_c) * 16u -
           1024u * (n % 4);   // the instruction's immediate offset (added to both addresses) gives it back
  };
#pragma unroll
  for (int n = 0; n < S::kLoadsMax; ++n)
    g_off[n] = kShift ? segment_off(n, a_odd, a_shift)
                      : tile_off(n, a_odd);
  if constexpr (S::kOwnOffsetsB) {
#pragma unroll
    for (int n = 0; n < S::kLoadsB; ++n) g_off_b[n] = kShift ? segment_off(n, 0, b_shift) : tile_off(n, 0);
  }
  // LDS -> fragment plan: fragment i of k-step ks: row 16*i + l%16 of the wavefront's rows,
  // logical chunk 4*ks + l/16
  const int fr = lane & 15, fg = lane >> 4;
  unsigned a_rd[2], b_rd[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    a_rd[ks] = (wm * S::WM + fr) * S::kRowBytes + S::swizzle(fr, 4 * ks + fg) * 16;
    b_rd[ks] = (wn * S::WN + fr) * S::kRowBytes + S::swizzle(fr, 4 * ks + fg) * 16;
  }

  float4_t acc[S::TM][S::TN];
#pragma unroll
  for (int i = 0; i < S::TM; ++i)
#pragma unroll
    for (int j = 0; j < S::TN; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

  const unsigned smem_addr = lds_address(smem);
  // Slot i of a k-step multiplies A fragment i with all B fragments; both operands have two
  // register sets (this k-step's and the next one's).
  half8_t afx[2][S::TM], bf[2][S::TN];
  // The requests are issued from inline assembly: the compiler then keeps exact counts for the
  // fragment reads (a direct-to-LDS load it knows about makes every LDS wait a full drain),
  // and the vector-memory waits are placed by hand below.
  // src: tile origin + k offset (scalar); lds_unit: LDS byte address of this wavefront's first
  // 1 KiB block in the destination unit.
  // M0 - the LDS destination of requests n .. n+3 (n % 4 == 0), which differ in the immediate
  // offset - is an INPUT of every request statement: the compiler writes it (once per group of
  // four: the statements do not change it) and cannot use the register for anything else between
  // that write and a request.  The s_nop is the wait state an M0 write needs in front of an
  // LDS-direct load; next to a request at the head of a slot it costs no issue time.
  auto request_at = [&](unsigned off, const char* src, unsigned lds_unit, int n) __attribute__((always_inline)) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 offset:%2"
                 :
                 : "v"(off), "s"(src), "n"(1024 * (n % 4)), "{m0}"(lds_unit + (n - n % 4) * 1024)
                 : "memory");
  };
  auto request = [&](const char* src, unsigned lds_unit, int n, auto of_b) __attribute__((always_inline)) {
    if constexpr (S::kOwnOffsetsB && decltype(of_b)::value) request_at(g_off_b[n], src, lds_unit, n);
    else request_at(g_off[n], src, lds_unit, n);
  };
  auto k_src = [&](const char* tile, int t) __attribute__((always_inline)) {
    return tile + (size_t)min(t, num_k_tiles - 1) * S::BK * 2;   // clamped past the end
  };
  const unsigned lds_wave_a = smem_addr + wave * S::kLoadsA * 1024, lds_wave_b = smem_addr + wave * S::kLoadsB * 1024;
  // Slot with the MFMAs issued from inline assembly, accumulators pinned to AGPRs, and the
  // slot's fragment reads placed by hand between them.  (With compiler-issued MFMAs the
  // register allocator, at exactly 256 live accumulators, shuffles accumulators through VGPRs
  // whenever the schedule changes slightly.)
  auto lds_read_b128 = [](unsigned addr) __attribute__((always_inline)) {
    return *(__attribute__((address_space(3))) const half8_t*)(size_t)addr;
  };
  // rd_a / rd_b: this lane's LDS byte address of fragment 0 of the next k-step's A / B operand
  // (unit base + row + swizzled chunk); fragment f is f * 2 KiB further, in the offset field.
  auto slot_pinned = [&](int buf, int i, unsigned rd_a, unsigned rd_b, auto&& between) __attribute__((always_inline)) {
    // The TN + TM fragment reads of the next k-step, B fragments first, are dealt to the first
    // kReadSlots slots; the last slot(s) read nothing, so the drain in front of the barrier
    // (and the one at the head of the next k-step) finds the reads already returned.
    const int first = S::reads_first(i);
    const int n_reads = S::reads_in(i);
    int done = 0;
#pragma unroll
    for (int j = 0; j < S::TN; ++j) {
      if constexpr (kBf16)
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(bf[buf][j]), "v"(afx[buf][i]));
      else
        asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(bf[buf][j]), "v"(afx[buf][i]));
      // after MFMA j: issue the next read if j is its position (reads spread evenly over the slot)
      if (done < n_reads && j == (done * S::TN) / n_reads + 1) {
        const int q = first + done;
        __builtin_amdgcn_sched_barrier(0);
        if (q < S::TN) bf[buf ^ 1][q] = lds_read_b128(rd_b + q * 16 * S::kRowBytes);
        else afx[buf ^ 1][q - S::TN] = lds_read_b128(rd_a + (q - S::TN) * 16 * S::kRowBytes);
        __builtin_amdgcn_sched_barrier(0);
        ++done;
      } else {
        between(j);   // a piece of scalar bookkeeping, if this gap has one
      }
    }
  };
  // Workgroup barrier in the middle of tile t: tile t+1 must have landed, the requests of
  // tiles t+2 .. t+kAhead-1 and of this tile's k-step 0 stay in flight.  The LDS wait and the
  // barrier are builtins so that the compiler knows every earlier fragment read has returned.
  constexpr int kInFlight = S::kInFlight;
  auto ring_barrier = [&]() __attribute__((always_inline)) {
    // one s_waitcnt: vmcnt(kInFlight) lgkmcnt(0); a builtin, so the compiler knows the LDS part
    __builtin_amdgcn_s_waitcnt((kInFlight & 15) | 0x70 | ((kInFlight >> 4) << 14));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // the requests of a k-step sit at the heads of its slots, evenly spread
  auto request_slot = [&](int i, const char* src, unsigned lds_unit, auto loads_c, auto of_b) __attribute__((always_inline)) {
    constexpr int kLoads = decltype(loads_c)::value;
#pragma unroll
    for (int n = 0; n < kLoads; ++n)
      if ((n * S::TM) / kLoads == i) request(src, lds_unit, n, of_b);
  };
  constexpr std::integral_constant<int, S::kLoadsA> kOfA{};
  constexpr std::integral_constant<int, S::kLoadsB> kOfB{};

  // The compiler does not know that the accumulators are written by MFMAs (they are issued
  // from assembly), so nothing would keep it from reading the youngest results right behind
  // the loop without the wait states the matrix pipe needs.  The delay therefore sits inside
  // the last iteration, in front of anything the register allocator may put on the exit
  // edge.  The iteration count is laundered through an empty asm so that the test is not
  // recognised as the exit condition and sunk out of the loop.
  auto settle_behind_last = [&](int t) __attribute__((always_inline)) {
    int t_seen = t;
    asm volatile("" : "+s"(t_seen));
    if (t_seen + 1 == num_k_tiles) asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
  };
#define TFK_PIN_S(x) asm volatile("" : "+s"(x))
#define TFK_PIN_V(x) asm volatile("" : "+v"(x))
  if constexpr (kShift) {
    // prologue: segments 0 .. kLines-1; the chunks in front of a row, in segments 0 and 1, are zeros
#pragma unroll
    for (int u = 0; u < S::kLines; ++u)
#pragma unroll
      for (int q = 0; q < S::kLoads; ++q) {
        const bool of_a = q < S::kLoadsA;
        const int n = of_a ? q : q - S::kLoadsA;
        const int shift = of_a ? a_shift : b_shift;
        const unsigned off = of_a ? g_off[n] : g_off_b[n];
        const char* tile = (of_a ? a_tile : b_tile) + u * (S::BK * 2);
        const unsigned unit = (of_a ? lds_wave_a : lds_wave_b + S::BM * S::kRowBytes) + u * S::kTileBytes;
        if (u < 2) {
          const bool in_front = 8 * u + segment_chunk(of_a ? n + a_odd : n, shift) - shift < pad_chunks;
          lds_dma_16B(in_front ? reinterpret_cast<const char*>(kZeros) : tile + (off + 1024u * (n % 4)), unit + n * 1024);
        } else {
          request_at(off, tile, unit, n);
        }
      }
    // all ones where this lane's chunk of a k-step lies in the second of the two segments
    int a_next[2], b_next[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      a_next[ks] = 4 * ks + fg + shift_of(A, m0 + fr) >= 8 ? -1 : 0;
      b_next[ks] = 4 * ks + fg + shift_of(B, n0 + fr) >= 8 ? -1 : 0;
    }
    constexpr unsigned kRingBytes = S::kLines * S::kTileBytes;
    auto ring = [](unsigned o) __attribute__((always_inline)) { return o >= kRingBytes ? o - kRingBytes : o; };
    const unsigned rdbase_a0 = smem_addr + a_rd[0], rdbase_a1 = smem_addr + a_rd[1];
    const unsigned rdbase_b0 = smem_addr + S::BM * S::kRowBytes + b_rd[0], rdbase_b1 = smem_addr + S::BM * S::kRowBytes + b_rd[1];
    const unsigned lds_b = lds_wave_b + S::BM * S::kRowBytes;
    wait_vmem<(S::kLines - 2) * S::kLoads>();   // segments 0 and 1 have landed
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    unsigned rd_a0 = rdbase_a0 + (a_next[0] & S::kTileBytes), rd_b0 = rdbase_b0 + (b_next[0] & S::kTileBytes);
#pragma unroll
    for (int f = 0; f < S::TN; ++f) bf[0][f] = lds_read_b128(rd_b0 + f * 16 * S::kRowBytes);
#pragma unroll
    for (int i = 0; i < S::TM; ++i) afx[0][i] = lds_read_b128(rd_a0 + i * 16 * S::kRowBytes);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
    unsigned s0 = 0, s1 = S::kTileBytes, s2 = 0;   // segments t, t+1 and t+2 in the ring
    unsigned step = S::kTileBytes;                 // from a segment to the next one's
    unsigned rd_a1 = rdbase_a1 + (a_next[1] & S::kTileBytes), rd_b1 = rdbase_b1 + (b_next[1] & S::kTileBytes);
    unsigned req_a = 0, req_b = 0;
    const char *src_a = a_tile, *src_b = b_tile;
    int kt = 0;
    // during k-step 0: where the fragments of (t+1, 0) are, and segment t+kLines, which takes the place of segment t in k-step 1
    auto prep0 = [&](int piece, int t) __attribute__((always_inline)) {
      __builtin_amdgcn_sched_barrier(0);
      switch (piece) {
        case 0: s1 = ring(s0 + S::kTileBytes); TFK_PIN_S(s1); break;
        case 1: s2 = ring(s1 + S::kTileBytes); TFK_PIN_S(s2); break;
        case 2: step = s2 - s1; TFK_PIN_S(step); rd_a0 = rdbase_a0 + s1 + (a_next[0] & step); TFK_PIN_V(rd_a0); break;
        case 3: rd_b0 = rdbase_b0 + s1 + (b_next[0] & step); TFK_PIN_V(rd_b0); break;
        case 4: req_a = lds_wave_a + s0; TFK_PIN_S(req_a); req_b = lds_b + s0; TFK_PIN_S(req_b); break;
        case 5: kt = t; TFK_PIN_S(kt); kt = min(kt + S::kLines, num_k_tiles); TFK_PIN_S(kt); break;
        case 6: src_a = a_tile + (size_t)(unsigned)(kt * (S::BK * 2)); TFK_PIN_S(src_a); break;
        case 7: src_b = b_tile + (size_t)(unsigned)(kt * (S::BK * 2)); TFK_PIN_S(src_b); break;
        default: break;
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto prep1 = [&](int piece) __attribute__((always_inline)) {
      __builtin_amdgcn_sched_barrier(0);
      switch (piece) {
        case 0: rd_a1 = rdbase_a1 + s1 + (a_next[1] & step); TFK_PIN_V(rd_a1); break;
        case 1: rd_b1 = rdbase_b1 + s1 + (b_next[1] & step); TFK_PIN_V(rd_b1); break;
        case 2: s0 = s1; TFK_PIN_S(s0); break;
        default: break;
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    for (int t = 0; t < num_k_tiles; ++t) {
      // The last segment ends behind the row: what lies there is never read, and not fetched either (the row's last chunk is,
      // again). Requests from here on ask for no other segment.
      if (t + S::kLines == num_k_tiles) {
#pragma unroll
        for (int n = 0; n < S::kLoadsA; ++n) g_off[n] -= 16u * (unsigned)max(0, segment_chunk(n + a_odd, a_shift) - (a_shift - 1));
#pragma unroll
        for (int n = 0; n < S::kLoadsB; ++n) g_off_b[n] -= 16u * (unsigned)max(0, segment_chunk(n, b_shift) - (b_shift - 1));
      }
#pragma unroll
      for (int i = 0; i < S::TM; ++i) {
        __builtin_amdgcn_sched_barrier(0);
        slot_pinned(0, i, rd_a1, rd_b1, [&](int j) __attribute__((always_inline)) { prep0(S::kPrep.piece[i * S::TN + j], t); });
      }
      __builtin_amdgcn_sched_barrier(0);
      ring_barrier();   // segment t is read out, segment t+2 has landed
#pragma unroll
      for (int i = 0; i < S::TM; ++i) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < S::kLoads; ++q)
          if ((q * S::TM) / S::kLoads == i) {
            if (q < S::kLoadsA) request_at(g_off[q], src_a, req_a, q);
            else request_at(g_off_b[q - S::kLoadsA], src_b, req_b, q - S::kLoadsA);
          }
        slot_pinned(1, i, rd_a0, rd_b0, [&](int j) __attribute__((always_inline)) { prep1(S::kPrep.piece[i * S::TN + j]); });
      }
      settle_behind_last(t);
    }
  } else {
    // prologue: tiles 0 .. kAhead-1 into the first 2 * kAhead units; fragments (0, 0) once
    // tile 0 is there
#pragma unroll
    for (int u = 0; u < 2 * S::kAhead; ++u)
#pragma unroll
      for (int n = 0; n < (u % 2 ? S::kLoadsB : S::kLoadsA); ++n) {
        const char* tile = u % 2 ? b_tile : a_tile;
        const unsigned unit = (u % 2 ? lds_wave_b : lds_wave_a) + u * S::kUnitBytes;
        if (u < 2 && k_pad != 0) {
          const bool in_front = S::swizzle(ld_row + 8 * (u % 2 ? n : n + a_odd), ld_c) * 8 < k_pad;
          const char* src = tile + ((S::kOwnOffsetsB && u % 2 ? g_off_b[n] : g_off[n]) + 1024u * (n % 4));
          lds_dma_16B(in_front ? reinterpret_cast<const char*>(kZeros) : src, unit + n * 1024);
        } else {
          if (u % 2) request(k_src(tile, u / 2), unit, n, std::true_type{});
          else request(k_src(tile, u / 2), unit, n, std::false_type{});
        }
      }
    wait_vmem<(S::kAhead - 1) * (S::kLoadsA + S::kLoadsB)>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int f = 0; f < S::TN; ++f)
      bf[0][f] = *reinterpret_cast<const half8_t*>(smem + S::kUnitBytes + b_rd[0] + f * 16 * S::kRowBytes);
#pragma unroll
    for (int i = 0; i < S::TM; ++i)
      afx[0][i] = *reinterpret_cast<const half8_t*>(smem + a_rd[0] + i * 16 * S::kRowBytes);
    // drained here, visibly to the compiler, so that the waits it places at the head of the loop
    // only have to cover the loop's own reads
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);

    // Ring bookkeeping, in bytes: oa = LDS offset of the unit holding A of tile t; B of tile t is
    // one unit further, A of t+1 two, ... (mod kUnits units).  A wavefront alone on its SIMD issues one
    // instruction every 4 cycles, so a 16-cycle MFMA hides at most three other instructions:
    // everything an iteration needs (fragment read bases, request destinations and sources) is
    // therefore computed during the previous k-step in pieces of at most three instructions,
    // each pinned into its own gap between two MFMAs of the slots that carry no fragment reads.
    constexpr unsigned kRingBytes = S::kUnits * S::kUnitBytes;
    auto ring = [](unsigned o) __attribute__((always_inline)) { return o >= kRingBytes ? o - kRingBytes : o; };
    const unsigned rdbase_a0 = smem_addr + a_rd[0], rdbase_a1 = smem_addr + a_rd[1];
    const unsigned rdbase_b0 = smem_addr + b_rd[0], rdbase_b1 = smem_addr + b_rd[1];
    const int last_tile = num_k_tiles - 1;
    unsigned oa = 0;                                             // A of tile t
    unsigned oa1 = 2 * S::kUnitBytes, ob1 = 3 * S::kUnitBytes;   // A, B of tile t+1
    unsigned rd_a1 = rdbase_a1, rd_b1 = rdbase_b1 + S::kUnitBytes;   // reads of (t, k-step 1)
    unsigned req_a = lds_wave_a + 2 * S::kAhead * S::kUnitBytes;       // A of t+kAhead
    const char* src_a = k_src(a_tile, S::kAhead);
    unsigned rd_a0 = 0, rd_b0 = 0, req_b = 0;                        // set during k-step 0
    const char* src_b = b_tile;
    int kt = 0;
    // pieces run in the read-free gaps from slot kPrepSlot on of k-step 0 / k-step 1
    auto prep0 = [&](int step, int t) __attribute__((always_inline)) {
      __builtin_amdgcn_sched_barrier(0);
      switch (step) {
        case 0: TFK_PIN_S(oa); oa1 = ring(oa + 2 * S::kUnitBytes); TFK_PIN_S(oa1); break;
        case 1: ob1 = ring(oa1 + S::kUnitBytes); TFK_PIN_S(ob1); break;
        case 2: rd_a0 = rdbase_a0 + oa1; TFK_PIN_V(rd_a0); break;
        case 3: rd_b0 = rdbase_b0 + ob1; TFK_PIN_V(rd_b0); break;
        case 4: req_b = lds_wave_b + oa; TFK_PIN_S(req_b); break;
        case 5: kt = t; TFK_PIN_S(kt); kt = min(kt + S::kAhead, last_tile); TFK_PIN_S(kt); break;
        case 6: src_b = b_tile + (size_t)(unsigned)(kt * (S::BK * 2)); TFK_PIN_S(src_b); break;
        default: break;
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto prep1 = [&](int step, int t) __attribute__((always_inline)) {
      __builtin_amdgcn_sched_barrier(0);
      switch (step) {
        case 0: oa = oa1; TFK_PIN_S(oa); rd_a1 = rdbase_a1 + oa; TFK_PIN_V(rd_a1); break;
        case 1: rd_b1 = rdbase_b1 + ob1; TFK_PIN_V(rd_b1); break;
        case 2: req_a = ring(oa + 2 * S::kAhead * S::kUnitBytes); TFK_PIN_S(req_a); break;
        case 3: req_a += lds_wave_a; TFK_PIN_S(req_a); break;
        case 4: kt = t; TFK_PIN_S(kt); kt = min(kt + S::kAhead + 1, last_tile); TFK_PIN_S(kt); break;
        case 5: src_a = a_tile + (size_t)(unsigned)(kt * (S::BK * 2)); TFK_PIN_S(src_a); break;
        default: break;
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    for (int t = 0; t < num_k_tiles; ++t) {
#pragma unroll
      for (int i = 0; i < S::TM; ++i) {
        __builtin_amdgcn_sched_barrier(0);
        request_slot(i, src_a, req_a, kOfA, std::false_type{});
        slot_pinned(0, i, rd_a1, rd_b1, [&](int j) __attribute__((always_inline)) {
          prep0(S::kPrep.piece[i * S::TN + j], t);
        });
      }
      __builtin_amdgcn_sched_barrier(0);
      ring_barrier();
#pragma unroll
      for (int i = 0; i < S::TM; ++i) {
        __builtin_amdgcn_sched_barrier(0);
        request_slot(i, src_b, req_b, kOfB, std::true_type{});
        slot_pinned(1, i, rd_a0, rd_b0, [&](int j) __attribute__((always_inline)) {
          prep1(S::kPrep.piece[i * S::TN + j], t);
        });
      }
      settle_behind_last(t);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  wait_vmem_all();  // the clamped tail requests must not outlive the workgroup's LDS
  // --- epilogue -----------------------------------------------------------------------------
  // acc[i][j][r] = C[.. + 16*i + l%16][.. + 16*j + 4*(l/16) + r].  For fp16 output the data is
  // re-dealt so that a store instruction writes 16 rows x 64 contiguous bytes with FOUR
  // ADJACENT lanes per row: the address unit merges adjacent lanes into one 64-byte access,
  // whereas lanes 16 apart cost one access each (measured: 64 accesses per instruction and
  // 9 k cycles of epilogue per wavefront).  Step 1: the 16-lane groups g and g^1 trade halves
  // of a pair of tiles (v_permlane16_swap), after which group 0/2 holds columns 0-7 / 8-15 of
  // tile j and group 1/3 the same of tile j+1, 16 bytes per lane.  Step 2: ds_bpermute moves
  // the 16 bytes of (row r, segment s) to lane 4*r + s.
  // (An odd N leaves the rows of C, and then the vectors of a store, without alignment.)
  typedef uint4_t out16B_t __attribute__((aligned(2)));
  typedef float4_t out4f_t __attribute__((aligned(4)));
  const int c_row0 = m0 + wm * S::WM;
  if constexpr (sizeof(OutT) == 2) {
    const int st_row = lane >> 2, st_seg = lane & 3;
    // segment s of a row lives in group {0, 2, 1, 3}[s] after step 1
    const int src_lane = st_row + 16 * (((st_seg & 1) << 1) | (st_seg >> 1));
    OutT* c_lane = C + (size_t)(c_row0 + st_row) * N + n0 + wn * S::WN + 8 * st_seg;
#pragma unroll
    for (int i = 0; i < S::TM; ++i)
#pragma unroll
      for (int j = 0; j < S::TN; j += 2) {
        typedef InT h2_t __attribute__((ext_vector_type(2)));
        unsigned x[2], y[2];
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          const h2_t hx = {(InT)acc[i][j][2 * d], (InT)acc[i][j][2 * d + 1]};
          const h2_t hy = {(InT)acc[i][j + 1][2 * d], (InT)acc[i][j + 1][2 * d + 1]};
          x[d] = __builtin_bit_cast(unsigned, hx);
          y[d] = __builtin_bit_cast(unsigned, hy);
#if defined(__HIP_DEVICE_COMPILE__)
          // x of the odd groups <-> y of the even groups
          auto sw = __builtin_amdgcn_permlane16_swap(x[d], y[d], false, false);
          x[d] = sw[0];
          y[d] = sw[1];
#endif
        }
        uint4_t v;
        v[0] = (unsigned)__builtin_amdgcn_ds_bpermute(4 * src_lane, (int)x[0]);
        v[1] = (unsigned)__builtin_amdgcn_ds_bpermute(4 * src_lane, (int)x[1]);
        v[2] = (unsigned)__builtin_amdgcn_ds_bpermute(4 * src_lane, (int)y[0]);
        v[3] = (unsigned)__builtin_amdgcn_ds_bpermute(4 * src_lane, (int)y[1]);
        *reinterpret_cast<out16B_t*>(c_lane + (size_t)(16 * i) * N + 16 * j) = v;
      }
  } else {
    const int c_col0 = n0 + wn * S::WN + 4 * fg;
#pragma unroll
    for (int i = 0; i < S::TM; ++i)
#pragma unroll
      for (int j = 0; j < S::TN; ++j)
        *reinterpret_cast<out4f_t*>(C + (size_t)(c_row0 + fr + 16 * i) * N + c_col0 + 16 * j) = acc[i][j];
  }
}

template <typename S, typename OutT, typename InT>
int launch_ring64(const void* A, const void* B, void* C, int M, int N, int K, hipStream_t st) {
  auto kern = gemm_ring64_kernel<S, InT, OutT>;
  constexpr int lds = S::kLdsBytes;
  static_assert(lds <= kMaxLdsBytes, "ring does not fit in LDS");
  TFK_LDS_OPT_IN(kern, lds);
  const int tiles_m = (M + S::BM - 1) / S::BM, tiles_n = (N + S::BN - 1) / S::BN;
  return launch_kernel(kern, dim3(tiles_m * tiles_n), dim3(S::kThreads), lds, st,
                       static_cast<const InT*>(A), static_cast<const InT*>(B),
                       static_cast<OutT*>(C), M, N, K, tiles_m, tiles_n);
}

// ------------------------------------------------------------------------------------------
// Few rows, few columns or few tiles: the wavefronts of a workgroup share ONE output tile of
// 16*TM x 16*TN and split K among themselves (k-tile t goes to wavefront t % kWaves), each streaming
// its own part of both operands through an LDS ring of its own: no barrier until the partial tiles
// are added up in LDS at the end.
//
// Such problems are bound by how fast a CU takes in its operands: a tile of 32 x 16 does 21 flops per
// byte.  Operand fragments read straight from memory into registers run into the address unit, which
// merges only ADJACENT lanes - the sixteen rows of a fragment lie 16 lanes apart, 64 accesses per
// KiB, a quarter of the L1's rate (32 x 4096 x 4096: 12.7 us).  LDS-direct requests of 8 rows x 128 bytes
// are whole lines: 7.8 us, 4.4 TB/s (the 64 x 64 bounds-checked kernel that ran before: 68.6).
// ------------------------------------------------------------------------------------------
template <int TM_, int TN_, int WAVES_>
struct SplitKShape {
  static constexpr int TM = TM_, TN = TN_, kWaves = WAVES_;
  static constexpr int kStages = 2;                           // k-tiles in a wavefront's ring
  static constexpr int BM = 16 * TM, BN = 16 * TN, BK = 64;
  static constexpr int kThreads = kWaves * kWaveSize;
  static constexpr int kFrags = TM + TN;                      // 16-row operand fragments per 32-deep step
  static constexpr int kLoads = 2 * kFrags;                   // 1 KiB requests (8 rows x 128 bytes) per k-tile
  static constexpr int kStageBytes = kLoads * 1024;
  static constexpr int kPitch = BN + 4;                       // floats per row of a partial tile in LDS
  static constexpr int kRingBytes = kWaves * kStages * kStageBytes;
  static constexpr int kPartBytes = kWaves * BM * kPitch * 4;
  static constexpr int kLdsBytes = kRingBytes > kPartBytes ? kRingBytes : kPartBytes;
  static_assert(kLoads < 64, "vmcnt is a 6-bit counter");
  // the same swizzle as the big kernel's: conflict-free fragment reads of 128-byte rows
  __host__ __device__ static constexpr int swizzle(int row, int c) { return c ^ ((row / 2) % 8); }
};

template <typename S, typename InT, typename OutT>
__global__ __launch_bounds__(S::kThreads) void gemm_split_k_kernel(
    const InT* __restrict__ A, const InT* __restrict__ B, OutT* __restrict__ C, int M, int N, int K, int tiles_m,
    int tiles_n) {
  using V8 = in8_t<InT>;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  // consecutive tiles of one XCD share columns of B (m runs fastest)
  const int pid = xcd_major(blockIdx.x, tiles_m * tiles_n);
  const int m0 = pid % tiles_m * S::BM, n0 = pid / tiles_m * S::BN;

  // Request n of a k-tile: rows 8n .. 8n+7 of A (n < 2 TM) or B, lane l fills physical chunk l % 8 of
  // row l / 8.  Rows past the edge re-fetch the last one.  The chunks of the last k-tile that lie
  // behind K fetch that tile's first chunk instead; their products are masked below.
  const char* a_tile = reinterpret_cast<const char*>(A + (size_t)m0 * K);
  const char* b_tile = reinterpret_cast<const char*>(B + (size_t)n0 * K);
  const int num_k_tiles = (K + S::BK - 1) / S::BK, last_tile = num_k_tiles - 1;
  unsigned off[S::kLoads], off_last[S::kLoads];
#pragma unroll
  for (int n = 0; n < S::kLoads; ++n) {
    const bool of_a = n < 2 * S::TM;
    const int row = (of_a ? n : n - 2 * S::TM) * 8 + lane / 8;
    const int c = S::swizzle(row, lane % 8);
    const unsigned base = (unsigned)min(row, (of_a ? M - m0 : N - n0) - 1) * (unsigned)K * 2u;
    off[n] = base + 16u * c;
    off_last[n] = last_tile * S::BK + 8 * c < K ? off[n] : base;
  }
  const unsigned ring = lds_address(smem) + wave * S::kStages * S::kStageBytes;
  auto request = [&](int stage, int kt) __attribute__((always_inline)) {
    const bool last = kt == last_tile;
#pragma unroll
    for (int n = 0; n < S::kLoads; ++n) {
      const char* src = (n < 2 * S::TM ? a_tile : b_tile) + (size_t)kt * (S::BK * 2);
      // (the LDS destination is an M0 input of the statement, the s_nop the wait state behind an M0 write)
      asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                   :
                   : "v"(last ? off_last[n] : off[n]), "s"(src), "{m0}"(ring + stage * S::kStageBytes + n * 1024)
                   : "memory");
    }
  };
  unsigned rd[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) rd[ks] = ring + lr * 128 + S::swizzle(lr, 4 * ks + lg) * 16;

  float4_t acc[S::TM][S::TN];
#pragma unroll
  for (int i = 0; i < S::TM; ++i)
#pragma unroll
    for (int j = 0; j < S::TN; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

  V8 fr[2][2][S::kFrags];   // [set][32-deep step][fragments of A, then of B]
  auto read = [&](int set, int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int f = 0; f < S::kFrags; ++f)
        fr[set][ks][f] =
            *(__attribute__((address_space(3))) const V8*)(size_t)(rd[ks] + stage * S::kStageBytes + f * 2048);
  };
  auto mask_behind_k = [&](int set) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      if (last_tile * S::BK + (4 * ks + lg) * 8 >= K) {
#pragma unroll
        for (int f = 0; f < S::kFrags; ++f)
#pragma unroll
          for (int t = 0; t < 8; ++t) fr[set][ks][f][t] = (InT)0.f;
      }
  };
  // waits until at most this wavefront's youngest k-tile, if there is one behind the awaited, is still in flight
  auto wait_for_tile = [&](bool one_behind) __attribute__((always_inline)) {
    if (one_behind) wait_vmem<S::kLoads>();
    else wait_vmem<0>();
  };
  const int mine = wave < num_k_tiles ? (last_tile - wave) / S::kWaves + 1 : 0;   // k-tiles of this wavefront
  auto tile_of = [&](int t) __attribute__((always_inline)) { return wave + t * S::kWaves; };
#pragma unroll
  for (int t = 0; t < S::kStages; ++t)
    if (t < mine) request(t, tile_of(t));
  if (mine > 0) {
    wait_for_tile(mine > 1);
    read(0, 0);
  }
  int stage = 0;   // of tile t
  // Tile t: its fragments are on their way into set t % 2; once they have arrived its stage takes tile
  // t + kStages, and the fragments of tile t + 1 are requested under the products of tile t.
  auto step = [&](int t, auto set_c) __attribute__((always_inline)) {
    constexpr int set = decltype(set_c)::value;
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
    if (t + S::kStages < mine) request(stage, tile_of(t + S::kStages));
    stage = stage + 1 == S::kStages ? 0 : stage + 1;
    if (t + 1 < mine) {
      wait_for_tile(t + 2 < mine);
      read(set ^ 1, stage);
    }
    if (K % S::BK != 0 && tile_of(t) == last_tile) mask_behind_k(set);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < S::TM; ++i)
#pragma unroll
        for (int j = 0; j < S::TN; ++j) acc[i][j] = mfma16_t<InT>(fr[set][ks][S::TM + j], fr[set][ks][i], acc[i][j]);
    __builtin_amdgcn_sched_barrier(0);
  };
  for (int t = 0; t < mine; t += 2) {
    step(t, std::integral_constant<int, 0>{});
    if (t + 1 < mine) step(t + 1, std::integral_constant<int, 1>{});
  }
  __syncthreads();   // every ring has been read: the partial tiles take their place

  float* s_part = reinterpret_cast<float*>(smem);
  float* own = s_part + wave * S::BM * S::kPitch;
#pragma unroll
  for (int i = 0; i < S::TM; ++i)
#pragma unroll
    for (int j = 0; j < S::TN; ++j)
      *reinterpret_cast<float4_t*>(own + (16 * i + lr) * S::kPitch + 16 * j + 4 * lg) = acc[i][j];
  __syncthreads();
  for (int f = tid; f < S::BM * S::BN / 4; f += S::kThreads) {
    const int row = f / (S::BN / 4), col = f % (S::BN / 4) * 4;
    float4_t sum = *reinterpret_cast<const float4_t*>(s_part + row * S::kPitch + col);
#pragma unroll
    for (int w = 1; w < S::kWaves; ++w)
      sum += *reinterpret_cast<const float4_t*>(s_part + (w * S::BM + row) * S::kPitch + col);
    if (m0 + row >= M) continue;
    OutT* dst = C + (size_t)(m0 + row) * N + n0 + col;
    if (n0 + col + 4 <= N) {
      typedef OutT out4_t __attribute__((ext_vector_type(4)));
      typedef out4_t out4_any_t __attribute__((aligned(sizeof(OutT))));   // rows of an odd N have no alignment
      *reinterpret_cast<out4_any_t*>(dst) = out4_t{(OutT)sum[0], (OutT)sum[1], (OutT)sum[2], (OutT)sum[3]};
    } else {
#pragma unroll
      for (int r = 0; r < 3; ++r)
        if (n0 + col + r < N) dst[r] = (OutT)sum[r];
    }
  }
}

template <typename S, typename OutT, typename InT>
int launch_split_k(const void* A, const void* B, void* C, int M, int N, int K, hipStream_t st) {
  auto kern = gemm_split_k_kernel<S, InT, OutT>;
  static_assert(S::kLdsBytes <= kMaxLdsBytes, "rings do not fit in LDS");
  if constexpr (S::kLdsBytes > 64 * 1024) TFK_LDS_OPT_IN(kern, S::kLdsBytes);
  const int tiles_m = (M + S::BM - 1) / S::BM, tiles_n = (N + S::BN - 1) / S::BN;
  return launch_kernel(kern, dim3(tiles_m * tiles_n), dim3(S::kThreads), S::kLdsBytes, st, static_cast<const InT*>(A),
                       static_cast<const InT*>(B), static_cast<OutT*>(C), M, N, K, tiles_m, tiles_n);
}

// ------------------------------------------------------------------------------------------
// Operands that do not start at a 16-byte boundary, and short K with many outputs: any M, N; K % 8 == 0.  Register-staged,
// bounds-checked, one LDS stage.
// ------------------------------------------------------------------------------------------
template <typename S, typename OutT, typename InT>
__global__ __launch_bounds__(S::kThreads) void gemm_guarded_kernel(
    const InT* __restrict__ A, const InT* __restrict__ B, OutT* __restrict__ C, int M,
    int N, int K) {
  __shared__ __attribute__((aligned(16))) char sa[S::kABytes];
  __shared__ __attribute__((aligned(16))) char sb[S::kBBytes];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int m0 = blockIdx.x * S::BM, n0 = blockIdx.y * S::BN;
  const int wm = wave / S::WAVES_N, wn = wave % S::WAVES_N;
  const int fr = lane & 31, fg = lane >> 5;

  float16_t acc[S::TM][S::TN];
#pragma unroll
  for (int i = 0; i < S::TM; ++i)
#pragma unroll
    for (int j = 0; j < S::TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  for (int k0 = 0; k0 < K; k0 += S::BK) {
    for (int f = tid; f < S::BM * S::kChunks; f += S::kThreads) {
      const int row = f / S::kChunks, c = f % S::kChunks;
      const int gr = m0 + row, gk = k0 + c * 8;
      uint4_t v = {0u, 0u, 0u, 0u};
      if (gr < M && gk < K) v = *reinterpret_cast<const uint4_t*>(A + (size_t)gr * K + gk);
      *reinterpret_cast<uint4_t*>(sa + row * S::BK * 2 + S::swizzle(row, c) * 16) = v;
    }
    for (int f = tid; f < S::BN * S::kChunks; f += S::kThreads) {
      const int row = f / S::kChunks, c = f % S::kChunks;
      const int gr = n0 + row, gk = k0 + c * 8;
      uint4_t v = {0u, 0u, 0u, 0u};
      if (gr < N && gk < K) v = *reinterpret_cast<const uint4_t*>(B + (size_t)gr * K + gk);
      *reinterpret_cast<uint4_t*>(sb + row * S::BK * 2 + S::swizzle(row, c) * 16) = v;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < S::kKSteps; ++kk) {
      in8_t<InT> af[S::TM], bf[S::TN];
#pragma unroll
      for (int i = 0; i < S::TM; ++i) {
        const int row = wm * S::WM + i * 32 + fr;
        af[i] = *reinterpret_cast<const in8_t<InT>*>(sa + row * S::BK * 2 + S::swizzle(row, 2 * kk + fg) * 16);
      }
#pragma unroll
      for (int j = 0; j < S::TN; ++j) {
        const int row = wn * S::WN + j * 32 + fr;
        bf[j] = *reinterpret_cast<const in8_t<InT>*>(sb + row * S::BK * 2 + S::swizzle(row, 2 * kk + fg) * 16);
      }
#pragma unroll
      for (int i = 0; i < S::TM; ++i)
#pragma unroll
        for (int j = 0; j < S::TN; ++j) acc[i][j] = mfma32_t<InT>(af[i], bf[j], acc[i][j]);
    }
    __syncthreads();
  }

#pragma unroll
  for (int i = 0; i < S::TM; ++i)
#pragma unroll
    for (int j = 0; j < S::TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = m0 + wm * S::WM + i * 32 + 8 * (r / 4) + 4 * fg + (r % 4);
        const int col = n0 + wn * S::WN + j * 32 + fr;
        if (row < M && col < N) store_out(C + (size_t)row * N + col, acc[i][j][r]);
      }
}

using ShapeSmall = GemmShape<64, 64, 32, 2, 2>;    // bounds-checked path

template <typename S, typename OutT, typename InT>
int launch_guarded(const void* A, const void* B, void* C, int M, int N, int K, hipStream_t st) {
  dim3 grid((M + S::BM - 1) / S::BM, (N + S::BN - 1) / S::BN);
  return launch_kernel(gemm_guarded_kernel<S, OutT, InT>, grid, dim3(S::kThreads), 0, st,
                       static_cast<const InT*>(A), static_cast<const InT*>(B),
                       static_cast<OutT*>(C), M, N, K);
}

// ------------------------------------------------------------------------------------------
// Which kernel: the one that a cost model expects to be done first.
//
// The tiles of a problem, the rounds in which 256 CUs do them and the k-tiles of each are known; what
// a k-tile costs is measured.  Microseconds, fitted to 264 problems (M 1-8192, N and K 64-8192, bf16, three
// to eight rotating operand sets; root mean square error 8-16% a kernel).  Taking the expected best is
// 3.5% behind taking the measured best of all kernels on average, and never 2x.
//   ring kernels:    start + rounds * (round + ktiles * (step + shared * fill + unaligned))
//     `shared` is what a CU pays for the others' requests, times how much of the chip a round fills: a
//     128 x 128 tile's k-tile takes 0.30 us with few workgroups, 0.56 with one on every CU (its
//     32 KiB a k-tile then ask 15 TB/s of the L2s), a 256 x 256 tile's 0.85 and 1.6 for four times the work.
//   split-K kernels: start + max(rounds * ktiles of one wavefront * step,
//                                tiles per CU * ktiles * (shared + unaligned)) + tiles per CU * round
//     the latency of one workgroup's chain, or the rate at which a CU takes in all of its workgroups.
// `unaligned` applies where K is no multiple of 64: rows then start anywhere in a 128-byte line.
// ------------------------------------------------------------------------------------------
struct GemmKernel {
  int bm, bn, waves;        // output tile; wavefronts that share its K (ring kernels: 1)
  int per_cu;               // workgroups that a CU holds
  bool ring;
  float start, round, step, shared, unaligned;
  int64_t min_tiles = 0, max_tiles = INT64_MAX;   // where the figures apply
};
constexpr GemmKernel kGemmKernels[] = {
    {16, 16, 4, 4, false, 2.25f, 0.18f, 0.208f, 0.056f, 0.005f},
    {16, 16, 8, 2, false, 2.32f, 0.42f, 0.279f, 0.057f, 0.005f},
    {32, 16, 4, 3, false, 2.36f, 0.28f, 0.259f, 0.089f, 0.009f},
    {32, 32, 1, 8, false, 2.41f, 0.13f, 0.294f, 0.100f, 0.050f},
    {32, 32, 4, 2, false, 2.30f, 0.50f, 0.342f, 0.128f, 0.012f},
    {64, 32, 4, 1, false, 2.42f, 1.44f, 0.527f, 0.235f, 0.042f},
    {64, 64, 4, 1, false, 2.87f, 2.12f, 0.785f, 0.324f, 0.092f},
    {128, 128, 1, 1, true, 0.58f, 3.23f, 0.298f, 0.260f, 0.205f},              // requests 4 tiles ahead
    {128, 128, 1, 1, true, 0.92f, 2.29f, 0.386f, 0.284f, 0.129f, 0, 256},      // 2 tiles ahead: starts sooner
    {128, 128, 1, 2, true, 2.30f, 1.51f, 0.160f, 0.349f, 0.176f, 257},         // ... and shares a CU in pairs
    {192, 128, 1, 1, true, 0.21f, 3.75f, 0.426f, 0.331f, 0.212f},
    {192, 192, 1, 1, true, 0.00f, 4.93f, 0.529f, 0.509f, 0.233f},
    {256, 128, 1, 1, true, 0.00f, 4.60f, 0.496f, 0.447f, 0.266f},
    {256, 192, 1, 1, true, 0.00f, 5.84f, 0.670f, 0.583f, 0.240f},
    {256, 256, 1, 1, true, 0.00f, 6.63f, 0.851f, 0.729f, 0.216f},
};
constexpr int kNumGemmKernels = sizeof(kGemmKernels) / sizeof(kGemmKernels[0]);

// Rows that start anywhere in a line: from K = 328 on these ring kernels fetch whole lines (Ring64Shape::kLines), which costs them a
// segment more at first and saves them 0.13-0.27 us a k-tile. Microseconds as above, fitted to 60 problems (M, N 128-8192, K
// 328-8192; 4-5% root mean square); picks are 2% behind the best of all kernels on average. us, k-tiles that start where rows
// start / whole lines: 1500 x 1500 x 3000, 128 x 128 31.0 / 22.6; 700 x 4096 x 4104 40.2 / 30.5; 2999 x 1544 x 1032,
// 192 x 128 18.7 / 17.3; 3333 x 2288 x 1944, 256 x 128 39.3 / 33.5, 192 x 192 35.3 / 33.6. (The larger tiles leave no room for a third
// segment, and two workgroups of 128 x 128 none for each other; below K = 328 the further segment costs as much as it saves:
// 8192 x 1000 x 328 14.0 / 13.5.)
constexpr int kLinesFrom = 328;
bool takes_lines(int K) { return K % 64 != 0 && K >= kLinesFrom; }
struct LinesKernel {
  int index;                // into kGemmKernels
  float start, round, step, shared;
};
constexpr LinesKernel kLinesKernels[] = {
    {7, 1.63f, 3.67f, 0.317f, 0.139f},
    {10, 1.32f, 4.65f, 0.430f, 0.167f},
    {11, 0.60f, 5.44f, 0.695f, 0.269f},
    {12, 1.36f, 4.11f, 0.660f, 0.281f},
};

// A tile of 160 x 128, figures between those of 128 x 128 and 192 x 128, for grids that the one gives a second round and the
// other leaves CUs idle on (2999 x 1544 x 1032: 208 tiles of 192 rows, 247 of 160). It takes the place of one of these two where it is
// expected to be done sooner. us, the pick / it, of one run each: 2999 x 1544 x 1032 17.3 / 16.6, 613 x 7874 x 2040 26.1 / 22.9, 2547 x
// 1739 x 6712 63.5 / 59.1; 56 such problems take 0.923 of the time (1.00 at most). Of K a multiple of 64, from 256 on: 0.961 over 119
// (1.02 at most): 2466 x 1722 x 256 8.4 / 7.8, 1571 x 3014 x 3008 33.3 / 30.0, 587 x 7483 x 2496 28.3 / 25.8. Not in place of the larger
// tiles: whole lines of 192 x 192, which the model would have it replace now and then, are ahead of it by 5% on average (10% at most)
// over 52 problems (5288 x 4630 x 1768, fp32 result, 94.8 / 104.4).
constexpr LinesKernel kBetween = {-1, 1.45f, 4.15f, 0.373f, 0.153f};
constexpr int kBetweenRows = 160, kBetweenColumns = 128;
constexpr GemmKernel kBetweenWhole = {kBetweenRows, kBetweenColumns, 1, 1, true, 0.40f, 3.49f, 0.362f, 0.296f, 0.f};

float expected_us(const GemmKernel& g, int64_t tiles, int ktiles, bool unaligned_rows, const LinesKernel* lines) {
  const int64_t rounds = (tiles + 256 * g.per_cu - 1) / (256 * g.per_cu);
  const float unaligned = unaligned_rows ? g.unaligned : 0.f;
  const float per_cu = tiles / 256.f;
  if (g.ring) {
    const float fill = std::min(1.f, per_cu / (rounds * g.per_cu));
    if (lines != nullptr) return lines->start + rounds * (lines->round + ktiles * (lines->step + lines->shared * fill));
    return g.start + rounds * g.per_cu * (g.round + ktiles * (g.step + g.shared * fill + unaligned));
  }
  const int chain = (ktiles + g.waves - 1) / g.waves;
  return g.start + std::max(rounds * chain * g.step, per_cu * ktiles * (g.shared + unaligned)) + per_cu * g.round;
}

// Up to K = 128 (16-bit results: 120) with many outputs, what counts is how C leaves, in which the table above does not go by the type (it was
// fitted to 16-bit results), and the bounds-checked kernel is in the race: its k-tiles are 32 deep, and
// several of its workgroups share a CU.  Microseconds, fitted to 521 problems (7 to 13% root mean square): start +
// round per round of the chip + per tile of a CU: tile, depth a k-tile, wide for an fp32 result, odd_k where K is no
// multiple of 64, odd_n where rows of C do not start at 16-byte boundaries.  Picks are 1.6% behind the best
// of all kernels on average and 20% at most; those of the table above 8% and 83% (517 x 3008 x 64, fp32 result:
// 128 x 128 ring 5.9 us, bounds-checked kernel 4.05; 1664 x 1472 x 64 6.2 and 4.8).
struct ShortKKernel {
  int index;                // into kGemmKernels; behind its end: the bounds-checked kernel
  int bm, bn, k_tile;
  float start, round, tile, depth, wide, odd_k, odd_n;
};
constexpr ShortKKernel kShortKKernels[] = {
    {3, 32, 32, 64, 2.93f, 0.f, 0.163f, 0.064f, 0.070f, 0.f, 0.010f},
    {8, 128, 128, 64, 3.34f, 1.31f, 0.303f, 0.415f, 1.54f, 0.178f, 0.277f},
    {11, 192, 192, 64, 2.83f, 3.90f, 0.288f, 0.896f, 3.32f, 0.584f, 0.811f},
    {12, 256, 128, 64, 2.54f, 3.80f, 0.153f, 0.853f, 3.18f, 0.559f, 0.640f},
    {13, 256, 192, 64, 2.68f, 5.32f, 0.f, 1.262f, 4.89f, 0.768f, 0.871f},
    {kNumGemmKernels, 64, 64, 32, 3.23f, 0.f, 0.254f, 0.168f, 0.296f, 0.f, 0.139f},
};

int pick_short_k_kernel(int M, int N, int K, bool c_is_f32) {
  const int64_t row_bytes = (int64_t)N * (c_is_f32 ? 4 : 2);
  int best = 3;
  float best_us = INFINITY;
#pragma unroll
  for (const ShortKKernel& g : kShortKKernels) {
    if (kGemmKernels[g.index % kNumGemmKernels].ring && (M < g.bm || N < g.bn || K < 64)) continue;
    if (g.index == kNumGemmKernels) {
      if (N > 65535 * 64) continue;   // its grid has columns of tiles in y
      // Its tiles are 64 columns wide, so rows of C that are no whole 128-byte lines leave it in parts of lines, which
      // costs from ~32 MiB of C on (5898 x 5498 x 64, fp32 result: 58 us, 128 x 128 ring 33; 8192 x 4160 x 64 33 and 36).
      if (K >= 64 && row_bytes % 128 != 0 && M * row_bytes > (int64_t)32 << 20) continue;
    }
    const int64_t tiles = (int64_t)((M + g.bm - 1) / g.bm) * ((N + g.bn - 1) / g.bn);
    const float per_tile = g.tile + (K + g.k_tile - 1) / g.k_tile * g.depth + (c_is_f32 ? g.wide : 0.f) +
                           (K % 64 != 0 ? g.odd_k : 0.f) + (row_bytes % 16 != 0 ? g.odd_n : 0.f);
    const float us = g.start + (tiles + 255) / 256 * g.round + tiles / 256.f * per_tile;
    if (us < best_us) {
      best = g.index;
      best_us = us;
    }
  }
  return best;
}

// What runs in place of `pick`, a kernel of the table: the tile between where it is ahead of a ring kernel of its kind, the same tile with whole
// lines where rows start anywhere in one. Their positions are those behind the bounds-checked kernel's.
constexpr int kLinesAt = kNumGemmKernels + 1, kBetweenWholeAt = kLinesAt + sizeof(kLinesKernels) / sizeof(kLinesKernels[0]),
              kBetweenLinesAt = kBetweenWholeAt + 1, kNumGemmLaunchers = kBetweenLinesAt + 1;
int stand_in(int pick, int M, int N, int K) {
  const bool lines = takes_lines(K);
  int at = pick;
  const LinesKernel* of_pick = nullptr;
  if (lines) {
    for (const LinesKernel& l : kLinesKernels)
      if (l.index == pick) {
        of_pick = &l;
        at = kLinesAt + (int)(&l - kLinesKernels);
      }
    if (of_pick == nullptr) return pick;
  } else if (K % 64 != 0 || K < 256 || pick < 7) {
    return pick;
  }
  if (pick > 10) return at;   // (tiles that are larger both ways)
  if (M < kBetweenRows || N < kBetweenColumns) return at;
  const GemmKernel& g = kGemmKernels[pick];
  const int ktiles = (K + 63) / 64;
  auto expected = [&](const GemmKernel& k, const LinesKernel* l) {
    return expected_us(k, (int64_t)((M + k.bm - 1) / k.bm) * ((N + k.bn - 1) / k.bn), ktiles, lines, l);
  };
  if (expected(kBetweenWhole, lines ? &kBetween : nullptr) < expected(g, of_pick)) return lines ? kBetweenLinesAt : kBetweenWholeAt;
  return at;
}

// The kernel of a call whose operands start at 16-byte boundaries: a position in the launchers of dispatch().
int pick_gemm_kernel(int M, int N, int K, bool c_is_f32) {
  // (2^35 elements of C with a K below the ring kernels' are more threads than a launch of the split-K kernels may have)
  if (K < 64 && (int64_t)M * N >= (int64_t)1 << 35) return kNumGemmKernels;
  if (K <= (c_is_f32 ? 128 : 120) && (int64_t)((M + 63) / 64) * ((N + 63) / 64) >= 96) return pick_short_k_kernel(M, N, K, c_is_f32);
  int best = 0, best_plain = 0;
  float best_us = INFINITY, best_plain_us = INFINITY;
  const int ktiles = (K + 63) / 64;
#pragma unroll   // the divisions are by constants then
  for (int i = 0; i < kNumGemmKernels; ++i) {
    const GemmKernel& g = kGemmKernels[i];
    if (g.ring && (M < g.bm || N < g.bn || K < 64)) continue;   // (what gemm_ring64_kernel asks for)
    const int64_t tiles = (int64_t)((M + g.bm - 1) / g.bm) * ((N + g.bn - 1) / g.bn);
    if (tiles < g.min_tiles || tiles > g.max_tiles) continue;
    const float plain_us = expected_us(g, tiles, ktiles, K % 64 != 0, nullptr);
    float us = plain_us;
    if (takes_lines(K))
      for (const LinesKernel& l : kLinesKernels)
        if (l.index == i) us = expected_us(g, tiles, ktiles, true, &l);
    if (us < best_us) {
      best = i;
      best_us = us;
    }
    if (plain_us < best_plain_us) {
      best_plain = i;
      best_plain_us = plain_us;
    }
  }
  // Where tiles of 256 x 192 or 256 x 256 would be picked if there were no whole lines they are: the two fits do not compare well there
  // (us, those / the whole-line tile that is expected to be ahead: 5530 x 3814 x 1184 55.0 / 68.5, 7568 x 5021 x 1424 113 / 135, 3727 x 6430 x
  // 1256 66 / 76; 80 such problems 1.077 of the time with whole lines, those tiles 0.3% behind the best of all).
  if (best_plain == 13 || best_plain == 14) return best_plain;
  return stand_in(best, M, N, K);
}

template <typename OutT, typename InT>
int dispatch(const void* A, const void* B, void* C, int M, int N, int K, hipStream_t st) {
  using Launcher = int (*)(const void*, const void*, void*, int, int, int, hipStream_t);
  static constexpr Launcher kLaunchers[] = {
      launch_split_k<SplitKShape<1, 1, 4>, OutT, InT>, launch_split_k<SplitKShape<1, 1, 8>, OutT, InT>,
      launch_split_k<SplitKShape<2, 1, 4>, OutT, InT>, launch_split_k<SplitKShape<2, 2, 1>, OutT, InT>,
      launch_split_k<SplitKShape<2, 2, 4>, OutT, InT>, launch_split_k<SplitKShape<4, 2, 4>, OutT, InT>,
      launch_split_k<SplitKShape<4, 4, 4>, OutT, InT>,
      launch_ring64<Ring64Shape<128, 128, 4>, OutT, InT>, launch_ring64<Ring64Shape<128, 128, 2>, OutT, InT>,
      launch_ring64<Ring64Shape<128, 128, 2>, OutT, InT>, launch_ring64<Ring64Shape<192, 128, 2>, OutT, InT>,
      launch_ring64<Ring64Shape<192, 192, 2>, OutT, InT>, launch_ring64<Ring64Shape<256, 128, 2>, OutT, InT>,
      launch_ring64<Ring64Shape<256, 192, 2>, OutT, InT>, launch_ring64<Ring64Shape<256, 256, 2>, OutT, InT>,
      launch_guarded<ShapeSmall, OutT, InT>,
      launch_ring64<Ring64Shape<128, 128, 2, 5>, OutT, InT>, launch_ring64<Ring64Shape<192, 128, 2, 4>, OutT, InT>,
      launch_ring64<Ring64Shape<192, 192, 2, 3>, OutT, InT>, launch_ring64<Ring64Shape<256, 128, 2, 3>, OutT, InT>,
      launch_ring64<Ring64Shape<kBetweenRows, kBetweenColumns, 2>, OutT, InT>,
      launch_ring64<Ring64Shape<kBetweenRows, kBetweenColumns, 2, 4>, OutT, InT>,
  };
  static_assert(sizeof(kLaunchers) / sizeof(kLaunchers[0]) == kNumGemmLaunchers,
                "a launcher per row of kGemmKernels, the bounds-checked kernel, one per row of kLinesKernels, the two of 160 rows");
  // LDS-direct requests take 16 bytes at a 16-byte boundary.
  if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B)) % 16 != 0)
    return kLaunchers[kNumGemmKernels](A, B, C, M, N, K, st);
  return kLaunchers[pick_gemm_kernel(M, N, K, sizeof(OutT) == 4)](A, B, C, M, N, K, st);
}

}  // namespace
}  // namespace tfk

namespace tfk {
namespace {
int check_gemm_args(const char* who, const void* A, const void* B, const void* C, int64_t M, int64_t N, int64_t K,
                    int tm, int tn, int tk, int num_stages, int pipeline_level) {
  TFK_REQUIRE(A && B && C, TF_ERR_INVALID_ARG, "%s: null pointer", who);
  TFK_REQUIRE(M > 0 && N > 0 && K > 0, TF_ERR_INVALID_ARG, "%s: M, N, K must be positive", who);
  TFK_REQUIRE(M < (1 << 30) && N < (1 << 30) && K < (1 << 22), TF_ERR_INVALID_ARG, "%s: dimension too large", who);
  TFK_REQUIRE(tm > 0 && tn > 0 && tk > 0, TF_ERR_INVALID_ARG, "%s: tile sizes must be positive", who);
  TFK_REQUIRE(M % tm == 0 && N % tn == 0 && K % tk == 0, TF_ERR_INVALID_ARG,
              "%s: tile [%d,%d,%d] does not divide problem [%lld,%lld,%lld]", who, tm, tn, tk,
              (long long)M, (long long)N, (long long)K);
  TFK_REQUIRE(num_stages >= 1 && num_stages <= 3, TF_ERR_INVALID_ARG, "%s: num_stages must be 1, 2 or 3", who);
  TFK_REQUIRE(pipeline_level >= 0 && pipeline_level <= 2, TF_ERR_INVALID_ARG,
              "%s: pipeline_level must be 0, 1 or 2", who);
  return TF_OK;
}
}  // namespace
}  // namespace tfk

extern "C" int tf_gemm_f16(const void* A, const void* B, void* C, int c_is_f16, int64_t M,
                           int64_t N, int64_t K, int tm, int tn, int tk, int num_stages,
                           int pipeline_level, void* stream) {
  using namespace tfk;
  if (int rc = check_gemm_args("tf_gemm_f16", A, B, C, M, N, K, tm, tn, tk, num_stages, pipeline_level)) return rc;
  TFK_REQUIRE(K % 8 == 0, TF_ERR_UNSUPPORTED, "tf_gemm_f16: K (%lld) must be a multiple of 8",
              (long long)K);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (c_is_f16) return dispatch<half_t, half_t>(A, B, C, (int)M, (int)N, (int)K, st);
  return dispatch<float, half_t>(A, B, C, (int)M, (int)N, (int)K, st);
}

extern "C" int tf_gemm(const void* A, const void* B, void* C, int dtype, int c_is_f32, int64_t M, int64_t N,
                       int64_t K, int tm, int tn, int tk, int num_stages, int pipeline_level, void* stream) {
  using namespace tfk;
  if (dtype == TF_DTYPE_F16)
    return tf_gemm_f16(A, B, C, c_is_f32 ? 0 : 1, M, N, K, tm, tn, tk, num_stages, pipeline_level, stream);
  TFK_REQUIRE(dtype == TF_DTYPE_BF16, TF_ERR_UNSUPPORTED, "tf_gemm: dtype must be TF_DTYPE_F16 or TF_DTYPE_BF16");
  if (int rc = check_gemm_args("tf_gemm", A, B, C, M, N, K, tm, tn, tk, num_stages, pipeline_level)) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  // bf16: the same kernels with the bf16 MFMAs (every kernel of this file is a template of the
  // operand type)
  TFK_REQUIRE(K % 8 == 0, TF_ERR_UNSUPPORTED, "tf_gemm: K (%lld) must be a multiple of 8", (long long)K);
  if (c_is_f32) return dispatch<float, bf16_t>(A, B, C, (int)M, (int)N, (int)K, st);
  return dispatch<bf16_t, bf16_t>(A, B, C, (int)M, (int)N, (int)K, st);
}

extern "C" int tf_gemm_kernel_index(int64_t M, int64_t N, int64_t K, int c_is_f32) {
  if (M <= 0 || N <= 0 || K <= 0 || M >= (1 << 30) || N >= (1 << 30) || K >= (1 << 22)) return -1;
  return tfk::pick_gemm_kernel((int)M, (int)N, (int)K, c_is_f32 != 0);
}
