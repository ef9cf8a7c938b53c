// Fused back-to-back GEMM for gfx950: D[M,P] = (A[M,K] * B[K,N]) * C[N,P], fp16 or bf16 in/out,
// fp32 accumulate; the intermediate A*B lives only in registers (rounded to the element type like
// the reference does, include/kernels/fused_two_gemms_device.cuh:200).
//
// Counterpart of ke_fused_two_gemms (include/kernels/fused_two_gemms_device.cuh:114-214) and its
// host launcher (src/kernels/fused_two_gemms.cu:66-144).  CDNA4 design:
//   * one workgroup = 64 rows of A (4 wavefronts x 16 rows), v_mfma_f32_16x16x32_f16;
//   * the first GEMM is computed transposed, S^T = B_buf * A^T, so that every lane ends up
//     holding one row m of A*B: the 16x16 accumulator layout (lane -> column m, registers ->
//     4 consecutive n) is, after fp16 conversion, exactly the A-operand fragment layout of
//     the second MFMA up to a permutation of the reduction index, which the C-operand loads
//     mirror.  No LDS round trip, no shuffles for the intermediate;
//   * B and C chunks go global -> LDS directly (global_load_lds_dwordx4) into XOR-swizzled
//     tiles shared by the 4 wavefronts; A fragments are private to a wavefront and are read
//     straight from global memory into registers;
//   * D leaves from registers, four adjacent lanes to 64 contiguous bytes of a row.
// Problems of several n-tiles stream (fused_two_gemms_stream.hip).
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "fused_two_gemms_stream.hpp"

namespace tfk {
namespace {

// The kernels move 16-bit elements without looking at them; the element type T (half_t or bf16_t)
// only selects the MFMA and the float -> T conversions.
template <typename T> using vec2_t = T __attribute__((ext_vector_type(2)));
template <typename T> using vec4_t = T __attribute__((ext_vector_type(4)));
template <typename T> using vec8_t = T __attribute__((ext_vector_type(8)));
template <typename T>
TFK_DEVICE float4_t mfma_t(vec8_t<T> a, vec8_t<T> b, float4_t c) {
  if constexpr (std::is_same_v<T, bf16_t>) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  else return mfma_16x16x32(a, b, c);
}

constexpr int kRowsPerBlock = 64;
constexpr int kWaves = 4;
constexpr int kThreads = kWaves * kWaveSize;

// Physical 16-byte chunk for logical chunk c of `row` in a tile whose rows hold CH chunks.
template <int CH>
__host__ __device__ constexpr int swz(int row, int c) {
  constexpr int kRowsPer256B = CH >= 16 ? 1 : 16 / CH;
  return c ^ ((row / kRowsPer256B) % CH);
}

// ------------------------------------------------------------------------------------------
// Plain kernel: one workgroup = 64 rows (4 wavefronts x 16), n-tiles of TN, k-chunks of KC.
//
// Per n-tile and k-chunk the order of events is chosen for latency (at the benchmark shape
// the whole kernel is one n-tile and one k-chunk, 64 MFMAs per wavefront, so its run time is
// the sum of one trip to memory and one short dependent chain):
//   * A fragments are requested FIRST (they come from HBM, the tiles of B and C from the L2),
//     then the B tile, then the C tile, all asynchronously; the first product starts as soon
//     as A and B have landed, with the C tile still in flight;
//   * fragment reads run one step ahead of the MFMAs across both products;
//   * B rows are dealt to the 16-row MFMA fragments so that the fp16-rounded accumulators of
//     the first product are the second MFMA's operand fragment for EIGHT CONSECUTIVE n
//     (fragment nt takes rows 32*(nt/2) + 8*(i/4) + 4*(nt%2) + i%4, i = 0..15): the matching C
//     fragment is then one 16-byte read;
//   * the second product is computed transposed (D^T = C^T * S^T), which leaves a lane with
//     four consecutive columns of one row of D; pairs of tiles are re-dealt with
//     v_permlane16_swap + ds_bpermute so that four adjacent lanes store 64 contiguous bytes.
//     No LDS staging of D, no barrier in the epilogue.
// ------------------------------------------------------------------------------------------
// row of the B tile that element i of 16-row fragment nt multiplies
__host__ __device__ constexpr int b_frag_row(int nt, int i) { return 32 * (nt / 2) + 8 * (i / 4) + 4 * (nt % 2) + i % 4; }
// XOR key of a B-tile row: the sixteen rows of a fragment get sixteen different keys
template <int CH>
__host__ __device__ constexpr int b_key(int row) {
  if constexpr (CH >= 16) return ((row >> 3) & 3) << 2 | (row & 3);
  else return (row / (16 / CH)) % CH;
}

template <typename T, int TN, int TP, int KC>
__global__ __launch_bounds__(kThreads) void fused_two_gemms_kernel(
    const T* __restrict__ A, const T* __restrict__ B, const T* __restrict__ C,
    T* __restrict__ D, int M, int N, int K, int P) {
  constexpr int kBCh = KC / 8;       // 16-byte chunks per sB row
  constexpr int kCCh = TN / 8;       // per sC row
  constexpr int kKSteps = KC / 32;
  constexpr int kNT = TN / 16;       // 16-wide n tiles of the first GEMM
  constexpr int kPT = TP / 16;       // 16-wide p tiles of the second GEMM
  constexpr int kSteps2 = TN / 32;
  constexpr int kBInstr = TN * kBCh / 64, kCInstr = (TP * kCCh + 63) / 64;   // 1 KiB requests per tile
  constexpr int kBPerWave = (kBInstr + kWaves - 1) / kWaves, kCPerWave = (kCInstr + kWaves - 1) / kWaves;
  static_assert(TN % 32 == 0 && KC % 32 == 0 && TP % 16 == 0, "whole MFMA base tiles");
  __shared__ __attribute__((aligned(1024))) char sB[TN * KC * 2];
  __shared__ __attribute__((aligned(1024))) char sC[kCInstr * 1024];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int m0 = blockIdx.x * kRowsPerBlock;
  const int p0 = blockIdx.y * TP;
  const size_t batch = blockIdx.z;
  A += batch * (size_t)M * K;
  B += batch * (size_t)N * K;
  C += batch * (size_t)P * N;
  D += batch * (size_t)M * P;

  // Every global access is a scalar base (tile origin, 64-bit, computed on the scalar unit) plus
  // a 32-bit byte offset per lane that stays inside the tile: the address arithmetic in front of
  // the first request is on this kernel's critical path (per-lane 64-bit pointers for the 4 + 16
  // requests of a wavefront cost ~1 us of the ~3.5 us the kernel ran).
  const int a_row = min(wave * 16 + lr, M - 1 - m0);  // clamped: rows past M are never stored
  const char* a_base = reinterpret_cast<const char*>(A + (size_t)m0 * K);
  const unsigned a_off = ((unsigned)a_row * (unsigned)K + 8u * lg) * 2u;
  const unsigned sB_addr = lds_address(sB), sC_addr = lds_address(sC);
  auto dma = [](unsigned off, const char* base, unsigned lds_addr) __attribute__((always_inline)) {
    // the LDS destination is an M0 INPUT of the statement: the compiler writes M0 itself and
    // cannot use the register for anything else between that write and the request; the s_nop
    // is the wait state an M0 write needs in front of an LDS-direct load
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(off), "s"(base), "{m0}"(lds_addr)
                 : "memory");
  };

  // 1 KiB request i of the B tile covers rows 64 / kBCh * i ..; lane l fills physical chunk
  // l % kBCh of its row with the logical chunk the key maps there.  The same for C with the
  // plain key.  Requests beyond the tile (a C tile smaller than 1 KiB) re-fetch row 0.
  auto request_b = [&](int n0, int k0) __attribute__((always_inline)) {
    const char* b_base = reinterpret_cast<const char*>(B + (size_t)n0 * K + k0);
#pragma unroll
    for (int q = 0; q < kBPerWave; ++q) {
      const int i = wave + kWaves * q;
      if (kBInstr % kWaves != 0 && i >= kBInstr) break;
      const int row = i * (64 / kBCh) + lane / kBCh;
      const int c = (lane % kBCh) ^ b_key<kBCh>(row);
      dma(((unsigned)row * (unsigned)K + (unsigned)c * 8u) * 2u, b_base, sB_addr + i * 1024);
    }
  };
  auto request_c = [&](int n0) __attribute__((always_inline)) {
    const char* c_base = reinterpret_cast<const char*>(C + (size_t)p0 * N + n0);
#pragma unroll
    for (int q = 0; q < kCPerWave; ++q) {
      const int i = wave + kWaves * q;
      if (kCInstr % kWaves != 0 && i >= kCInstr) break;
      const int row = min(i * (64 / kCCh) + lane / kCCh, TP - 1);
      const int c = swz<kCCh>(row, lane % kCCh);
      dma(((unsigned)row * (unsigned)N + (unsigned)c * 8u) * 2u, c_base, sC_addr + i * 1024);
    }
  };
  // requests of this wavefront that are still allowed in flight when B (and A) must be there
  const int c_requests = (kCInstr % kWaves == 0 || wave < kCInstr % kWaves) ? kCPerWave : kCPerWave - 1;

  auto read_b = [&](vec8_t<T>* dst, int ks) __attribute__((always_inline)) {
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt) {
      const int row = b_frag_row(nt, lr);
      dst[nt] = *reinterpret_cast<const vec8_t<T>*>(sB + row * KC * 2 + ((ks * 4 + lg) ^ b_key<kBCh>(row)) * 16);
    }
  };
  auto read_c = [&](vec8_t<T>* dst, int s2) __attribute__((always_inline)) {
#pragma unroll
    for (int pt = 0; pt < kPT; ++pt) {
      const int row = pt * 16 + lr;
      dst[pt] = *reinterpret_cast<const vec8_t<T>*>(sC + row * TN * 2 + swz<kCCh>(row, 4 * s2 + lg) * 16);
    }
  };

  float4_t acc2[kPT];
#pragma unroll
  for (int pt = 0; pt < kPT; ++pt) acc2[pt] = float4_t{0.f, 0.f, 0.f, 0.f};

  for (int n0 = 0; n0 < N; n0 += TN) {
    float4_t acc1[kNT];
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt) acc1[nt] = float4_t{0.f, 0.f, 0.f, 0.f};

    for (int k0 = 0; k0 < K; k0 += KC) {
      const bool first_chunk = k0 == 0;
      // previous readers of sB (and, at a new n-tile, of sC) are done
      if (n0 != 0 || k0 != 0) barrier_lds_only();
      vec8_t<T> af[kKSteps];
      // All three kinds of request are issued from assembly, so that the compiler places no
      // vector-memory waits of its own (it would drain everything, the C tile included, in
      // front of the first LDS read or the first use of an A fragment).
      {
        const char* a_chunk = a_base + (size_t)k0 * 2;
#pragma unroll
        for (int ks = 0; ks < kKSteps; ++ks)
          // (early-clobber outputs: a fragment register never doubles as the address register of
          //  a later request)
          asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3"
                       : "=&v"(af[ks])
                       : "v"(a_off), "s"(a_chunk), "n"(ks * 64)
                       : "memory");
      }
      // the A requests are on their way before the arithmetic of the B and C requests starts.
      // Between here and the wait below the compiler believes the fragment registers written
      // although the data is still in flight: nothing in between reads them (only requests and
      // their scalar address arithmetic are issued), and tests/test_gpu_fused_two_gemms.py::
      // test_every_plain_kernel_instance_is_exact pins that, for every instance of this kernel and
      // both element types, on problems with several k-chunks and n-tiles.
      __builtin_amdgcn_sched_barrier(0);
      request_b(n0, k0);
      if (first_chunk) request_c(n0);
      // A and B have landed once at most this wavefront's C requests are outstanding (loads
      // retire in order); the fragment registers are re-defined behind the wait so that no use
      // of them can be scheduled in front of it.
      if (first_chunk && c_requests == kCPerWave) {
        asm volatile("s_waitcnt vmcnt(%0)" : : "n"(kCPerWave) : "memory");
      } else if (first_chunk && kCPerWave > 1) {
        asm volatile("s_waitcnt vmcnt(%0)" : : "n"(kCPerWave > 1 ? kCPerWave - 1 : 0) : "memory");
      } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
#pragma unroll
      for (int ks = 0; ks < kKSteps; ++ks) asm volatile("" : "+v"(af[ks]));
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");

      // first product, transposed: acc1[nt] += B rows (fragment nt) x A^T, reads one step ahead
      vec8_t<T> bf[2][kNT];
      read_b(bf[0], 0);
#pragma unroll
      for (int ks = 0; ks < kKSteps; ++ks) {
        if (ks + 1 < kKSteps) read_b(bf[(ks + 1) & 1], ks + 1);
#pragma unroll
        for (int nt = 0; nt < kNT; ++nt) acc1[nt] = mfma_t<T>(bf[ks & 1][nt], af[ks], acc1[nt]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // the C tile has landed for everybody
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    // second product, transposed: lane (m = lr, group lg) holds A*B[m][32*s2 + 8*lg + 0..7] in
    // acc1[2*s2][0..3], acc1[2*s2 + 1][0..3]; acc2[pt] += C rows (p) x that
    vec8_t<T> cf[2][kPT];
    read_c(cf[0], 0);
#pragma unroll
    for (int s2 = 0; s2 < kSteps2; ++s2) {
      if (s2 + 1 < kSteps2) read_c(cf[(s2 + 1) & 1], s2 + 1);
      vec8_t<T> pa;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pa[r] = (T)acc1[2 * s2][r];
        pa[4 + r] = (T)acc1[2 * s2 + 1][r];
      }
#pragma unroll
      for (int pt = 0; pt < kPT; ++pt) acc2[pt] = mfma_t<T>(cf[s2 & 1][pt], pa, acc2[pt]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // Epilogue: acc2[pt][r] = D[m0 + 16*wave + lr][p0 + 16*pt + 4*lg + r].
  const int d_row0 = m0 + wave * 16;
  if constexpr (kPT % 2 == 0) {
    // Pairs of tiles: the 16-lane groups g and g^1 trade halves (v_permlane16_swap), after which
    // group 0/2 holds columns 0-7 / 8-15 of tile pt and group 1/3 the same of tile pt+1, 16 bytes
    // per lane; ds_bpermute then moves the 16 bytes of (row r, segment s) to lane 4*r + s, so
    // that a store writes 16 rows x 64 contiguous bytes with four adjacent lanes per row.
    const int st_row = lane >> 2, st_seg = lane & 3;
    const int src_lane = st_row + 16 * (((st_seg & 1) << 1) | (st_seg >> 1));
    T* d_lane = D + (size_t)(d_row0 + st_row) * P + p0 + 8 * st_seg;
    const bool row_ok = d_row0 + st_row < M;
    uint4_t v[kPT / 2];
#pragma unroll
    for (int pt = 0; pt < kPT; pt += 2) {
      typedef vec2_t<T> h2_t;
      unsigned x[2], y[2];
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const h2_t hx = {(T)acc2[pt][2 * d], (T)acc2[pt][2 * d + 1]};
        const h2_t hy = {(T)acc2[pt + 1][2 * d], (T)acc2[pt + 1][2 * d + 1]};
        x[d] = __builtin_bit_cast(unsigned, hx);
        y[d] = __builtin_bit_cast(unsigned, hy);
#if defined(__HIP_DEVICE_COMPILE__)
        auto sw = __builtin_amdgcn_permlane16_swap(x[d], y[d], false, false);
        x[d] = sw[0];
        y[d] = sw[1];
#endif
      }
      v[pt / 2][0] = (unsigned)__builtin_amdgcn_ds_bpermute(4 * src_lane, (int)x[0]);
      v[pt / 2][1] = (unsigned)__builtin_amdgcn_ds_bpermute(4 * src_lane, (int)x[1]);
      v[pt / 2][2] = (unsigned)__builtin_amdgcn_ds_bpermute(4 * src_lane, (int)y[0]);
      v[pt / 2][3] = (unsigned)__builtin_amdgcn_ds_bpermute(4 * src_lane, (int)y[1]);
    }
    // streaming stores: D is written once and not read again here, and an ordinary store next
    // to the operand reads costs this latency-bound kernel 10%
    if (row_ok) {
#pragma unroll
      for (int pt = 0; pt < kPT; pt += 2)
        __builtin_nontemporal_store(v[pt / 2], reinterpret_cast<uint4_t*>(d_lane + 16 * pt));
    }
  } else {
    // a single 16-column tile: 8 bytes per lane
#pragma unroll
    for (int pt = 0; pt < kPT; ++pt) {
      vec4_t<T> v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = (T)acc2[pt][r];
      if (d_row0 + lr < M)
        *reinterpret_cast<vec4_t<T>*>(D + (size_t)(d_row0 + lr) * P + p0 + 16 * pt + 4 * lg) = v;
    }
  }
}

template <typename T, int TN, int TP, int KC>
int launch(const void* A, const void* B, const void* C, void* D, int batch, int M, int N, int K,
           int P, hipStream_t st) {
  dim3 grid((M + kRowsPerBlock - 1) / kRowsPerBlock, P / TP, batch);
  return launch_kernel(fused_two_gemms_kernel<T, TN, TP, KC>, grid, dim3(kThreads), 0, st,
                       static_cast<const T*>(A), static_cast<const T*>(B),
                       static_cast<const T*>(C), static_cast<T*>(D), M, N, K, P);
}

template <typename T, int TN, int TP>
int pick_kc(const void* A, const void* B, const void* C, void* D, int batch, int M, int N, int K,
            int P, hipStream_t st) {
  if (K % 128 == 0) return launch<T, TN, TP, 128>(A, B, C, D, batch, M, N, K, P, st);
  return launch<T, TN, TP, 32>(A, B, C, D, batch, M, N, K, P, st);
}

template <typename T, int TN>
int pick_tp(const void* A, const void* B, const void* C, void* D, int batch, int M, int N, int K,
            int P, hipStream_t st) {
  if (P % 128 == 0) return pick_kc<T, TN, 128>(A, B, C, D, batch, M, N, K, P, st);
  if (P % 64 == 0) return pick_kc<T, TN, 64>(A, B, C, D, batch, M, N, K, P, st);
  return pick_kc<T, TN, 16>(A, B, C, D, batch, M, N, K, P, st);
}

}  // namespace
}  // namespace tfk

namespace tfk {
namespace {
int check_fused_args(const char* who, const void* A, const void* B, const void* C, const void* D, int64_t batch,
                     int64_t M, int64_t N, int64_t K, int64_t P, int tm, int tn, int tk, int tp) {
  TFK_REQUIRE(A && B && C && D, TF_ERR_INVALID_ARG, "%s: null pointer", who);
  TFK_REQUIRE(batch > 0 && M > 0 && N > 0 && K > 0 && P > 0, TF_ERR_INVALID_ARG, "%s: sizes must be positive", who);
  TFK_REQUIRE(batch < 65536 && M < (1 << 30) && N < (1 << 24) && K < (1 << 24) && P < (1 << 24),
              TF_ERR_INVALID_ARG, "%s: dimension too large", who);
  TFK_REQUIRE(tm > 0 && tn > 0 && tk > 0 && tp > 0, TF_ERR_INVALID_ARG, "%s: tile sizes must be positive", who);
  TFK_REQUIRE(M % tm == 0 && N % tn == 0 && K % tk == 0 && P % tp == 0, TF_ERR_INVALID_ARG,
              "%s: tile [%d,%d,%d,%d] does not divide problem [%lld,%lld,%lld,%lld]", who, tm, tn, tk, tp,
              (long long)M, (long long)N, (long long)K, (long long)P);
  TFK_REQUIRE(K % 32 == 0 && N % 32 == 0 && P % 16 == 0, TF_ERR_UNSUPPORTED,
              "%s: needs K %% 32 == 0, N %% 32 == 0, P %% 16 == 0 (got K=%lld N=%lld P=%lld); zero-pad K and N "
              "(the torch op does)", who, (long long)K, (long long)N, (long long)P);
  return TF_OK;
}
}  // namespace
}  // namespace tfk

namespace tfk {
namespace {
// The plain kernel for element type T (arguments already checked)
template <typename T>
int run_plain(const void* A, const void* B, const void* C, void* D, int64_t batch, int64_t M, int64_t N, int64_t K,
              int64_t P, hipStream_t st) {
  if (N % 128 == 0) return pick_tp<T, 128>(A, B, C, D, (int)batch, (int)M, (int)N, (int)K, (int)P, st);
  return pick_tp<T, 32>(A, B, C, D, (int)batch, (int)M, (int)N, (int)K, (int)P, st);
}

// Which problems stream (fused_two_gemms_stream.hip), and how they are cut.
//
// The plain kernel is made for one n-tile: it starts ~1 us sooner and several of its workgroups share a CU, but it
// loads, waits and multiplies one tile after the other, by k-chunks of 32 unless K % 128 == 0, once for every 16
// columns of D unless P % 64 == 0.  us, bf16, plain / streaming: N = 128, K = P = 128, 16384 rows 5.1 / 6.2, 262144 rows
// 36 / 50; N = 256, K = P = 64, 32768 rows 5.9 / 6.5; N = 320 10.5 / 6.9; N = 256, K = 96, P = 48, 16384 rows 5.7 / 6.2,
// 32768 rows 11.0 / 6.5; N = 192, K = P = 128, 64 rows 7.6 / 5.8.
bool takes_plain(int64_t batch, int64_t M, int64_t N, int64_t K, int64_t P) {
  if (N % 32 != 0 || K % 32 != 0 || P % 16 != 0) return false;   // (it would have to be padded in memory)
  return (N <= 128 || (N <= 256 && N % 128 == 0 && K < 128)) && (P % 64 == 0 || M * batch <= 16384);
}
bool may_stream(int64_t batch, int64_t M, int64_t N, int64_t K, int64_t P) {
  return K > 32 && K <= 128 && P <= 128 && K % 8 == 0 && P % 8 == 0 && N % 8 == 0 &&
         (M + 63) / 64 < (1 << 20) && !takes_plain(batch, M, N, K, P);
}

// Rows per workgroup (64 or 128) and the cut along N, by expected time: a workgroup takes its tiles in turn, one on
// a CU; parts cost a second launch and a trip of fp32 sums through memory (and with the workspace ~10.5 us of the calling
// thread, against 6-7 for one launch).  Fitted to 330 problems (64..32768
// rows, N 16..8192, the K and P of the sweep), 1.2% behind the best of up to 12 plans each on average.  Without room for
// partial sums (`may_cut` false) there is one part.
FusedPlan plan_stream(int64_t batch, int64_t M, int64_t N, int64_t K, int64_t P, bool may_cut) {
  const int64_t tiles = (N + 63) / 64;
  const double k_steps = (double)((K + 31) / 32), p_blocks = P <= 64 ? 4 : P <= 96 ? 6 : 8;
  FusedPlan plan = {64, 1, (int)tiles};
  double best = 0;
  auto consider = [&](int rows, int64_t wanted) {
    const int64_t row_blocks = (M + rows - 1) / rows * batch;
    const int64_t per = (tiles + wanted - 1) / wanted, parts = (tiles + per - 1) / per;
    const int64_t groups = row_blocks * parts, rounds = (groups + 255) / 256;
    const double tile = rows == 64 ? 0.128 + 0.038 * k_steps + 0.027 * p_blocks : 0.131 + 0.027 * k_steps + 0.052 * p_blocks;
    const double fill = 0.847 + 0.153 * std::min(1.0, (double)groups / 256.0);
    double t = (rows == 64 ? 5.5 : 5.7) + (rows == 64 ? 1.1 : 1.6) * (double)(rounds - 1) + (double)(rounds * per) * tile * fill;
    if (parts > 1) t = std::max(10.5, t + 3.0 + 0.315e-6 * 4.0 * (double)(parts * batch * M * P));
    if (best == 0 || t < best) {
      best = t;
      plan = {rows, (int)parts, (int)per};
    }
  };
  for (int rows : {64, 128}) {
    const int64_t row_blocks = (M + rows - 1) / rows * batch;
    consider(rows, 1);
    if (!may_cut) continue;
    for (int64_t target : {256, 512})
      if (target / row_blocks > 1) consider(rows, std::min(tiles, target / row_blocks));
    if (row_blocks <= 256)
      for (int64_t parts = 2; parts < tiles && parts * row_blocks <= 512; parts *= 2) consider(rows, parts);
  }
  return plan;
}

bool aligned16(const void* A, const void* B, const void* C, const void* D) {
  return (reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(C) |
          reinterpret_cast<uintptr_t>(D)) % 16 == 0;
}

size_t partial_bytes(const FusedPlan& plan, int64_t batch, int64_t M, int64_t P) {
  return plan.parts > 1 ? (size_t)plan.parts * (size_t)batch * (size_t)M * (size_t)P * sizeof(float) : 0;
}

// What a problem runs with `room` bytes for partial sums; rows = 0: the plain kernel.
FusedPlan plan_fused(int64_t batch, int64_t M, int64_t N, int64_t K, int64_t P, size_t room) {
  if (!may_stream(batch, M, N, K, P)) return {0, 1, 0};
  const FusedPlan plan = plan_stream(batch, M, N, K, P, room > 0);
  return partial_bytes(plan, batch, M, P) <= room ? plan : plan_stream(batch, M, N, K, P, false);
}

int run_fused(const void* A, const void* B, const void* C, void* D, bool bf16, int64_t batch, int64_t M, int64_t N,
              int64_t K, int64_t P, FusedPlan plan, void* workspace, hipStream_t st) {
  if (plan.rows > 0 && aligned16(A, B, C, D)) {
    const FusedCall call = {A, B, C, D, workspace, bf16, (int)batch, (int)M, (int)N, (int)K, (int)P, st};
    return run_fused_stream(call, plan);
  }
  if (bf16) return run_plain<bf16_t>(A, B, C, D, batch, M, N, K, P, st);
  return run_plain<half_t>(A, B, C, D, batch, M, N, K, P, st);
}
}  // namespace
}  // namespace tfk

extern "C" int tf_fused_two_gemms_f16(const void* A, const void* B, const void* C, void* D,
                                      int64_t batch, int64_t M, int64_t N, int64_t K, int64_t P,
                                      int tm, int tn, int tk, int tp, void* stream) {
  using namespace tfk;
  if (int rc = check_fused_args("tf_fused_two_gemms_f16", A, B, C, D, batch, M, N, K, P, tm, tn, tk, tp)) return rc;
  return run_fused(A, B, C, D, false, batch, M, N, K, P, plan_fused(batch, M, N, K, P, 0), nullptr, static_cast<hipStream_t>(stream));
}

extern "C" size_t tf_fused_two_gemms_workspace_bytes(int dtype, int64_t batch, int64_t M, int64_t N, int64_t K,
                                                     int64_t P) {
  using namespace tfk;
  if ((dtype != TF_DTYPE_F16 && dtype != TF_DTYPE_BF16) || batch <= 0 || M <= 0 || N <= 0 || K <= 0 || P <= 0) return 0;
  return partial_bytes(plan_fused(batch, M, N, K, P, SIZE_MAX), batch, M, P);
}

extern "C" int tf_fused_two_gemms_rows(int64_t batch, int64_t M, int64_t N, int64_t K, int64_t P, size_t workspace_bytes) {
  if (batch <= 0 || M <= 0 || N <= 0 || K <= 0 || P <= 0) return 0;
  return tfk::plan_fused(batch, M, N, K, P, workspace_bytes).rows;
}

extern "C" int tf_fused_two_gemms_ws(const void* A, const void* B, const void* C, void* D, int dtype, int64_t batch,
                                     int64_t M, int64_t N, int64_t K, int64_t P, int tm, int tn, int tk, int tp,
                                     void* workspace, size_t workspace_bytes, void* stream) {
  using namespace tfk;
  if (workspace == nullptr || workspace_bytes == 0 || (dtype != TF_DTYPE_F16 && dtype != TF_DTYPE_BF16))
    return tf_fused_two_gemms(A, B, C, D, dtype, batch, M, N, K, P, tm, tn, tk, tp, stream);
  if (int rc = check_fused_args("tf_fused_two_gemms_ws", A, B, C, D, batch, M, N, K, P, tm, tn, tk, tp)) return rc;
  const FusedPlan plan = plan_fused(batch, M, N, K, P, workspace_bytes);
  TFK_REQUIRE(plan.parts == 1 || reinterpret_cast<uintptr_t>(workspace) % 16 == 0, TF_ERR_INVALID_ARG,
              "tf_fused_two_gemms_ws: workspace must be 16-byte aligned");
  return run_fused(A, B, C, D, dtype == TF_DTYPE_BF16, batch, M, N, K, P, plan, workspace, static_cast<hipStream_t>(stream));
}

extern "C" int tf_fused_two_gemms_narrow(const void* A, const void* B, const void* C, void* D, int dtype, int64_t batch,
                                         int64_t M, int64_t N, int64_t K, int64_t P, void* workspace,
                                         size_t workspace_bytes, void* stream) {
  using namespace tfk;
  TFK_REQUIRE(A && B && C && D, TF_ERR_INVALID_ARG, "tf_fused_two_gemms_narrow: null pointer");
  TFK_REQUIRE(batch > 0 && M > 0 && N > 0 && K > 0 && P > 0, TF_ERR_INVALID_ARG,
              "tf_fused_two_gemms_narrow: sizes must be positive");
  TFK_REQUIRE(batch < 65536 && M < (1 << 30) && N < (1 << 24), TF_ERR_INVALID_ARG,
              "tf_fused_two_gemms_narrow: dimension too large");
  TFK_REQUIRE(dtype == TF_DTYPE_F16 || dtype == TF_DTYPE_BF16, TF_ERR_UNSUPPORTED,
              "tf_fused_two_gemms_narrow: dtype must be TF_DTYPE_F16 or TF_DTYPE_BF16");
  TFK_REQUIRE(may_stream(batch, M, N, K, P) && aligned16(A, B, C, D), TF_ERR_UNSUPPORTED,
              "tf_fused_two_gemms_narrow: needs 32 < K <= 128, P <= 128, multiples of 8 (got K=%lld N=%lld P=%lld) and "
              "operands at 16-byte boundaries, and takes no problem that tf_fused_two_gemms runs in one n-tile",
              (long long)K, (long long)N, (long long)P);
  TFK_REQUIRE(workspace == nullptr || reinterpret_cast<uintptr_t>(workspace) % 16 == 0, TF_ERR_INVALID_ARG,
              "tf_fused_two_gemms_narrow: workspace must be 16-byte aligned");
  const FusedPlan plan = plan_fused(batch, M, N, K, P, workspace != nullptr ? workspace_bytes : 0);
  return run_fused(A, B, C, D, dtype == TF_DTYPE_BF16, batch, M, N, K, P, plan, workspace, static_cast<hipStream_t>(stream));
}

extern "C" int tf_fused_two_gemms(const void* A, const void* B, const void* C, void* D, int dtype, int64_t batch,
                                  int64_t M, int64_t N, int64_t K, int64_t P, int tm, int tn, int tk, int tp,
                                  void* stream) {
  using namespace tfk;
  if (dtype == TF_DTYPE_F16) return tf_fused_two_gemms_f16(A, B, C, D, batch, M, N, K, P, tm, tn, tk, tp, stream);
  TFK_REQUIRE(dtype == TF_DTYPE_BF16, TF_ERR_UNSUPPORTED,
              "tf_fused_two_gemms: dtype must be TF_DTYPE_F16 or TF_DTYPE_BF16");
  // bf16: the same kernels with the bf16 MFMA, a bf16 intermediate and bf16 output
  if (int rc = check_fused_args("tf_fused_two_gemms", A, B, C, D, batch, M, N, K, P, tm, tn, tk, tp)) return rc;
  return run_fused(A, B, C, D, true, batch, M, N, K, P, plan_fused(batch, M, N, K, P, 0), nullptr, static_cast<hipStream_t>(stream));
}
