// Fused back-to-back GEMM for narrow K and P (up to 128 each): tiles of B and C stream through LDS, over any N.
//
// A workgroup is 8 wavefronts on 64 * kRB rows of A.  Four of them side by side take 16 * kRB rows each, and the two
// such sets (h = 0, 1) take one half of every 64-wide n-tile each: a wavefront multiplies 32 rows of the B tile with its A
// rows (S^T, 16 x 16 accumulators), rounds the result to 16 bits, which is the A operand of the second product for the
// same 32 n (as in fused_two_gemms.hip: the B rows are dealt so that a lane's eight are consecutive), and multiplies that
// with 32 columns of the C tile.  At the end the two sets trade halves of their partial sums through LDS.
//
// What bounds it: LDS reads, matrix products and the tiles' way from the L2 are about level with 128 rows (kRB = 2,
// K = P = 128: 128 KiB of fragments = 1024 cycles a tile, 64 MFMAs a SIMD = 1024, 32 KiB through the LDS-direct path
// ~800); with 64 rows the same LDS reads serve half the products.  Measured, a tile takes 0.75 us with 128 rows and
// 0.53 with 64 (two wavefronts per SIMD; the kernel before, a wavefront to 16 rows of whole tiles: 1.23 and 0.8),
// and a workgroup 5.5 us beside its tiles, 2.5-6 more where it leaves 8-16 MiB of partial sums.  us, bf16, before /
// now: 4000 rows x N 4096, K = P = 128 24.0 / 19.2 (two launches: 16.4 and 4.6 traced), N 4080 (whose tail took the plain
// kernel) 71.7 / 19.3; 8192 x 8192 49.9 / 38.1, K = P = 64 81 / 24.7, K 96, P 48 92 / 25.7; K 48, P 80 (padded
// copies) 16384 x 128 27.6 / 6.8.
//
// Ring: kStages tiles; tile t + 1 has landed when tile t is multiplied, so that its B fragments are requested behind
// the second product of tile t and no wavefront starts a tile waiting for LDS; the others are in flight.  A's rows
// take the same way into registers, through the LDS that D leaves by.
//
// Nothing is padded in memory: chunks of 8 k beyond K are zeros in the registers of both operands, rows beyond P are
// computed on a copy of the last one and not stored, and the last n-tile overlaps its neighbour (N < 64: is
// completed with copies), with the n that are not its own zeros in both operands of the second product.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "fused_two_gemms_stream.hpp"

namespace tfk {
namespace {

template <typename T> using vec4_t = T __attribute__((ext_vector_type(4)));
template <typename T> using vec8_t = T __attribute__((ext_vector_type(8)));
template <typename T>
TFK_DEVICE float4_t mfma_t(vec8_t<T> a, vec8_t<T> b, float4_t c) {
  if constexpr (std::is_same_v<T, bf16_t>) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  else return mfma_16x16x32(a, b, c);
}

constexpr int kTN = 64;        // n per tile
constexpr int kRowWaves = 4;   // wavefronts side by side along the rows
constexpr int kWavesS = 8;

// Physical 16-byte chunk of logical chunk c in an LDS row of CH chunks: the sixteen rows that a fragment read touches
// at one logical chunk lie in sixteen different 16-byte bank groups.
template <int CH>
__host__ __device__ constexpr int swz(int row, int c) {   // consecutive rows (A, C)
  if constexpr (CH >= 16) return c ^ (row % 16);
  else return c ^ ((row / 2) % 8);
}
// row of the B tile that element i of 16-row fragment nt multiplies, and the key that suits those rows
__host__ __device__ constexpr int b_frag_row(int nt, int i) { return 32 * (nt / 2) + 8 * (i / 4) + 4 * (nt % 2) + i % 4; }
template <int CH>
__host__ __device__ constexpr int swz_b(int row, int c) {
  if constexpr (CH >= 16) return c ^ ((((row >> 3) & 3) << 2) | (row & 3));
  else return c ^ ((((row >> 3) & 3) << 1) | ((row >> 1) & 1));
}

template <int kKS, int kPT, int kRB>
struct StreamShape {
  static constexpr int kKP = kKS <= 2 ? 64 : 128;          // LDS row pitch of A and B, in elements
  static constexpr int kRows = 16 * kRB * kRowWaves;
  static constexpr int kBBytes = kTN * kKP * 2, kCBytes = 16 * kPT * kTN * 2;
  static constexpr int kStage = kBBytes + kCBytes;
  static constexpr int kABytes = kRows * kKP * 2, kDBytes = kRows * kPT * 16 * 2;
  static constexpr int kAD = kABytes > kDBytes ? kABytes : kDBytes;   // A on its way in, D on its way out
  static constexpr int kFit = (kMaxLdsBytes - kAD) / kStage;
  static constexpr int kStages = kFit > 6 ? 6 : kFit;
  static constexpr int kLds = kAD + kStages * kStage;
  static constexpr int kExchange = kWavesS * (kPT / 2) * kRB * 1024;
  static_assert(kPT % 2 == 0 && kStages >= 4 && kExchange <= kStages * kStage, "LDS plan");
};

template <typename T, int kKS, int kPT, int kRB>
__global__ __launch_bounds__(kWavesS * 64) void fused_stream_kernel(
    const T* __restrict__ A, const T* __restrict__ B, const T* __restrict__ C, T* __restrict__ D,
    float* __restrict__ W, int M, int N, int K, int P, int parts, int tiles_per_part) {
  using S = StreamShape<kKS, kPT, kRB>;
  constexpr int kCh = S::kKP / 8;                  // chunks per row of A and B in LDS
  constexpr int kAInstr = S::kABytes / 1024, kBInstr = S::kBBytes / 1024, kInstr = S::kStage / 1024;
  constexpr int kReq = (kInstr + kWavesS - 1) / kWavesS;   // requests of a tile per wavefront (a surplus one repeats another)
  constexpr int kAReq = kAInstr / kWavesS;
  static_assert(kAInstr % kWavesS == 0, "A: whole requests for every wavefront");
  constexpr int kStages = S::kStages, kAhead = kStages - 1;
  static_assert(kAhead * kReq + kAReq < 64, "vmcnt is a 6-bit counter");
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  char* ring = smem + S::kAD;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave_id = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave = wave_id % kRowWaves, half = wave_id / kRowWaves;
  const int lr = lane & 15, lg = lane >> 4;
  // (parts are the fast index: ids go round-robin to the 8 XCDs, so that a part's tiles are fetched into
  // one or a few of their L2s and not into all)
  const int part = blockIdx.x % parts, m0 = blockIdx.x / parts * S::kRows;
  const size_t batch = blockIdx.z;
  A += batch * (size_t)M * K;
  B += batch * (size_t)N * K;
  C += batch * (size_t)P * N;
  D += batch * (size_t)M * P;
  const unsigned a_lds = lds_address(smem), ring_lds = lds_address(ring);

  // this workgroup's n-tiles: [t_begin, t_begin + n_tiles)
  const int all_tiles = (N + kTN - 1) / kTN;
  const int t_begin = part * tiles_per_part;
  const int n_tiles = min(tiles_per_part, all_tiles - t_begin);

  // ---- requests: 1 KiB each, scalar tile base + a 32-bit lane offset computed once --------------------------
  auto dma = [](unsigned off, const char* base, unsigned lds_addr) __attribute__((always_inline)) {
    // (the LDS destination is an M0 input of the statement; the s_nop is the wait state an M0 write needs)
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "{m0}"(lds_addr) : "memory");
  };
  const int k_chunks = K / 8;
#pragma unroll
  for (int q = 0; q < kAReq; ++q) {
    const int i = wave_id + kWavesS * q;
    const int row = i * (64 / kCh) + lane / kCh;
    const int c = min(swz<kCh>(row, lane % kCh), k_chunks - 1);
    const int m = min(m0 + row, M - 1) - m0;   // rows past M are never stored
    dma(((unsigned)m * (unsigned)K + (unsigned)c * 8u) * 2u, reinterpret_cast<const char*>(A + (size_t)m0 * K), a_lds + i * 1024);
  }
  unsigned req_off[kReq], req_lds[kReq];
  bool req_b[kReq];
#pragma unroll
  for (int q = 0; q < kReq; ++q) {
    int i = wave_id + kWavesS * q;
    if (i >= kInstr) i -= kInstr;
    req_b[q] = i < kBInstr;
    req_lds[q] = i * 1024;
    if (i < kBInstr) {
      const int row = i * (64 / kCh) + lane / kCh;
      const int c = min(swz_b<kCh>(row, lane % kCh), k_chunks - 1);
      req_off[q] = ((unsigned)min(row, N - 1) * (unsigned)K + (unsigned)c * 8u) * 2u;
    } else {
      const int row = (i - kBInstr) * 8 + lane / 8;
      const int c = min(swz<8>(row, lane % 8), N / 8 - 1);
      req_off[q] = ((unsigned)min(row, P - 1) * (unsigned)N + (unsigned)c * 8u) * 2u;
    }
  }
  // first n of tile t (the last one is moved back to end at N)
  auto tile_n0 = [&](int t) __attribute__((always_inline)) { return max(0, min((t_begin + t) * kTN, N - kTN)); };
  auto request_tile = [&](int t) __attribute__((always_inline)) {
    const int n0 = tile_n0(min(t, n_tiles - 1));   // (past the end: lands in a stage that nobody reads again)
    const char* b_base = reinterpret_cast<const char*>(B + (size_t)n0 * K);
    const char* c_base = reinterpret_cast<const char*>(C + n0);
    const unsigned stage = ring_lds + (t % kStages) * S::kStage;
#pragma unroll
    for (int q = 0; q < kReq; ++q) dma(req_off[q], req_b[q] ? b_base : c_base, stage + req_lds[q]);
  };
#pragma unroll
  for (int t = 0; t < kAhead; ++t) request_tile(t);

  // ---- fragments ----------------------------------------------------------------------------------------
  const bool k_tail = K % 32 != 0;                                      // the last step of the first product is half full
  const bool k_valid = (4 * (kKS - 1) + lg) < k_chunks;                 // this lane's chunk of it
  const vec8_t<T> zero8 = {};
  vec8_t<T> af[kKS][kRB];
  vec8_t<T> bf[kKS][2], cf[kPT];
  auto read_b = [&](int t) __attribute__((always_inline)) {
    const char* sB = ring + (t % kStages) * S::kStage;
#pragma unroll
    for (int ks = 0; ks < kKS; ++ks)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int row = b_frag_row(2 * half + j, lr);
        bf[ks][j] = *reinterpret_cast<const vec8_t<T>*>(sB + row * S::kKP * 2 + swz_b<kCh>(row, 4 * ks + lg) * 16);
      }
    if (k_tail) {
#pragma unroll
      for (int j = 0; j < 2; ++j) bf[kKS - 1][j] = k_valid ? bf[kKS - 1][j] : zero8;
    }
  };
  auto read_c = [&](int t) __attribute__((always_inline)) {
    const char* sC = ring + (t % kStages) * S::kStage + S::kBBytes;
#pragma unroll
    for (int pt = 0; pt < kPT; ++pt) {
      const int row = 16 * pt + lr;
      cf[pt] = *reinterpret_cast<const vec8_t<T>*>(sC + row * kTN * 2 + swz<8>(row, 4 * half + lg) * 16);
    }
  };

  barrier_keep_vmem<(kAhead - 1) * kReq>();   // A and tile 0 have landed
#pragma unroll
  for (int ks = 0; ks < kKS; ++ks)
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) {
      const int row = (wave * kRB + rb) * 16 + lr;
      af[ks][rb] = *reinterpret_cast<const vec8_t<T>*>(smem + row * S::kKP * 2 + swz<kCh>(row, 4 * ks + lg) * 16);
    }
  if (k_tail) {
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) af[kKS - 1][rb] = k_valid ? af[kKS - 1][rb] : zero8;
  }
  read_b(0);

  float4_t acc2[kPT][kRB];
#pragma unroll
  for (int pt = 0; pt < kPT; ++pt)
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) acc2[pt][rb] = float4_t{0.f, 0.f, 0.f, 0.f};

  auto multiply_tile = [&](int t, auto masked_c) __attribute__((always_inline)) {
    read_c(t);
    float4_t acc1[2][kRB];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) acc1[j][rb] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < kKS; ++ks)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int rb = 0; rb < kRB; ++rb) acc1[j][rb] = mfma_t<T>(bf[ks][j], af[ks][rb], acc1[j][rb]);
    __builtin_amdgcn_sched_barrier(0);
    read_b(t + 1);   // (behind the last tile: a stage of older data, not used)
    // lane (m = lr, group lg) holds A*B[m][n0 + 32*half + 8*lg + 0..7] in acc1[0][rb], acc1[1][rb]
    vec8_t<T> pa[kRB];
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pa[rb][r] = (T)acc1[0][rb][r];
        pa[rb][4 + r] = (T)acc1[1][rb][r];
      }
    if constexpr (decltype(masked_c)::value) {
      const int n0 = tile_n0(t), n = 32 * half + 8 * lg;
      const bool own = n0 + n >= (t_begin + t) * kTN && n0 + n < N;
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) pa[rb] = own ? pa[rb] : zero8;
#pragma unroll
      for (int pt = 0; pt < kPT; ++pt) cf[pt] = own ? cf[pt] : zero8;
    }
#pragma unroll
    for (int pt = 0; pt < kPT; ++pt)
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) acc2[pt][rb] = mfma_t<T>(pa[rb], cf[pt], acc2[pt][rb]);
    __builtin_amdgcn_sched_barrier(0);
  };
  // tile t + 1 has landed (own requests; behind the barrier everybody's), and everybody is done with tile t - 1,
  // whose stage is filled next
  auto next_tile = [&](int t) __attribute__((always_inline)) {
    wait_vmem<(kAhead - 2) * kReq>();
    barrier_only();
    request_tile(t + kAhead);
  };
  const int whole = min(n_tiles, N / kTN - t_begin);   // tiles that are all their own
  int t = 0;
  for (; t < whole; ++t) {
    next_tile(t);
    multiply_tile(t, std::false_type{});
  }
  if (t < n_tiles) {
    next_tile(t);
    multiply_tile(t, std::true_type{});
  }

  // ---- the two sets trade halves: set h keeps column blocks [h * kPT / 2, (h + 1) * kPT / 2) -------------
  wait_vmem_all();   // the surplus requests: the ring is used for the exchange, and must not be written behind the end
  __syncthreads();
  constexpr int kHalf = kPT / 2;
  float4_t* trade = reinterpret_cast<float4_t*>(ring) + lane;   // [half][wave][kHalf * kRB][64]
  float4_t out[kHalf][kRB];
  auto give_and_keep = [&](auto h_c) __attribute__((always_inline)) {
    constexpr int h = decltype(h_c)::value;
#pragma unroll
    for (int i = 0; i < kHalf; ++i)
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) {
        trade[((h * kRowWaves + wave) * kHalf * kRB + i * kRB + rb) * 64] = acc2[(1 - h) * kHalf + i][rb];
        out[i][rb] = acc2[h * kHalf + i][rb];
      }
  };
  if (half == 0) give_and_keep(std::integral_constant<int, 0>{});
  else give_and_keep(std::integral_constant<int, 1>{});
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kHalf; ++i)
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) out[i][rb] += trade[(((1 - half) * kRowWaves + wave) * kHalf * kRB + i * kRB + rb) * 64];

  // out[i][rb][r] = D[m0 + (wave * kRB + rb) * 16 + 4*lg + r][(half * kHalf + i) * 16 + lr]
  const int p_lane = half * kHalf * 16 + lr;
  if (W != nullptr) {
    // fp32 partial sums straight from the registers: 16 adjacent lanes write 64 contiguous bytes
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + (wave * kRB + rb) * 16 + 4 * lg + r;
        float* w = W + ((batch * parts + part) * (size_t)M + m) * P + p_lane;
        if (m < M) {
#pragma unroll
          for (int i = 0; i < kHalf; ++i)
            if (p_lane + 16 * i < P) __builtin_nontemporal_store(out[i][rb][r], w + 16 * i);
        }
      }
    return;
  }
  // 16-bit result, staged through LDS for 16-byte stores along rows
  T* sD = reinterpret_cast<T*>(smem);
  constexpr int kDPitch = kPT * 16;
#pragma unroll
  for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
    for (int i = 0; i < kHalf; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sD[((wave * kRB + rb) * 16 + 4 * lg + r) * kDPitch + p_lane + 16 * i] = (T)out[i][rb][r];
  __syncthreads();
  constexpr int kDChunks = kDPitch / 8;
  for (int f = tid; f < S::kRows * kDChunks; f += kWavesS * 64) {
    const int row = f / kDChunks, c = f % kDChunks;
    if (m0 + row < M && c * 8 < P)
      __builtin_nontemporal_store(*reinterpret_cast<const uint4_t*>(sD + row * kDPitch + c * 8),
                                  reinterpret_cast<uint4_t*>(D + (size_t)(m0 + row) * P + c * 8));
  }
}

// D[b][i] = 16-bit(sum over parts of W[b][part][i]), i over the `elems` = M * P elements of a problem.  64 lanes take
// 4 elements each, kGroups wavefronts every kGroups-th part, up to eight loads in flight: one thread that walked all the parts of
// its elements took a trip to memory for each (64 rows x N 8192, both launches: 22.8 / 9.7 us).
constexpr int kGroups = 4;
template <typename T, int kFlight>
__global__ __launch_bounds__(kGroups * 64) void fused_sum_parts_kernel(const float* __restrict__ W, T* __restrict__ D,
                                                                       int parts, size_t elems) {
  __shared__ float4_t sums[kGroups][64];
  const int lane = threadIdx.x & 63, group = threadIdx.x >> 6;
  const size_t i = ((size_t)blockIdx.x * 64 + lane) * 4;
  const bool in = i < elems;
  const float* w = W + (size_t)blockIdx.z * parts * elems + (in ? i : 0);
  float4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int first = group; first < parts; first += kGroups * kFlight) {
    float4_t v[kFlight];
#pragma unroll
    for (int j = 0; j < kFlight; ++j)   // (past the last part: the last one again, not added)
      v[j] = __builtin_nontemporal_load(reinterpret_cast<const float4_t*>(w + (size_t)min(first + kGroups * j, parts - 1) * elems));
#pragma unroll
    for (int j = 0; j < kFlight; ++j)
      if (first + kGroups * j < parts) acc += v[j];
  }
  sums[group][lane] = acc;
  __syncthreads();
  if (group != 0 || !in) return;
#pragma unroll
  for (int g = 1; g < kGroups; ++g) acc += sums[g][lane];
  const vec4_t<T> h = {(T)acc[0], (T)acc[1], (T)acc[2], (T)acc[3]};
  *reinterpret_cast<vec4_t<T>*>(D + (size_t)blockIdx.z * elems + i) = h;
}

template <typename T, int kKS, int kPT, int kRB>
int launch_stream(const FusedCall& c, FusedPlan plan) {
  using S = StreamShape<kKS, kPT, kRB>;
  auto kern = fused_stream_kernel<T, kKS, kPT, kRB>;
  TFK_LDS_OPT_IN(kern, S::kLds);
  const dim3 grid((unsigned)((c.M + S::kRows - 1) / S::kRows) * (unsigned)plan.parts, 1, c.batch);
  float* w = plan.parts > 1 ? static_cast<float*>(c.workspace) : nullptr;
  if (int rc = launch_kernel(kern, grid, dim3(kWavesS * 64), S::kLds, c.stream, static_cast<const T*>(c.A),
                       static_cast<const T*>(c.B), static_cast<const T*>(c.C), static_cast<T*>(c.D), w, c.M, c.N, c.K, c.P,
                       plan.parts, plan.tiles_per_part)) return rc;
  if (plan.parts == 1) return TF_OK;
  const size_t elems = (size_t)c.M * c.P;
  auto sum = plan.parts <= kGroups       ? fused_sum_parts_kernel<T, 1>
             : plan.parts <= 2 * kGroups ? fused_sum_parts_kernel<T, 2>
             : plan.parts <= 4 * kGroups ? fused_sum_parts_kernel<T, 4>
                                         : fused_sum_parts_kernel<T, 8>;
  return launch_kernel(sum, dim3((unsigned)((elems / 4 + 63) / 64), 1, c.batch), dim3(kGroups * 64), 0, c.stream, w,
                       static_cast<T*>(c.D), plan.parts, elems);
}
template <typename T, int kKS, int kPT>
int pick_rows(const FusedCall& c, FusedPlan plan) {
  return plan.rows == 128 ? launch_stream<T, kKS, kPT, 2>(c, plan) : launch_stream<T, kKS, kPT, 1>(c, plan);
}
template <typename T, int kKS>
int pick_p(const FusedCall& c, FusedPlan plan) {
  if (c.P <= 64) return pick_rows<T, kKS, 4>(c, plan);
  if (c.P <= 96) return pick_rows<T, kKS, 6>(c, plan);
  return pick_rows<T, kKS, 8>(c, plan);
}
template <typename T>
int pick_k(const FusedCall& c, FusedPlan plan) {
  if (c.K <= 64) return pick_p<T, 2>(c, plan);
  if (c.K <= 96) return pick_p<T, 3>(c, plan);
  return pick_p<T, 4>(c, plan);
}
}  // namespace

int run_fused_stream(const FusedCall& c, FusedPlan plan) {
  return c.bf16 ? pick_k<bf16_t>(c, plan) : pick_k<half_t>(c, plan);
}

}  // namespace tfk
