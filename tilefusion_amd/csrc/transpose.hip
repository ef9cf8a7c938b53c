// Transposes a batch of matrices of 16-bit elements: out[b][c][r] = in[b][r][c], for keys stored [D, Lkv] that no
// attention kernel reads as they are (lengths that are no multiple of 8, wide heads, heads between the tuned sizes).
//
// A workgroup takes a 64 x 64 tile through LDS: rows come as 8-byte loads at any even address (rows of an odd length have
// no alignment), leave as 16-byte stores.  Bound by memory: [64, 128, 4096] in 20.5 us (6.5 TB/s;
// torch's transposed copy 99), [32, 256, 1024] 5.4 (28.8), an odd [64, 64, 1337] 6.0 (14.5); from about 4 us (7) for small
// ones it is the launch.  Attention with such a key: 1024 x 1024 x 256 causal 45.2 us (68.7 with torch's copy), 777 x 777 x
// 128 38.5 (49.6), 1337 x 1337 x 64 causal 35.0 (41.8).
#include "common.hpp"

namespace tfk {
namespace {

constexpr int kTile = 64, kTransposeThreads = 256;
// 66 elements a row in LDS: the rows that a gather of one column touches lie in different banks
constexpr int kTransposePitch = kTile + 2;

__global__ __launch_bounds__(kTransposeThreads) void transpose_kernel(const unsigned short* __restrict__ in,
                                                                      unsigned short* __restrict__ out, int rows, int cols) {
  __shared__ unsigned short tile[kTile * kTransposePitch];
  const int tid = threadIdx.x;
  const int c0 = blockIdx.x * kTile, r0 = blockIdx.y * kTile;
  in += (size_t)blockIdx.z * rows * cols;
  out += (size_t)blockIdx.z * rows * cols;
  typedef unsigned short four_t __attribute__((ext_vector_type(4)));
  typedef four_t four_any_t __attribute__((aligned(2)));
  four_t v[kTile / 16];
#pragma unroll
  for (int i = 0; i < kTile / 16; ++i) {
    const int r = min(r0 + 16 * i + tid / 16, rows - 1), c = c0 + 4 * (tid % 16);
    const unsigned short* src = in + (size_t)r * cols;
    if (c + 4 <= cols) {
      v[i] = *reinterpret_cast<const four_any_t*>(src + c);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[i][e] = src[min(c + e, cols - 1)];   // (beyond the end: not stored)
    }
  }
#pragma unroll
  for (int i = 0; i < kTile / 16; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) tile[(16 * i + tid / 16) * kTransposePitch + 4 * (tid % 16) + e] = v[i][e];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kTile / 32; ++i) {
    const int c = 32 * i + tid / 8, r = 8 * (tid % 8);
    if (c0 + c >= cols || r0 + r >= rows) continue;
    unsigned short x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = tile[(r + e) * kTransposePitch + c];
    unsigned short* dst = out + (size_t)(c0 + c) * rows + r0 + r;
    if (rows % 8 == 0) {
      uint4_t w;
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = x[2 * e] | (unsigned)x[2 * e + 1] << 16;
      *reinterpret_cast<uint4_t*>(dst) = w;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (r0 + r + e < rows) dst[e] = x[e];
    }
  }
}

}  // namespace
}  // namespace tfk

extern "C" int tf_transpose_16bit(const void* in, void* out, int64_t batch, int64_t rows, int64_t cols, void* stream) {
  using namespace tfk;
  TFK_REQUIRE(in && out, TF_ERR_INVALID_ARG, "tf_transpose_16bit: null pointer");
  TFK_REQUIRE(batch > 0 && rows > 0 && cols > 0, TF_ERR_INVALID_ARG, "tf_transpose_16bit: sizes must be positive");
  TFK_REQUIRE(batch < 65536 && rows < (1 << 21) && cols < (1 << 24), TF_ERR_INVALID_ARG, "tf_transpose_16bit: dimension too large");
  TFK_REQUIRE(reinterpret_cast<uintptr_t>(in) % 2 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0, TF_ERR_INVALID_ARG,
              "tf_transpose_16bit: out must start at a 16-byte boundary");
  const dim3 grid((unsigned)((cols + kTile - 1) / kTile), (unsigned)((rows + kTile - 1) / kTile), (unsigned)batch);
  return launch_kernel(transpose_kernel, grid, dim3(kTransposeThreads), 0, static_cast<hipStream_t>(stream),
                       static_cast<const unsigned short*>(in), static_cast<unsigned short*>(out), (int)rows, (int)cols);
}
