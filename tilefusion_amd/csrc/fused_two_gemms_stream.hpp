// The streaming form of the fused back-to-back GEMM (fused_two_gemms_stream.hip).
#pragma once

#include "common.hpp"

namespace tfk {

struct FusedCall {
  const void *A, *B, *C;
  void *D, *workspace;   // workspace: parts * batch * M * P floats where the plan has more than one part
  bool bf16;
  int batch, M, N, K, P;
  hipStream_t stream;
};
// `rows` (64 or 128) rows of A per workgroup; the n-tiles of 64 in `parts` ranges of `tiles_per_part`.
struct FusedPlan { int rows, parts, tiles_per_part; };

// K, P <= 128; K, N, P multiples of 8; operands at 16-byte boundaries.
int run_fused_stream(const FusedCall& c, FusedPlan plan);

}  // namespace tfk
