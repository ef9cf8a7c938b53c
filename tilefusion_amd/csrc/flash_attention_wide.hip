// Flash-attention instances for head dimensions above 128 (V as it comes).
#include "flash_attention.hpp"

namespace tfk {
namespace {
template <typename T, int D>
int launch_wide(const AttentionCall& c) {
  if (c.splits > 1) return launch_split<T, D, false>(c);
  if (c.causal) return launch_w<T, D, D, false, false, true, 4, 1, false>(c);
  if (c.rows == 128) return launch_w<T, D, D, false, false, false, 8, 1, false>(c);
  return launch_w<T, D, D, false, false, false, 4, 1, false>(c);
}
template <typename T>
int pick_wide(const AttentionCall& c, int D) {
  if (D == 160) return launch_wide<T, 160>(c);
  if (D == 192) return launch_wide<T, 192>(c);
  return launch_wide<T, 256>(c);
}
}  // namespace

int run_attention_wide(const AttentionCall& c, int D) { return c.bf16 ? pick_wide<bf16_t>(c, D) : pick_wide<half_t>(c, D); }

}  // namespace tfk
