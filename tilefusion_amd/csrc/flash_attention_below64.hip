// Flash-attention instances for head dimensions 40 to 56 (multiples of 8).
#include "flash_attention.hpp"

int tfk::run_attention_below64(const AttentionCall& c) { return launch_tail<64>(c); }
