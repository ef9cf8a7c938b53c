// Flash-attention instances for head dimensions 104 to 120 (multiples of 8).
#include "flash_attention.hpp"

int tfk::run_attention_below128(const AttentionCall& c) { return launch_tail<128>(c); }
