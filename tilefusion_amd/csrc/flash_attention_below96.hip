// Flash-attention instances for head dimensions 72 to 88 (multiples of 8).
#include "flash_attention.hpp"

int tfk::run_attention_below96(const AttentionCall& c) { return launch_tail<96>(c); }
