// Flash-attention instances for head dimension 64.
#include "flash_attention.hpp"

int tfk::run_attention_d64(const AttentionCall& c) { return launch<64>(c); }
