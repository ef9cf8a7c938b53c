// Flash-attention instances for head dimension 128.
#include "flash_attention.hpp"

int tfk::run_attention_d128(const AttentionCall& c) { return launch<128>(c); }
