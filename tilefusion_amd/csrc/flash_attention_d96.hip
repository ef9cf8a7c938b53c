// Flash-attention instances for head dimension 96.
#include "flash_attention.hpp"

int tfk::run_attention_d96(const AttentionCall& c) { return launch<96>(c); }
