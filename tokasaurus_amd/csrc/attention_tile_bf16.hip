// Paged attention in 32-bit arithmetic on the matrix cores: the kernels for bfloat16 storage (attention_tile_f32.h).
#include "attention_tile_f32.h"

void attention_tile_launch_bf16(const AttentionTileCall& a) { at_launch_sizes<bf16_t>(a); }
