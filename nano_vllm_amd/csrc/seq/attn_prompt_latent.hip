// Windowed attention of latent rows for steps of prompts, the queries' product with W_uk in front of it in the same kernel (attn_prompt.h).
#include "attn_prompt.h"

int window_attn_prompt_latent(const WindowAttnArgs& a, hipStream_t stream) { return launch_prompt<256, 192, 8, false, true>(a, stream); }
