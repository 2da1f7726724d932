// Windowed attention of latent rows for steps of prompts, the queries' product with W_uk in front of it, the results' with W_uv behind it, in the same kernel (attn_prompt.h).
#include "attn_prompt.h"

int window_attn_prompt_latent(const WindowAttnArgs& a, hipStream_t stream) {
  return a.uv ? launch_prompt<256, 192, 8, false, 2>(a, stream) : launch_prompt<256, 192, 8, false, 1>(a, stream);
}
