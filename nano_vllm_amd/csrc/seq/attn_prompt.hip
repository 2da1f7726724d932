// Windowed attention for steps of prompts: the instantiations without pooled blocks (attn_prompt.h).
#include "attn_prompt.h"

int window_attn_prompt(const WindowAttnArgs& a, hipStream_t stream) {
  return a.d == 128 ? launch_prompt<128, 128, 4, false>(a, stream) : launch_prompt<256, 192, 8, false>(a, stream);
}
