// Windowed attention for steps of prompts: the instantiation with pooled blocks, capped scores and row factors (attn_prompt.h).
#include "attn_prompt.h"

int window_attn_prompt_extended(const WindowAttnArgs& a, hipStream_t stream) { return launch_prompt<128, 128, 4, true>(a, stream); }
