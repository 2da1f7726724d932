// The recurrences of nvs_ssd_scan, nvs_decay_scan and nvs_gated_memory_scan in chunks of 16 tokens on the matrix cores
// (scan_chunk.hip); recurrent.hip decides between them and the walk over single tokens.
#pragma once
#include "seq_common.h"

struct ScanArgs {
  int form;                          // 0 state-space duality, 1 constant decay, 2 exponential gates (recurrent.hip explains them)
  const float* xbc;                  // form 0: x | B | C, 32-bit
  const void* proj;                  // `dtype`
  int64_t proj_stride, dt_col, x_col, b_col, c_col, i_col, f_col;
  const float* decay;
  const void *dt_bias, *A_log, *D, *i_bias, *f_bias;
  int heads, P, N, G;                // P: state rows, form 2's normaliser included
  const int32_t *cu_q, *ctx0, *slot;
  float *S, *M, *y, *den, *ws;
  float cap, c_scale;
  int seg_len, nseg;
  int by_length;                     // portions longest first (2 to 64 of them)
};

// segments for the chunk kernel (seg_len 0: none)
void scan_chunk_plan(int heads, int P, int nseq, int64_t max_q, int* seg_len, int* nseg);
// whether sizes and addresses suit the chunk kernel
bool scan_chunk_fits(const ScanArgs& a, int dtype);
int scan_chunk_launch(const ScanArgs& a, int dtype, int nseq, void* stream);
// the same for steps of single tokens (scan_token.hip)
bool scan_token_fits(const ScanArgs& a, int dtype);
int scan_token_launch(const ScanArgs& a, int dtype, int nseq, void* stream);
