// The recurrences of ssd_launch (recurrent.hip explains their forms) for steps of single tokens: what a decode step does per sequence and head is read a state of P x N
// 32-bit numbers, add one term, multiply by the query, write it back. Bound by memory.
//
// A workgroup of four wavefronts per (portion, head). A row of the state is N / 4 neighbouring lanes of four entries, so a wavefront reads and writes whole lines, and a lane
// asks for all its rows' pieces (16 of a 128 x 128 state) before anything else; the token's operands come straight from where they are, nothing goes through LDS.
// The sums over a row's lanes are taken for all rows at once: at each halving of the distance a lane gives half of its rows away, so 16 rows take
// 16 exchanges instead of 80. Steps come here whose longest portion is one token; should one be longer than the caller said, its tokens are walked one by one.
//
// MI355X, 64 sequences x 8 heads of 128 x 128 (34 MB read and written), constant decay: 16 us; 64 sequences x 64 heads of 64 x 128 (268 MB), state-space duality 44 us = 6.1 TB/s
// (the walk of recurrent.hip, a row spread over 16 entries per lane and the token's operands staged in LDS behind a barrier: 27 and 79).
#include "scan_chunk.h"

namespace {

template <typename T, int LN, int IT, int FORM>
__global__ __launch_bounds__(256) void scan_token_kernel(const ScanArgs a) {
  constexpr int N = LN * 4, STEP = 256 / LN, PY = STEP * IT;           // rows of a pass, rows that are outputs
  const int s = blockIdx.y, h = blockIdx.x, tid = threadIdx.x, sub = tid % LN, col = sub * 4, row0 = tid / LN;
  const int64_t q0 = a.cu_q[s], q1 = a.cu_q[s + 1];
  if (q1 <= q0) return;
  const int64_t at = (int64_t)a.slot[s] * a.heads + h;
  const bool fresh = a.ctx0[s] == 0, norm = FORM == 2 && row0 == 0;    // form 2: the first row's lanes keep the normaliser's as well
  float* Sh = a.S + at * a.P * N + col;
  float st[IT][4], sn[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < IT; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) st[i][e] = 0.f;
  if (!fresh) {
#pragma unroll
    for (int i = 0; i < IT; ++i) ldv<4>(Sh + (int64_t)(row0 + i * STEP) * N, st[i]);
    if (norm) ldv<4>(Sh + (int64_t)PY * N, sn);
  }
  const T* proj = (const T*)a.proj;
  const int inner = a.heads * PY, grp = h / (a.heads / a.G);
  const int64_t width = inner + 2 * a.G * N;
  float A = 0.f, D = 0.f, dtb = 0.f, bi = 0.f, bf = 0.f, m = 0.f;
  if (FORM == 0) A = -expf(ldf((const T*)a.A_log + h)), D = ldf((const T*)a.D + h), dtb = ldf((const T*)a.dt_bias + h);
  if (FORM == 2) {
    bi = ldf((const T*)a.i_bias + h), bf = ldf((const T*)a.f_bias + h);
    if (!fresh) m = a.M[at];
    __syncthreads();                                // (everybody has read it before one thread writes the new one)
  }
#pragma unroll 1
  for (int64_t t = q0; t < q1; ++t) {
    float k[4], q[4], x[IT], decay = 1.f, step = 1.f;
    const T* row = proj + t * a.proj_stride;
    if (FORM == 0) {
      const float* src = a.xbc + t * width;
      ldv<4>(src + inner + grp * N + col, k);
      ldv<4>(src + inner + (a.G + grp) * N + col, q);
#pragma unroll
      for (int i = 0; i < IT; ++i) x[i] = src[h * PY + row0 + i * STEP];
      step = softplusf_(ldf(row + a.dt_col + h) + dtb);
      decay = expf(A * step);
    } else {
      ldv<4>(row + a.b_col + grp * N + col, k);
      ldv<4>(row + a.c_col + grp * N + col, q);
#pragma unroll
      for (int i = 0; i < IT; ++i) x[i] = ldf(row + a.x_col + h * PY + row0 + i * STEP);
      if (FORM == 1) {
        decay = a.decay[h];
#pragma unroll
        for (int e = 0; e < 4; ++e) k[e] = siluf_(k[e]), q[e] = siluf_(q[e]);
#pragma unroll
        for (int i = 0; i < IT; ++i) x[i] = siluf_(x[i]);
      } else {
        const float zc = a.cap * tanhf((ldf(row + a.f_col + h) + bf) / a.cap);
        const float gi = a.cap * tanhf((ldf(row + a.i_col + h) + bi) / a.cap), gf = fminf(zc, 0.f) - log1pf(expf(-fabsf(zc)));
        const float mn = fmaxf(gf + m, gi);
        step = expf(gi - mn), decay = expf(gf + m - mn);
        m = mn;
#pragma unroll
        for (int e = 0; e < 4; ++e) q[e] *= a.c_scale;
      }
    }
    float part[IT];
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const float dx = step * x[i];
      part[i] = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        st[i][e] = decay * st[i][e] + k[e] * dx;
        part[i] += st[i][e] * q[e];
      }
    }
    if (FORM == 2) {
      float acc = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sn[e] = decay * sn[e] + k[e] * step;
        acc += sn[e] * q[e];
      }
#pragma unroll
      for (int o = LN / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
      if (tid == 0) a.den[t * a.heads + h] = fmaxf(fabsf(acc), expf(-m)) + 1e-6f;
    }
    int mine = 0;                                   // the row (of IT) that this lane's sum is in the end
#pragma unroll
    for (int o = LN / 2, left = IT; o > 0; o >>= 1) {
      const bool up = (sub & o) != 0;
      if (left > 1) {
        left >>= 1;
#pragma unroll
        for (int j = 0; j < IT / 2; ++j)
          if (j < left) {
            const float give = up ? part[j] : part[j + left], keep = up ? part[j + left] : part[j];
            part[j] = keep + __shfl_xor(give, o, 64);
          }
        mine += up ? left : 0;
      } else {
        part[0] += __shfl_xor(part[0], o, 64);
      }
    }
    if (sub % (LN / IT) == 0) {
      const int r = row0 + mine * STEP;
      float out = part[0];
      if (FORM == 0) out += D * a.xbc[t * width + h * PY + r];
      a.y[t * inner + h * PY + r] = out;
    }
  }
#pragma unroll
  for (int i = 0; i < IT; ++i) stv<4>(Sh + (int64_t)(row0 + i * STEP) * N, st[i]);
  if (norm) stv<4>(Sh + (int64_t)PY * N, sn);
  if (FORM == 2 && tid == 0) a.M[at] = m;
}

template <typename T, int LN, int IT>
void launch_token(const ScanArgs& a, int nseq, hipStream_t st) {
  const dim3 grid(a.heads, (unsigned)nseq), block(256);
  if (a.form == 0) scan_token_kernel<T, LN, IT, 0><<<grid, block, 0, st>>>(a);
  else if (a.form == 1) scan_token_kernel<T, LN, IT, 1><<<grid, block, 0, st>>>(a);
  else scan_token_kernel<T, LN, IT, 2><<<grid, block, 0, st>>>(a);
}

}  // namespace

bool scan_token_fits(const ScanArgs& a, int dtype) {
  const int rows = a.form == 2 ? a.P - 1 : a.P;
  if (!((a.N == 64 && (rows == 32 || rows == 64 || rows == 128)) || (a.N == 128 && (rows == 32 || rows == 64 || rows == 128)))) return false;
  if ((uintptr_t)a.S % 16) return false;
  if (a.form == 0) return (uintptr_t)a.xbc % 16 == 0;
  const int size = dtype == NVS_BF16 ? 2 : 4;
  return ((a.b_col | a.c_col | a.proj_stride) & 3) == 0 && (uintptr_t)a.proj % (4 * size) == 0;
}

int scan_token_launch(const ScanArgs& a, int dtype, int nseq, void* stream) {
  const int rows = a.form == 2 ? a.P - 1 : a.P;
  hipStream_t st = (hipStream_t)stream;
  NVS_DISPATCH(dtype, {
    if (a.N == 64) {
      if (rows == 32) launch_token<T, 16, 2>(a, nseq, st);
      else if (rows == 64) launch_token<T, 16, 4>(a, nseq, st);
      else launch_token<T, 16, 8>(a, nseq, st);
    } else {
      if (rows == 32) launch_token<T, 32, 4>(a, nseq, st);
      else if (rows == 64) launch_token<T, 32, 8>(a, nseq, st);
      else launch_token<T, 32, 16>(a, nseq, st);
    }
  });
  return nvs_check_launch("recurrence of single tokens");
}
