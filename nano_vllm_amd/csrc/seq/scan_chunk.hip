// The matrix-state recurrences of recurrent.hip for portions of many tokens: chunks of 16 tokens as small 32-bit matrix products.
#include "scan_chunk.h"
#include "f32_tiles.h"
#include <type_traits>

namespace {

// Within a chunk, with L_i the logarithm of the decay from the chunk's start to behind token i and w_j the step of token j,
//   y_i = exp(L_i) S C_i + sum_{j <= i} exp(L_i - L_j) w_j (C_i . B_j) x_j,     S <- exp(L_15) S + sum_j exp(L_15 - L_j) w_j x_j B_j^T,
// so a chunk is three products: C S^T (16 x N x P), (C B^T, masked and weighted) x (16 x N x 16 and 16 x 16 x P) and the outer
// products (P x 16 x N). All on v_mfma_f32_16x16x4_f32, whose products and sums are 32-bit ones. The exponents are differences of
// 64-bit sums of exponents above -200, so a pair's weight is as exact as its own exponent however strongly the chunk decays as a whole. Form 2 has
// exp(F_i - F_j + i_j - m_i) in place of exp(L_i - L_j) w_j and exp(F_i + m_before - m_i) in place of exp(L_i), m the running maximum.
// A short last chunk is filled with tokens that change nothing (B = C = x = 0, no decay, no step).
//
// A workgroup takes NW * 16 rows p of one (portion, head)'s state, a wavefront 16 of them: its N / 16 accumulator tiles hold
// S[n = 16 t + 4 (lane / 16) + r][p = lane % 16], which IS the operand layout of C S^T if the four tokens' entries of a product
// step are taken as n = 16 t + 4 (lane / 16) + r, r the step: the state never leaves its registers. The same trick feeds C B^T,
// computed transposed, to the next product. C B^T is shared: each wavefront sums N / NW of the columns, one chunk ahead, and the
// parts meet in LDS. So do the weights of a chunk, computed a pair (i, j) per thread one chunk ahead. One barrier per chunk: B and
// C go through three LDS images (read by this chunk, read ahead, being written), the loads of the chunk after those are in flight.
//
// What bounds it: the 32-bit matrix rate, 76 instructions of 32 cycles per wavefront and chunk at N = 128 (54 % of all cycles busy
// with them over 32 portions of 1,000 tokens, 64 heads of 64 x 128), and with few workgroups the chain through a chunk, 2.3 us a
// chunk alone on a compute unit. Measured against the walk over single tokens, nine portions of 33 to 4,096 tokens, 13,550 in all:
// 64 heads of 64 x 128 (form 0) 5,200 -> 650 us, 32 heads of 128 x 128 (form 1) 3,470 -> 700, 8 heads of 128 x 128 (form 2)
// 1,600 -> 250; one portion of 16,384: 3,650 -> 860, 3,690 -> 900, 1,690 -> 245. Errors against 64 bits, first nine portions,
// outputs / states: 1.3e-7 / 1.0e-7 -> 1.2e-7 / 0.9e-7, 1.9e-7 / 5.0e-7 -> 1.3e-7 / 3.7e-7, 2.0e-7 / 1.9e-7 -> 1.8e-7 / 1.4e-7.
// Ragged portions are taken longest first (recurrent.hip says when), so that they end together: 12 of 175 to 1,400 tokens, 64 heads, forms 0, 1, 2 412 712 820 -> 358 569 658 us.
// Form 1's SiLU, a third of its vector instructions, which no 32-bit matrix instruction runs beside (49 + 51 % of all cycles over 16 portions of 512), is the short one of
// seq_common.h, with the same errors (the same portions 758 -> 712 us, 32 of 100 tokens 227 -> 215).
constexpr int CT = 16;                              // tokens of a chunk
constexpr int WST = 20;                             // row stride of the 16 x 16 weights in LDS
constexpr int SB = 4;                               // chunks whose weights are computed together: a token per lane

// inclusive sum / running maximum over the 16 lanes of a row, in 64 bits
template <int CTRL>
__device__ __forceinline__ double row_shifted(double v, double fill) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v), f = __builtin_bit_cast(uint64_t, fill);
  const uint32_t lo = __builtin_amdgcn_update_dpp((int)(uint32_t)f, (int)(uint32_t)b, CTRL, 0xf, 0xf, false);
  const uint32_t hi = __builtin_amdgcn_update_dpp((int)(uint32_t)(f >> 32), (int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ double row_running_sum(double v) {
  v += row_shifted<0x111>(v, 0.);                   // row_shr:1, 2, 4, 8
  v += row_shifted<0x112>(v, 0.);
  v += row_shifted<0x114>(v, 0.);
  v += row_shifted<0x118>(v, 0.);
  return v;
}
__device__ __forceinline__ double row_running_max(double v) {
  v = fmax(v, row_shifted<0x111>(v, v));
  v = fmax(v, row_shifted<0x112>(v, v));
  v = fmax(v, row_shifted<0x114>(v, v));
  v = fmax(v, row_shifted<0x118>(v, v));
  return v;
}
// e^v, with what rounding the exponent to 32 bits leaves
__device__ __forceinline__ float exp_(double v) {
  const float c = (float)fmax(v, -1e30), e = expf(c);
  return v < -1e30 ? 0.f : fmaf(e, (float)(v - (double)c), e);
}
__device__ __forceinline__ double lane_of(double v, int lane) { return __shfl(v, lane, 64); }

// MODE as in recurrent.hip: 0 the whole portion, 1 a segment's local state only, 2 a segment's outputs from the state before it,
// which scan_states_kernel puts in the place of the local states in between.
// BY_LENGTH: of 2 to 64 portions the longest is the first.
template <typename T, int NT, int NW, int FORM, int MODE, bool BY_LENGTH>
__global__ __launch_bounds__(NW * 64, NW / 2) void scan_chunk_kernel(const ScanArgs a) {
  constexpr int N = 16 * NT, LD = N + 4, NTH = NW * 64;
  typedef typename std::conditional<FORM == 0, float, T>::type TB;            // what B and C are stored as
  constexpr int VE = 16 / sizeof(TB), ROWU = N / VE, UNITS = (MODE == 1 ? 1 : 2) * CT * ROWU, UP = (UNITS + NTH - 1) / NTH;
  constexpr int KT = NT >= NW ? NT / NW : 1, KW = NT / KT;   // state tiles whose part of C B^T a wavefront sums; wavefronts that do
  __shared__ __attribute__((aligned(16))) float bc[3][2][CT][LD];
  __shared__ __attribute__((aligned(16))) float part[2][KW][64][4];
  __shared__ __attribute__((aligned(16))) float wt[2][FORM == 1 ? 1 : SB][CT][WST];    // (form 1: once for all, what rounding left in [1])
  __shared__ __attribute__((aligned(16))) float win[2][FORM == 1 ? 1 : SB][2][CT];      // decay from the chunk's start, and what rounding left of it; form 2: exp(-m)
  __shared__ __attribute__((aligned(16))) float nq[FORM == 2 ? 2 : 1][KW][CT];     // form 2: the parts of n . q
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, l16 = lane & 15, g = lane >> 4;
  const int h = blockIdx.x, seg = blockIdx.z % a.nseg, blk = blockIdx.z / a.nseg;
  const int heads = a.heads, P = a.P;
  PortionSpan span;
  if constexpr (BY_LENGTH) span = portion_by_length(a.cu_q, gridDim.y, blockIdx.y);
  const int s = BY_LENGTH ? span.s : blockIdx.y;
  const int64_t t0 = BY_LENGTH ? span.t0 : a.cu_q[s], t1 = BY_LENGTH ? span.t1 : a.cu_q[s + 1];
  const int64_t q0 = MODE == 0 ? t0 : t0 + (int64_t)seg * a.seg_len;
  const int64_t q1 = MODE == 0 ? t1 : (q0 + a.seg_len < t1 ? q0 + a.seg_len : t1);
  if (q1 <= q0) return;
  const bool last = q1 == t1, fresh = a.ctx0[s] == 0;
  if (MODE == 1 && last && seg > 0) return;         // nobody starts from the last segment's state
  const int pb = (blk * NW + w) * 16, p = pb + l16;
  const int Py = FORM == 2 ? P - 1 : P;             // rows that are outputs
  const bool mine = p < Py;                         // (a lane without a row repeats the last one and stores nothing)
  const bool sums = KW == NW || w < KW;             // form 2: and that part of the normaliser n
  const int64_t pair = (int64_t)s * heads + h;
  const T* proj = (const T*)a.proj;

  // ---- the state this workgroup starts from
  constexpr int WD = FORM == 2 ? 3 : 1;
  float* wst = a.ws + pair * (a.nseg + 1) * P * N + (int64_t)p * N + 4 * g;
  float* wdec = a.ws + (int64_t)gridDim.y * heads * (a.nseg + 1) * P * N + pair * (a.nseg + 1) * WD;
  float* Sh = a.S + (((int64_t)a.slot[s] * heads + h) * P + p) * N + 4 * g;
  const int64_t nrow = (int64_t)(Py - p) * N + 16 * w * KT;                  // from row p to this wavefront's part of n
  f32x4_t st[NT], nst[KT];                          // n as 16 equal columns
  float mrun = 0.f;
  double fsum = 0.;
  double dprod = 1.;
#pragma unroll
  for (int t = 0; t < NT; ++t) st[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < KT; ++t) nst[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if (FORM == 2) {
    if (!fresh) mrun = a.M[(int64_t)a.slot[s] * heads + h];
    if (MODE == 2) mrun = seg ? wdec[seg * WD + 2] : wdec[1];
  }
  if (MODE == 2) {                                  // the state before this segment
    const float* src = wst + (int64_t)seg * P * N;
    if (mine) {
#pragma unroll
      for (int t = 0; t < NT; ++t) st[t] = *(const f32x4_t*)(src + 16 * t);
    }
    if (FORM == 2 && sums) {
#pragma unroll
      for (int t = 0; t < KT; ++t) nst[t] = *(const f32x4_t*)(src + nrow + 16 * t);
    }
  } else if (!fresh && (MODE == 0 || seg == 0)) {
    if (mine) {
#pragma unroll
      for (int t = 0; t < NT; ++t) st[t] = *(const f32x4_t*)(Sh + 16 * t);
    }
    if (FORM == 2 && sums) {
#pragma unroll
      for (int t = 0; t < KT; ++t) nst[t] = *(const f32x4_t*)(Sh + nrow + 16 * t);
    }
  }
  // (a lane of each row of 16 stores n, whose columns are equal)
  auto store_state = [&](float* dst) {
    if (mine) {
#pragma unroll
      for (int t = 0; t < NT; ++t) *(f32x4_t*)(dst + 16 * t) = st[t];
    }
    if (FORM == 2 && sums && l16 == 0) {
#pragma unroll
      for (int t = 0; t < KT; ++t) *(f32x4_t*)(dst + nrow + 16 * t) = nst[t];
    }
  };
  if (MODE == 1) {                                  // the portion's starting state, for mode 2; a segment by itself starts from none
    if (seg == 0) {
      store_state(wst);
      if (FORM == 2 && tid == 0) wdec[1] = mrun;
#pragma unroll
      for (int t = 0; t < NT; ++t) st[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < KT; ++t) nst[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    if (last) return;                               // (a portion of one segment: only its starting state was needed)
    if (FORM == 2) mrun = -1e30f;
  }

  // ---- operands
  const int inner = heads * P, grp = h / (heads / a.G);
  const int64_t brow = FORM == 0 ? inner + 2 * a.G * N : a.proj_stride;
  const TB* Bp = FORM == 0 ? (const TB*)a.xbc + inner + grp * N : (const TB*)a.proj + a.b_col + (int64_t)h * N;
  const TB* Cp = FORM == 0 ? (const TB*)a.xbc + inner + (a.G + grp) * N : (const TB*)a.proj + a.c_col + (int64_t)h * N;
  const TB* Xp = FORM == 0 ? (const TB*)a.xbc + h * P : (const TB*)a.proj + a.x_col + (int64_t)h * Py;
  float A = 0.f, Dh = 0.f, dtb = 0.f, bi = 0.f, bf = 0.f;
  if (FORM == 0) A = -expf(ldf((const T*)a.A_log + h)), Dh = ldf((const T*)a.D + h), dtb = ldf((const T*)a.dt_bias + h);
  if (FORM == 2) bi = ldf((const T*)a.i_bias + h), bf = ldf((const T*)a.f_bias + h);
  if (FORM == 1 && tid < 256) {                     // the weights are powers of one number: [i][j] holds power i - j
    const double d = a.decay[h];
    const int i = tid >> 4, n = i - l16;
    double v = 1.;
    for (int k = 0; k < n; ++k) v *= d;
    if (n < 0) v = 0.;
    wt[0][0][i][l16] = (float)v, wt[1][0][i][l16] = (float)(v - (double)(float)v);
    if (l16 == 0) {
      v *= d;
      win[0][0][0][i] = (float)v, win[0][0][1][i] = (float)(v - (double)(float)v);
    }
  }

  typedef __attribute__((ext_vector_type(4))) uint32_t raw_t;
  raw_t raw[UP];                                    // B and C of the chunk after the two in LDS
  TB xraw[4];                                       // x of the next chunk, tokens 4 g + 0..3
  T g0 = (T)0.f, g1 = (T)0.f;                                        // gates of the chunk whose weights are computed next: token l16
  // (tokens behind the portion's end: its last token is read, and zeros are staged)
  const int pc = mine ? p : Py - 1;
  auto row_of = [&](int64_t t) { return t < q1 ? t : q1 - 1; };
  auto load_bc = [&](int64_t tb) {
#pragma unroll
    for (int u = 0; u < UP; ++u) {
      const int e = tid + u * NTH, which = e / (CT * ROWU), k = e / ROWU % CT, c = e % ROWU;
      if (UNITS % NTH == 0 || e < UNITS) raw[u] = *(const raw_t*)((which ? Cp : Bp) + row_of(tb + k) * brow + c * VE);
    }
  };
  auto stage_bc = [&](int buf, int64_t tb) {
#pragma unroll
    for (int u = 0; u < UP; ++u) {
      const int e = tid + u * NTH, which = e / (CT * ROWU), k = e / ROWU % CT, c = e % ROWU;
      if (UNITS % NTH == 0 || e < UNITS) {
        float* dst = &bc[buf][which][k][c * VE];
        const bool in = tb + k < q1;
        float v[VE];
#pragma unroll
        for (int i = 0; i < VE; ++i) {
          const uint32_t word = raw[u][i * 4 / VE];
          const uint32_t bits = VE == 4 ? word : (i % 2 ? word & 0xffff0000u : word << 16);
          v[i] = __builtin_bit_cast(float, bits);
          if (FORM == 1) v[i] = silu_hw(v[i]);
          if (FORM == 2 && which) v[i] *= a.c_scale;
          if (!in) v[i] = 0.f;
        }
#pragma unroll
        for (int i = 0; i < VE; i += 4) *(float4*)(dst + i) = make_float4(v[i], v[i + 1], v[i + 2], v[i + 3]);
      }
    }
  };
  auto load_x = [&](int64_t tb) {
#pragma unroll
    for (int r = 0; r < 4; ++r) xraw[r] = Xp[row_of(tb + 4 * g + r) * brow + pc];
  };
  auto load_gates = [&](int64_t tb) {
    if (FORM == 1 || tid >= 256) return;
    g0 = proj[row_of(tb + lane) * a.proj_stride + (FORM == 0 ? a.dt_col : a.i_col) + h];
    if (FORM == 2) g1 = proj[row_of(tb + lane) * a.proj_stride + a.f_col + h];
  };
  // the weights of the four chunks from tb on, in wt / win [buf]: each of the first four wavefronts has all their tokens, one per
  // lane, and writes one chunk's weights, lane (4 g + e, j = l16)
  auto weights = [&](int64_t tb, int buf) {
    if (FORM == 1 || tid >= 256 || tb >= q1) return;
    const bool valid = tb + lane < q1;
    float wij[4], wi, em = 0.f;
    if (FORM == 0) {
      const float dt = valid ? softplusf_(ldf(&g0) + dtb) : 0.f;
      // (below -200 a decay is 0 whatever follows; the sums stay small enough to tell the exponents of the tokens behind it apart, and finite)
      const double l = valid ? (double)A * (double)dt : 0., L = row_running_sum(l < -200. ? -200. : l), Lj = lane_of(L, 16 * w + l16);
      const float dj = __shfl(dt, 16 * w + l16, 64);
#pragma unroll
      for (int e = 0; e < 4; ++e) wij[e] = exp_(lane_of(L, 16 * w + 4 * g + e) - Lj) * dj;
      wi = exp_(Lj);
    } else {
      const float zc = a.cap * tanhf((ldf(&g1) + bf) / a.cap);
      const double f = valid ? (double)(fminf(zc, 0.f) - log1pf(expf(-fabsf(zc)))) : 0.;          // log sigmoid
      const double ig = valid ? (double)(a.cap * tanhf((ldf(&g0) + bi) / a.cap)) : -1e300;
      const double F = row_running_sum(f), v = ig - F, vm = row_running_max(v);
      float before = mrun;                          // the maximum before this lane's chunk
#pragma unroll
      for (int k = 0; k < SB; ++k) {
        const double Fk = lane_of(F, 16 * k + 15);
        if (g == k) before = mrun;
        fsum += Fk;
        mrun = (float)(Fk + fmax(lane_of(vm, 16 * k + 15), (double)mrun));
      }
      const float m = (float)(F + fmax(vm, (double)before));
      const double vj = lane_of(v, 16 * w + l16);
      const float mj = __shfl(m, 16 * w + l16, 64);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        wij[e] = exp_(lane_of(F, 16 * w + 4 * g + e) + vj - (double)__shfl(m, 16 * w + 4 * g + e, 64));
      wi = exp_(lane_of(F, 16 * w + l16) + (double)__shfl(before, 16 * w, 64) - (double)mj);
      em = expf(-mj);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) wt[buf][w][4 * g + e][l16] = l16 <= 4 * g + e ? wij[e] : 0.f;
    if (g == 0) {
      win[buf][w][0][l16] = wi;
      if (FORM == 2) win[buf][w][1][l16] = em;
    }
  };
  // this wavefront's part of B C^T (rows j, columns i)
  auto couple = [&](int src, int buf) {
    if (MODE == 1 || !sums) return;
    f32x4_t c[4] = {};
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      const int n = 16 * (w * KT + t) + 4 * g;
      const f32x4_t bv = *(const f32x4_t*)&bc[src][0][l16][n], cv = *(const f32x4_t*)&bc[src][1][l16][n];
#pragma unroll
      for (int r = 0; r < 4; ++r) c[r] = mfma4(bv[r], cv[r], c[r]);
    }
    *(f32x4_t*)part[buf][w][lane] = (c[0] + c[1]) + (c[2] + c[3]);
  };
  // form 2, the first wavefront: token l16's share of n . q from inside the chunk, its decay and exp(-m); n . q is complete a
  // barrier later
  float own = 0.f, own_in = 0.f, own_m = 0.f;
  auto divisors = [&](int64_t tb, int buf) {
    if (FORM != 2 || MODE == 1 || tid >= CT || tb < q0 || tb + tid >= q1) return;
    float v = 0.f;
#pragma unroll
    for (int k = 0; k < KW; ++k) v += nq[buf][k][tid];
    a.den[(tb + tid) * heads + h] = fmaxf(fabsf(v * own_in + own), own_m) + 1e-6f;
  };

  load_bc(q0);
  load_gates(q0);
  load_x(q0);
  stage_bc(0, q0);
  load_bc(q0 + CT);
  weights(q0, 0);
  load_gates(q0 + SB * CT);
  stage_bc(1, q0 + CT);
  load_bc(q0 + 2 * CT);
  lds_barrier();
  couple(0, 0);
  int b3 = 0, b2 = 0, ws = 0, wk = 0;               // this chunk's images, parts and weights
  for (int64_t tb = q0; tb < q1; tb += CT) {
    lds_barrier();
    divisors(tb - CT, b2 ^ 1);
    const int n3 = b3 == 2 ? 0 : b3 + 1, w3 = n3 == 2 ? 0 : n3 + 1;
    // (form 1: a short last chunk is behind its last token with that token's weights; elsewhere the tokens that fill it see to that)
    const int le = FORM == 1 && q1 - tb < CT ? (int)(q1 - tb) - 1 : CT - 1;
    const float gc = win[ws][wk][0][le], gl = FORM == 1 ? win[ws][wk][1][le] : 0.f;
    const f32x4_t we = *(const f32x4_t*)&wt[ws][wk][le][4 * g];              // weights in the state behind the chunk
    if (MODE == 1) dprod *= (double)gc + (double)gl;
    constexpr bool early = NW == 4;                 // (eight wavefronts have half the registers each)
    f32x4_t cv[NT];
    if (MODE != 1 && early) {
#pragma unroll
      for (int t = 0; t < NT; ++t) cv[t] = *(const f32x4_t*)&bc[b3][1][l16][16 * t + 4 * g];
    }
    float xv[4], xw[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      xv[r] = ldf(&xraw[r]);
      if (FORM == 1) xv[r] = silu_hw(xv[r]);
      if (tb + 4 * g + r >= q1) xv[r] = 0.f;
      xw[r] = xv[r] * we[r];
    }
    load_x(tb + CT);
    stage_bc(w3, tb + 2 * CT);
    load_bc(tb + 3 * CT);
    couple(n3, b2 ^ 1);
    // C S^T in several short sums, so that few roundings follow one another on a large value: four, and where there are registers
    // four per half of the state
    constexpr bool halves = FORM == 1 || NW == 4;
    f32x4_t y[4] = {}, yo = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if (MODE != 1) {
        if (!early) cv[t] = *(const f32x4_t*)&bc[b3][1][l16][16 * t + 4 * g];
#pragma unroll
        for (int r = 0; r < 4; ++r) y[r] = mfma4(cv[t][r], st[t][r], y[r]);
        if (halves && t == NT / 2 - 1) {
          yo = (y[0] + y[1]) + (y[2] + y[3]);
#pragma unroll
          for (int r = 0; r < 4; ++r) y[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) st[t][r] = FORM == 1 ? fmaf(st[t][r], gc, st[t][r] * gl) : st[t][r] * gc;
#pragma unroll
      for (int r = 0; r < 4; ++r) st[t] = mfma4(bc[b3][0][4 * g + r][16 * t + l16], xw[r], st[t]);
    }
    if (FORM == 2 && sums) {                        // n, whose value is the constant 1
      f32x4_t q = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < KT; ++t) {
        const int n = 16 * (w * KT + t);
        if (MODE != 1) {
          const f32x4_t c = *(const f32x4_t*)&bc[b3][1][l16][n + 4 * g];
#pragma unroll
          for (int r = 0; r < 4; ++r) q = mfma4(c[r], nst[t][r], q);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) nst[t][r] *= gc;
#pragma unroll
        for (int r = 0; r < 4; ++r) nst[t] = mfma4(bc[b3][0][4 * g + r][n + l16], we[r], nst[t]);
      }
      if (MODE != 1 && l16 == 0) *(f32x4_t*)&nq[b2][w][4 * g] = q;
    }
    if (MODE != 1) {
      f32x4_t pt[KW];
#pragma unroll
      for (int k = 0; k < KW; ++k) pt[k] = *(const f32x4_t*)part[b2][k][lane];
#pragma unroll
      for (int o = 1; o < KW; o *= 2)
#pragma unroll
        for (int k = 0; k < KW; k += 2 * o) pt[k] += pt[k + o];
      f32x4_t m = pt[0];
      yo += (y[0] + y[1]) + (y[2] + y[3]);
      const f32x4_t wv = *(const f32x4_t*)&wt[ws][wk][l16][4 * g], wi = *(const f32x4_t*)&win[ws][wk][0][4 * g];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (FORM == 1) {
          yo[r] = fmaf(yo[r], wi[r], yo[r] * win[0][0][1][4 * g + r]);
          m[r] = fmaf(m[r], wv[r], m[r] * wt[1][0][l16][4 * g + r]);
        } else {
          yo[r] *= wi[r], m[r] *= wv[r];
        }
        if (4 * g + r > l16) m[r] = 0.f;
      }
      // x of every token meets every output of the chunk in this product, above the diagonal with a weight of 0: a value that is not finite
      // (rare: or a sum of four that overflows) goes to the outputs behind it alone, token by token
      const bool odd = !((fabsf(xv[0]) + fabsf(xv[1])) + (fabsf(xv[2]) + fabsf(xv[3])) < INFINITY);
      if (__ballot(odd) == 0ull) {
#pragma unroll
        for (int r = 0; r < 4; ++r) yo = mfma4(m[r], xv[r], yo);
      } else {
#pragma unroll 1
        for (int j0 = 0; j0 < CT; j0 += 4) {        // m[i][j] is in lane i + 16 (j / 4), x[j][p] in lane p + 16 (j / 4), entry j % 4
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const float xj = __shfl(xv[k], 4 * j0 + l16, 64);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float mij = __shfl(m[k], 4 * j0 + 4 * g + r, 64);
              if (j0 + k <= 4 * g + r) yo[r] = fmaf(mij, xj, yo[r]);
            }
          }
        }
      }
      if (FORM == 2 && w == 0) {
        own = (m[0] + m[1]) + (m[2] + m[3]);
        own += __shfl_xor(own, 16, 64);
        own += __shfl_xor(own, 32, 64);
        own_in = win[ws][wk][0][l16], own_m = win[ws][wk][1][l16];
      }
      float* yp = a.y + (tb + 4 * g) * heads * Py + h * Py + p;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (mine && tb + 4 * g + r < q1) yp[r * heads * Py] = FORM == 0 ? yo[r] + Dh * xv[r] : yo[r];
    }
    if (FORM == 1) {
    } else if (++wk == SB) {
      wk = 0, ws ^= 1;
    } else if (wk == SB - 1) {
      weights(tb + 2 * CT, ws ^ 1);
      load_gates(tb + (2 + SB) * CT);
    }
    b3 = n3, b2 ^= 1;
  }
  if (FORM == 2 && MODE != 1) {
    lds_barrier();
    divisors(q0 + (q1 - 1 - q0) / CT * CT, b2 ^ 1);
  }
  if (MODE == 1) {
    store_state(wst + (int64_t)(seg + 1) * P * N);
    if (blk == 0 && tid == 0) {
      if (FORM == 2) wdec[(seg + 1) * WD] = (float)fsum, wdec[(seg + 1) * WD + 1] = mrun;
      else wdec[seg + 1] = (float)dprod;
    }
  } else if (last) {
    store_state(Sh);
    if (FORM == 2 && tid == 0) a.M[(int64_t)a.slot[s] * heads + h] = mrun;
  }
}

// Between the passes: entry k + 1 of a (portion, head), segment k's local state, becomes the state behind that segment. Four state
// entries per thread; a chain of one multiplication and addition per segment, its loads four segments ahead.
template <bool GATES>
__global__ __launch_bounds__(256) void scan_states_kernel(float* __restrict__ ws, const int32_t* __restrict__ cu_q, int seg_len, int nseg,
                                                          int64_t PN) {
  const int h = blockIdx.y, s = blockIdx.z, heads = gridDim.y;
  const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4, pair = (int64_t)s * heads + h;
  const int ns = (int)((cu_q[s + 1] - cu_q[s] + seg_len - 1) / seg_len);
  if (e >= PN || ns < 2) return;
  constexpr int WD = GATES ? 3 : 1;
  float* st = ws + pair * (nseg + 1) * PN + e;
  float* wdec = ws + (int64_t)gridDim.z * heads * (nseg + 1) * PN + pair * (nseg + 1) * WD;
  f32x4_t v = *(const f32x4_t*)st;
  float m = GATES ? wdec[1] : 0.f;
  for (int k0 = 1; k0 < ns; k0 += 4) {
    f32x4_t l[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) l[k] = *(const f32x4_t*)(st + (k0 + k < ns ? k0 + k : ns - 1) * PN);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (k0 + k >= ns) break;
      float dk = wdec[(k0 + k) * WD], bk = 1.f;
      if (GATES) {
        const float ml = wdec[(k0 + k) * WD + 1], mn = fmaxf(m + dk, ml);
        dk = expf(m + dk - mn), bk = expf(ml - mn), m = mn;
        if (e == 0) wdec[(k0 + k) * WD + 2] = m;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = dk * v[r] + bk * l[k][r];
      *(f32x4_t*)(st + (k0 + k) * PN) = v;
    }
  }
}

int waves_of(const ScanArgs& a) { return (a.form == 2 ? a.P - 1 : a.P) > 64 ? 8 : 4; }

template <typename T, int NT, int NW, int FORM>
void launch_form(const ScanArgs& a, int nseq, hipStream_t stream) {
  const int blocks = ((FORM == 2 ? a.P - 1 : a.P) + NW * 16 - 1) / (NW * 16);
  const dim3 grid(a.heads, (unsigned)nseq, (unsigned)(blocks * a.nseg)), block(NW * 64);
  if (a.seg_len) {
    const int64_t PN = (int64_t)a.P * a.N;
    scan_chunk_kernel<T, NT, NW, FORM, 1, false><<<grid, block, 0, stream>>>(a);
    scan_states_kernel<FORM == 2><<<dim3((unsigned)((PN / 4 + 255) / 256), a.heads, (unsigned)nseq), dim3(256), 0, stream>>>(
        a.ws, a.cu_q, a.seg_len, a.nseg, PN);
    scan_chunk_kernel<T, NT, NW, FORM, 2, false><<<grid, block, 0, stream>>>(a);
  } else {
    a.by_length ? scan_chunk_kernel<T, NT, NW, FORM, 0, true><<<grid, block, 0, stream>>>(a) : scan_chunk_kernel<T, NT, NW, FORM, 0, false><<<grid, block, 0, stream>>>(a);
  }
}

template <typename T, int NT, int NW>
void launch_sized(const ScanArgs& a, int nseq, hipStream_t stream) {
  if (a.form == 0) launch_form<T, NT, NW, 0>(a, nseq, stream);
  else if (a.form == 1) launch_form<T, NT, NW, 1>(a, nseq, stream);
  else launch_form<T, NT, NW, 2>(a, nseq, stream);
}

}  // namespace

void scan_chunk_plan(int heads, int P, int nseq, int64_t max_q, int* seg_len, int* nseg) {
  *seg_len = 0;
  *nseg = 1;
  // Segments cost a second pass over B and x (about half a scan) and pay where a step waits for its longest portion. Measured, 128 x
  // 128 states: 288 workgroups over portions of 33 to 4,096 tokens 1,010 -> 700 us, 256 over 32 even portions of 1,000 tokens
  // 300 -> 400, 32 for one of 300 tokens 82 -> 69, 8 for one of 16,384 4,000 -> 245 (64 segments: more cost more in states than they
  // give); 576 workgroups of 64 x 128 over 33 to 4,096 tokens 650 -> 720.
  const int64_t groups = (int64_t)heads * nseq * (P > 129 ? (P + 127) / 128 : 1);      // workgroups (of four or eight wavefronts)
  if (groups >= 512 || max_q < (groups >= 256 ? 2048 : 256)) return;
  int64_t parts = (2048 + groups - 1) / groups;
  if (parts > 64) parts = 64;
  int64_t sl = (max_q / parts + 15) / 16 * 16;
  if (sl < 128) sl = 128;
  const int ns = (int)((max_q + sl - 1) / sl);
  if (ns < 2) return;
  *seg_len = (int)sl;
  *nseg = ns;
}

bool scan_chunk_fits(const ScanArgs& a, int dtype) {
  if (a.N != 64 && a.N != 128) return false;
  if (a.form == 2 && a.P > 129) return false;       // one workgroup keeps the maximum of a (portion, head)
  uintptr_t al = (uintptr_t)a.S | (uintptr_t)a.ws;
  if (a.form == 0) {
    if (a.heads * a.P % 4) return false;
    al |= (uintptr_t)a.xbc;
  } else {
    const int64_t e = dtype == NVS_BF16 ? 8 : 4;
    if (a.proj_stride % e || a.b_col % e || a.c_col % e) return false;
    al |= (uintptr_t)a.proj;
  }
  return al % 16 == 0;
}

int scan_chunk_launch(const ScanArgs& a, int dtype, int nseq, void* stream) {
#define NVS_SCAN_SIZED(NT)                                                                 \
  do {                                                                                     \
    if (waves_of(a) == 8) NVS_DISPATCH(dtype, launch_sized<T, NT, 8>(a, nseq, (hipStream_t)stream)); \
    else NVS_DISPATCH(dtype, launch_sized<T, NT, 4>(a, nseq, (hipStream_t)stream));        \
  } while (0)
  if (a.N == 128) NVS_SCAN_SIZED(8);
  else NVS_SCAN_SIZED(4);
#undef NVS_SCAN_SIZED
  return nvs_check_launch("the chunked scan");
}
