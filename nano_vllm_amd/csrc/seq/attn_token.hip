// Windowed attention over the paged cache for steps of single tokens (bf16, 128-wide heads or latent rows of 256 with values of 192; no pooled blocks).
//
// What bounds it: reading the keys and values that are seen, once (64 sequences of some 500 visible tokens, 8 kv heads of 128: 124 MB), and for few
// sequences how long one workgroup's chain is. attn_prompt.h's kernel lets all wavefronts share every tile of 64 keys, so a query's tiles come
// one after the other, 16 rounds of 3 us for a window of 1,024, and half of its wavefronts have no query. Here a workgroup has one token and up to 16
// query heads of a kv head (a column each of the 16-wide products), and its NW wavefronts take every NW-th tile of 32 keys, each with a place of its own in
// LDS that is refilled as soon as the operands are in registers: no barrier until the wavefronts' maxima, sums and outputs are put together.
//
// As everywhere here: S^T = K Q^T and O^T += V^T P^T, a lane owns one query (lane & 15). Row i of key block kb is key 8 (i >> 2) + 4 kb + (i & 3), so that the
// eight weights of a lane are eight consecutive keys, its operand of the second product as they are. Keys that are not visible weigh 0 and their
// values are taken as 0 (what a page holds there may not be finite).
//
// MI355X, attn_prompt.h's kernel (packed heads: attn_window_core.h's) and here, us: 64 sequences of 200 to 1,500 tokens, window 1,024, 32 heads over 8 kv heads 53 -> 36
// (5.5 TB/s), causal 67 -> 44; 16 heads over 8, one sequence of 100 / 1,000 / 30,000 tokens 16 -> 6.5, 33 -> 11, 565 -> 221, 256 sequences 212 -> 168;
// packed: 64 heads over one, 24 sequences of 2,500 92 -> 22, 16 over 2, 224 sequences 160 -> 110; latent rows, 16 heads, 1 / 64 / 192 sequences
// 62 -> 19, 91 -> 30, 200 -> 86. Four wavefronts instead of eight: 38, 46, 7, 15, 289, 163 in the same order.
#include "attn_window_core.h"

int window_attn_token(const WindowAttnArgs& a, hipStream_t stream);

namespace {

typedef __attribute__((address_space(3))) void lds_void_t;
typedef const __attribute__((address_space(1))) void global_void_t;

constexpr float LOG2E = 1.4426950408889634f, HIDDEN = -3e38f;

template <int D, int DV, int NW>
__global__ __launch_bounds__(64 * NW) void window_attn_token_kernel(const WindowAttnArgs A) {
  constexpr int KB = 32 * D * 2, VB = DV * 64, RING = KB + VB, KU = D / 8, KR = KB / 1024, VR = VB / 1024, DC = D / 32, DB = DV / 16;
  extern __shared__ __attribute__((aligned(128))) char lds[];          // rings; cos and sin [NW][D / 2]; maxima and sums [NW][16]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, lq = lane >> 4;
  const int hpg = A.H / A.G, per = (hpg + 15) / 16, g = blockIdx.y / per, h0 = g * hpg + blockIdx.y % per * 16;
  const int heads = (g + 1) * hpg - h0 < 16 ? (g + 1) * hpg - h0 : 16, h = h0 + (li < heads ? li : 0);
  const int64_t t = blockIdx.x;
  // what the queries need is requested before the tiles: the counter that tells what has landed counts in order
  const bf16_t* qp = (const bf16_t*)A.q + t * A.q_stride + (int64_t)h * D + 8 * lq;
  const bf16_t* qw = A.qnorm ? (const bf16_t*)A.qnorm + (A.q_row ? (int64_t)h * D : 0) + 8 * lq : nullptr;
  bf16x8_t qb[DC], wb[DC];
  float freq[D / 128], q_row = 1.f;
#pragma unroll
  for (int c = 0; c < DC; ++c) qb[c] = *(const bf16x8_t*)(qp + 32 * c);
  if (qw) {
#pragma unroll
    for (int c = 0; c < DC; ++c) wb[c] = *(const bf16x8_t*)(qw + 32 * c);
  }
#pragma unroll
  for (int j = 0; j < D / 128; ++j) freq[j] = lane + 64 * j < A.rot_dims / 2 ? A.rot_freq[lane + 64 * j] : 0.f;
  if (A.q_row) q_row = A.q_row[t];
  __builtin_amdgcn_sched_barrier(0);
  const int s = A.tseq[t], pos = A.ctx0[s] + (int)t - A.cu_q[s];
  const int lo = vis_lo(pos, A.window, A.chunk), first = lo >> 5, tiles = (pos >> 5) - first + 1;
  const int32_t* __restrict__ bt = A.block_tables + (int64_t)s * A.bt_stride;
  char* ring = lds + wave * RING;
  // requests. K: row = token, 16-byte unit u of token r at u ^ (r & 3 | (r >> 3 & 3) << 2); V: row = value column, 32 tokens, unit u of column c at
  // u ^ (c >> 2 & 3): the 16 rows of an operand read lie on all banks once
  uint32_t koff[KR], voff[VR];
#pragma unroll
  for (int i = 0; i < KR; ++i) {
    const int r = i * (64 / KU) + lane / KU, u = (lane % KU) ^ ((r & 3) | (r >> 3 & 3) << 2);
    koff[i] = (uint32_t)((r * A.G * D + u * 8) * 2);
  }
#pragma unroll
  for (int i = 0; i < VR; ++i) {
    const int c = i * 16 + (lane >> 2), u = (lane & 3) ^ (c >> 2 & 3);
    voff[i] = (uint32_t)((c * A.block_size + u * 8) * 2);
  }
  const auto page_of = [&](int i) { return bt[((first + i) * 32) >> A.bs_shift]; };
  const auto request = [&](int i, int page) {
    const int off = ((first + i) * 32) & (A.block_size - 1);
    const char* kp = (const char*)A.k_cache + ((((int64_t)page << A.bs_shift) + off) * A.G + g) * D * 2;
    const char* vp = (const char*)A.v_cache + (((((int64_t)page * A.G + g) * DV) << A.bs_shift) + off) * 2;
#pragma unroll
    for (int k = 0; k < KR; ++k) __builtin_amdgcn_global_load_lds((global_void_t*)(kp + koff[k]), (lds_void_t*)(ring + k * 1024), 16, 0, 0);
#pragma unroll
    for (int k = 0; k < VR; ++k) __builtin_amdgcn_global_load_lds((global_void_t*)(vp + voff[k]), (lds_void_t*)(ring + KB + k * 1024), 16, 0, 0);
  };
  int i = wave, page = i < tiles ? page_of(i) : 0;
  if (i < tiles) request(i, page);
  if (i + NW < tiles) page = page_of(i + NW);

  // ---- queries: lane holds entries 32 c + 8 lq .. + 7 of head li, normed, turned and scaled
  {
    float2* turn = (float2*)(lds + NW * RING) + wave * (D / 2);        // (each wavefront's own: no barrier)
#pragma unroll
    for (int j = 0; j < D / 128; ++j) {
      if (lane + 64 * j < A.rot_dims / 2) {
        float sn, cs;
        sincosf((float)pos * freq[j], &sn, &cs);
        turn[lane + 64 * j] = make_float2(cs, sn);
      }
    }
    float r = A.scale * query_temp(pos, A.qt_coef, A.qt_every);
    if (A.q_row) {
      r *= q_row;
    } else if (qw) {
      float ss = 0.f;
#pragma unroll
      for (int c = 0; c < DC; ++c)
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += (float)qb[c][e] * (float)qb[c][e];
      ss += __shfl_xor(ss, 16, 64), ss += __shfl_xor(ss, 32, 64);
      r *= rsqrtf(ss / (float)D + A.eps);
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      float w[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) w[e] = qw ? (float)wb[c][e] : 1.f;
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const int col = 32 * c + 8 * lq + e;
        float a = (float)qb[c][e] * r * w[e], b = (float)qb[c][e + 1] * r * w[e + 1];
        if (col < A.rot_dims) {                      // the pair (2i, 2i+1) turns by pos * freq[i]
          const float2 f = turn[col >> 1];
          const float a2 = a * f.x - b * f.y;
          b = b * f.x + a * f.y;
          a = a2;
        }
        qb[c][e] = (bf16_t)a, qb[c][e + 1] = (bf16_t)b;
      }
    }
  }
  // a sink is a score in the denominator without a value: the first wavefront's sum starts from it (once per query). One that weighs nothing beside any
  // score is none: the maximum lies above that of a tile in which nothing is seen
  const float sink = A.sink && wave == 0 ? A.sink[h] : -INFINITY;
  const bool none = sink < -1e30f;
  float m = none ? -1e30f : sink, l = none || lq != 0 ? 0.f : 1.f;
  f32x4_t o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const char* kread = ring + (8 * (li >> 2) + (li & 3)) * D * 2;
  const char* vread = ring + KB + li * 64 + (lq ^ (li >> 2)) * 16;
#pragma unroll 1
  for (; i < tiles; i += NW) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0F70);              // vmcnt(0): the tile landed
    __builtin_amdgcn_sched_barrier(0);
    bf16x8_t kf[2][DC];
    u32x4_t vf[DB];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int c = 0; c < DC; ++c) kf[kb][c] = *(const bf16x8_t*)(kread + kb * 4 * D * 2 + (((c * 4 + lq) ^ li) * 16));
#pragma unroll
    for (int db = 0; db < DB; ++db) vf[db] = *(const u32x4_t*)(vread + db * 16 * 64);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);              // lgkmcnt(0): it is read, its place can be filled again
    __builtin_amdgcn_sched_barrier(0);
    if (i + NW < tiles) {
      request(i + NW, page);
      if (i + 2 * NW < tiles) page = page_of(i + 2 * NW);
    }
    f32x4_t sc[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int c = 0; c < DC; ++c)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) sc[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[kb][c], qb[c], sc[kb], 0, 0, 0);
    float p[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) p[e] = sc[e >> 2][e & 3];
    if (A.softcap > 0.f) {
#pragma unroll
      for (int e = 0; e < 8; ++e) p[e] = capped(p[e], A.softcap);
    }
    const int j0 = (first + i) * 32;
    if (j0 < lo || j0 + 31 > pos) {
      unsigned keep[4];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int key = j0 + 8 * lq + e;
        const bool seen = key >= lo && key <= pos;
        if (!seen) p[e] = HIDDEN;
        const unsigned half = seen ? (e & 1 ? 0xffff0000u : 0xffffu) : 0u;
        keep[e >> 1] = e & 1 ? keep[e >> 1] | half : half;
      }
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int k = 0; k < 4; ++k) vf[db][k] &= keep[k];
    }
    float mx = HIDDEN;
#pragma unroll
    for (int e = 0; e < 8; ++e) mx = fmaxf(mx, p[e]);
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    const float mn = fmaxf(m, fmaxf(mx, __shfl_xor(mx, 32, 64)));
    if (__ballot(mn != m) != 0ull) {
      const float alpha = __builtin_amdgcn_exp2f((m - mn) * LOG2E);
      l *= alpha;
      m = mn;
#pragma unroll
      for (int db = 0; db < DB; ++db) o[db] *= alpha;
    }
    bf16x8_t pb;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float w = __builtin_amdgcn_exp2f((p[e] - m) * LOG2E);
      l += w;
      pb[e] = (bf16_t)w;
    }
#pragma unroll
    for (int db = 0; db < DB; ++db) o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, vf[db]), pb, o[db], 0, 0, 0);
  }

  // ---- the wavefronts' parts: each leaves its own in its ring
  l += __shfl_xor(l, 16, 64), l += __shfl_xor(l, 32, 64);
  float2* parts = (float2*)(lds + NW * RING + NW * D * 4);
  if (lq == 0) parts[wave * 16 + li] = make_float2(m, l);
#pragma unroll
  for (int db = 0; db < DB; ++db) *(f32x4_t*)(ring + (db * 64 + lane) * 16) = o[db];
  __syncthreads();
  if (li >= heads) return;
  float top = -INFINITY, sum = 0.f, f[NW];           // (the lane's query is the same in every pass below)
#pragma unroll
  for (int w = 0; w < NW; ++w) top = fmaxf(top, parts[w * 16 + li].x);
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const float2 e = parts[w * 16 + li];
    f[w] = __builtin_amdgcn_exp2f((e.x - top) * LOG2E);
    sum += f[w] * e.y;
  }
  const float inv = 1.f / sum;
  typedef __attribute__((ext_vector_type(4))) __bf16 b4_t;
  bf16_t* op = (bf16_t*)A.out + (t * A.H + h) * DV;
  const bf16_t* gp = A.gate ? (const bf16_t*)A.gate + t * A.gate_stride + (int64_t)h * A.gate_w : nullptr;
  const bool wide = gp && A.gate_w != 1;
  const float ginv = gp && !wide ? inv * sigmoid_hw((float)gp[0]) : inv;
  for (int db = wave; db < DB; db += NW) {
    f32x4_t v = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) v += f[w] * *(const f32x4_t*)(lds + w * RING + (db * 64 + lane) * 16);
    const int c = db * 16 + lq * 4;
    b4_t out;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float x = v[k] * ginv;
      if (wide) x *= sigmoid_hw((float)gp[c + k]);
      out[k] = (bf16_t)x;
    }
    *(b4_t*)(op + c) = out;
  }
}

template <int D, int DV, int NW>
int launch_token(WindowAttnArgs a, hipStream_t stream) {
  a.bs_shift = __builtin_ctz(a.block_size);
  constexpr int LDS = NW * (32 * D * 2 + DV * 64 + D * 4 + 128);
  const auto kernel = window_attn_token_kernel<D, DV, NW>;
  NVS_LDS_ROOM(kernel, LDS, "nvs_window_attn");
  kernel<<<dim3((unsigned)a.n, (unsigned)(a.G * ((a.H / a.G + 15) / 16))), dim3(64 * NW), LDS, stream>>>(a);
  return nvs_check_launch("nvs_window_attn (single tokens)");
}

}  // namespace

int window_attn_token(const WindowAttnArgs& a, hipStream_t stream) {
  return a.d == 128 ? launch_token<128, 128, 8>(a, stream) : launch_token<256, 192, 4>(a, stream);
}
