// Windowed attention over the paged cache, pipelined (bf16, 128-wide heads or latent rows of 256 with values of 192): device code shared by the
// translation units that instantiate it (attn_prompt.hip: windows, blocks, causal; attn_prompt_latent.hip: latent rows whose queries come unfinished; attn_prompt_pool.hip: the same with pooled blocks, capped
// scores and row factors). Masks, sink, temperature, norm, rotation and gate mean what they mean in attn_window_core.h, whose kernels take every
// other size.
#pragma once
#include "attn_window_core.h"

int window_attn_prompt(const WindowAttnArgs& a, hipStream_t stream);               // attn_prompt.hip
int window_attn_prompt_extended(const WindowAttnArgs& a, hipStream_t stream);      // attn_prompt_pool.hip
int window_attn_prompt_latent(const WindowAttnArgs& a, hipStream_t stream);        // attn_prompt_latent.hip

namespace {

typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((address_space(3))) void lds_void_t;
typedef const __attribute__((address_space(1))) void global_void_t;

__device__ __forceinline__ void dma16(const void* src, char* lds_at) {          // 64 lanes: LDS [lds_at + 16 lane] <- 16 bytes at src
  __builtin_amdgcn_global_load_lds((global_void_t*)src, (lds_void_t*)lds_at, 16, 0, 0);
}
__device__ __forceinline__ float other_half(float v) {                          // the value of lane ^ 32
  const unsigned u = __builtin_bit_cast(unsigned, v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, (threadIdx.x & 32) ? r[0] : r[1]);
}
// (a, b) turns. Which of a sum's two products is rounded by itself is said here: left to the compiler, it changed with code around it, and from one pair of a row to the next.
__device__ __forceinline__ void turn_pair(float& a, float& b, float cs, float sn) {
  const float a2 = __builtin_fmaf(a, cs, -(b * sn));
  b = __builtin_fmaf(b, cs, a * sn);
  a = a2;
}
template <int N>
struct Int { static constexpr int value = N; };
template <int BEGIN, int END, typename F>
__device__ __forceinline__ void static_for(const F& f) {                        // f(Int<BEGIN>) ... f(Int<END - 1>): the index is a constant
  if constexpr (BEGIN < END) {
    f(Int<BEGIN>{});
    static_for<BEGIN + 1, END>(f);
  }
}

constexpr float LOG2E = 1.4426950408889634f;
constexpr float HIDDEN = -3e38f;                  // a masked score: its weight is 0 whatever the maximum is

// A wavefront owns 32 consecutive queries of one head and walks over tiles of 64 keys, which all wavefronts of the workgroup share: `hw` heads of one
// kv head times NW / hw groups of 32 queries. K and V tiles come straight into LDS, double-buffered, a round ahead.
//
// Everything is computed transposed, so that a lane owns ONE query (column lane & 31; the two halves of the wavefront hold different keys or value
// columns of it) and a maximum or sum over keys needs one exchange between the halves:
//   S^T [32 keys x 32 queries] = K Q^T, O^T [32 columns x 32 queries] += V^T P^T      (v_mfma_f32_32x32x16_bf16)
// Row r of a block of 32 keys is key 16 (r >> 4) + 8 ((r >> 2) & 1) + 4 ((r >> 3) & 1) + (r & 3): the 16 scores a lane gets are then two runs of 8
// consecutive keys, which, as bf16 weights, are its operand of the second product as they are.
//
// 128-wide heads (PIPE): in one round the matrix cores compute the sums of the round before and the scores of the round after, and between
// those products stand pieces of this round's maximum and weights, so that a wavefront keeps both units busy; two workgroups of four wavefronts
// fit a compute unit. Rows of 256: scores, weights, sums one after the other, by two wavefronts per SIMD (a workgroup of eight: 256 registers hold
// one round's scores only) that fill each other's gaps.
//
// What bounds it: per round and wavefront 32 MFMAs (rows of 256: 56) of 32 clocks, as much of the LDS pipe's time for eight wavefronts, and about 1,000
// clocks of vector work; the matrix units run at 0.92-1.03 PFLOP/s on one prompt of 16,384 tokens. On shorter ones the time before the first and
// behind the last round shows: queries, norm and rotation are prepared while the first tile is on its way, cos and sin once per position and
// workgroup. 64 queries per wavefront (half the LDS reads) need the accumulation registers, and the compiler's moves to and from them cost more.
// MI355X, 13,550 tokens in 9 prompts, before (window_attn_mfma_lds_kernel) and now, us: 32 / 8 heads, window 1024, norm and gate 1300 -> 351, blocks of
// 1024 with rotation 936 -> 255; 16 / 8 heads, causal, rotation, sink 764 -> 189; latent rows, 16 heads, window 1024 and causal 1013 -> 240.
// HEADS: latent rows whose queries come unfinished (1) and whose results leave through W_uv too (2)
template <int D, int DV, int NW, bool EXT, int HEADS = 0>
__global__ __launch_bounds__(64 * NW, D == 128 ? 2 : 1) void window_attn_prompt_kernel(const WindowAttnArgs A) {
  constexpr bool PIPE = D == 128;
  constexpr int KB = 64 * D * 2, VB = DV * 128, TILE = KB + VB, KU = D / 8, KI = KB / 1024 / NW, VI = VB / 1024 / NW, DC = D / 16, DB = DV / 32;
  extern __shared__ __attribute__((aligned(128))) char lds[];                   // K tile, V tile; K tile, V tile
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), ql = lane & 31, hi = lane >> 5;
  const int H = A.H, G = A.G, hpg = H / G, hw = A.hw, chunks = hpg / hw, window = A.window, chunk = A.chunk, bs = A.block_size;
  const int rows = H / hw, BQ = (NW / hw) * 32;
  const int place = (int)(blockIdx.x + gridDim.x * blockIdx.y), y = place % rows, g = y / chunks, h = g * hpg + (y % chunks) * hw + wave % hw;
  int btile = place / rows, s = 0, len = 0, row0 = 0, c0 = 0;
  if (A.nseq <= 64) {
    // Tiles go by their place among the positions, the furthest first, whatever portion they are of, and heads before tiles: what begins last is short. (Portion by portion and
    // head by head the last quarter of the time had fewer than half of the workgroups. 14,200 tokens in 9 prompts, four layers of latent rows 2,899 -> 2,808 us, of 16 / 8 heads
    // 3,940 -> 3,860; the clock then falls from 2.1 to 1.9 GHz.) A portion has tiles at places first .. last - 1; the tiles from a place on are counted for 64 places at once, a lane each
    const int i = lane < A.nseq ? lane : 0, at = A.cu_q[i], n_i = lane < A.nseq ? A.cu_q[i + 1] - at : 0, c_i = A.ctx0[i], first = c_i / BQ, last = first + (n_i + BQ - 1) / BQ;
    const auto from = [&](int p) {
      int sum = 0;
      for (int j = 0; j < A.nseq; ++j) {
        const int f = __builtin_amdgcn_readlane(first, j), e = __builtin_amdgcn_readlane(last, j);
        sum += max(e - max(p, f), 0);
      }
      return sum;
    };
    int stride = 64, sum = from(lane * stride);     // the furthest place, `low`, with more than btile tiles from it on
    uint64_t more = __ballot(sum > btile);
    while (more >> 63) stride <<= 6, sum = from(lane * stride), more = __ballot(sum > btile);
    if (!more) return;                              // the whole workgroup leaves
    int low = (__builtin_popcountll(more) - 1) * stride;
    while (stride >>= 6) {
      sum = from(low + lane * stride), more = __ballot(sum > btile);
      if (stride == 1) break;
      low += (__builtin_popcountll(more) - 1) * stride;
    }
    const int step = __builtin_popcountll(more) - 1;
    low += step;
    const uint64_t there = __ballot(first <= low && low < last);
    const int behind = __builtin_amdgcn_readlane(sum, step) - __builtin_popcountll(there);
    const int before = __builtin_amdgcn_mbcnt_hi((uint32_t)(there >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)there, 0));
    s = __builtin_ctzll(__ballot((there >> lane & 1) && before == btile - behind));
    len = __builtin_amdgcn_readlane(n_i, s), row0 = __builtin_amdgcn_readlane(at, s), c0 = __builtin_amdgcn_readlane(c_i, s);
    btile = low - __builtin_amdgcn_readlane(first, s);
  } else {
    // 64 portions at a time, their tile counts summed over the lanes
    for (int base = 0;; base += 64) {
      const int i = base + lane;
      const int first = i <= A.nseq ? A.cu_q[i] : 0, n_i = i < A.nseq ? A.cu_q[i + 1] - first : 0, tiles = (n_i + BQ - 1) / BQ;
      int sum = tiles;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int up = __shfl_up(sum, d, 64);
        sum += lane >= d ? up : 0;
      }
      const uint64_t in = __ballot(btile < sum);
      if (in != 0) {
        const int at = __builtin_ctzll(in);
        s = base + at;
        len = __builtin_amdgcn_readlane(n_i, at);
        row0 = __builtin_amdgcn_readlane(first, at);
        btile -= __builtin_amdgcn_readlane(sum - tiles, at);
        break;
      }
      btile -= __builtin_amdgcn_readlane(sum, 63);
      if (base + 64 >= A.nseq) return;              // the whole workgroup leaves
    }
    btile = (len + BQ - 1) / BQ - 1 - btile;        // the last query tiles of a portion, which see the most, go first
    c0 = __builtin_amdgcn_readfirstlane(A.ctx0[s]);
  }
  const int rel0 = btile * BQ + wave / hw * 32, p_first = c0 + rel0, p_hi = p_first + 31;
  const int b_first = c0 + btile * BQ, b_last = c0 + (btile * BQ + BQ < len ? btile * BQ + BQ : len) - 1;
  const int32_t* __restrict__ bt = A.block_tables + (int64_t)s * A.bt_stride;

  // ---- rounds: EXT: [0, npr) hold 64 pooled blocks each, the others 64 tokens, the first from a multiple of 64 on
  const int lo = vis_lo(b_first, window, chunk);
  const int nb_last = EXT ? seen_blocks(b_last, window, A.pool) : 0, npr = EXT ? (nb_last + 63) >> 6 : 0;
  const int jt = (lo & ~63) - npr * 64;
  const int rounds = npr + ((b_last - (lo & ~63)) >> 6) + 1;
  // the rounds every query of this wavefront sees in whole
  const int nb_first = EXT ? seen_blocks(p_first, window, A.pool) : 0, lo_hi = vis_lo(p_hi, window, chunk);
  // Rounds none of them sees are left out: a weight of 0 times a value that is not finite is NaN, in outputs of tokens that do not see it. All
  // behind `final` are such rounds (-1: a wavefront of nobody's queries) and, without pooled blocks, those that end before `lo_first`. (The branches
  // cost 0 to 3 % of whole prompts; single tokens with capped scores and one head over each of eight, 64 sequences, 148 -> 109 us.)
  const int final = rel0 < len ? (c0 + (rel0 + 31 < len ? rel0 + 31 : len - 1) - jt) >> 6 : -1, lo_first = vis_lo(p_first, window, chunk);
  const auto early = [&](int it) { return !EXT && jt + it * 64 + 63 < lo_first; };

  // ---- requests. K tile: row = token, 2 D bytes, 16-byte unit u of token t at u ^ (t & 15). V tile: row = value column, 64 tokens = 128 bytes, unit u of
  // column c at u ^ ((c >> 1) & 7). Both make the 16-byte operand reads of 16 neighbouring lanes cover all banks once.
  uint32_t koff[KI], voff[VI];                      // bytes from the tile's first row
  int kblk[KI], vblk[2];                            // EXT: unit of 8 blocks of a request's rows; of a lane's tokens (even, odd requests)
#pragma unroll
  for (int i = 0; i < KI; ++i) {
    const int r = (wave * KI + i) * (64 / KU) + lane / KU;
    int u = (lane % KU) ^ (r & 15);
    if (HEADS && u < 24) u = u / 6 * 6 + u % 2 * 3 + u % 6 / 2;                 // (the order in which a lane gets its query's entries, below)
    koff[i] = (uint32_t)(((EXT ? r & 7 : r) * G * D + u * 8) * 2);
    kblk[i] = r >> 3;
  }
#pragma unroll
  for (int i = 0; i < VI; ++i) {
    const int c = (wave * VI + i) * 8 + (lane >> 3), u = (lane & 7) ^ ((c >> 1) & 7);
    const int column = HEADS == 2 ? (c & ~12) | (c & 4) << 1 | (c & 8) >> 1 : c;      // (a lane then holds 8 columns in a row, below)
    voff[i] = (uint32_t)((EXT ? c * 8 : column * bs + u * 8) * 2);
    if (i < 2) vblk[i] = u;
  }
  // Pages (EXT: units of pooled blocks) are looked up a round before the requests that use them: a lookup inside a request would wait for
  // everything in flight. kpg, vpg: of the next K and V tile to be requested (EXT: of a wavefront's first and last rows, of its even and odd requests).
  int kpg[2] = {}, vpg[2] = {};
  const auto unit_of = [&](int it, int u) {         // unit u of pooled round it (one that nobody sees: the round's first)
    return pool_unit(it * 8 + (it * 64 + u * 8 < nb_last ? u : 0), A.pool, bs, bt);
  };
  const auto page_of = [&](int it) { return bt[(jt + it * 64) >> A.bs_shift]; };
  const auto lookup_k = [&](int it) {
    if (it >= rounds) return;
    if (EXT && it < npr) kpg[0] = unit_of(it, kblk[0]), kpg[1] = unit_of(it, kblk[KI - 1]);
    else kpg[0] = page_of(it);
  };
  const auto lookup_v = [&](int it) {
    if (it >= rounds) return;
    if (EXT && it < npr) vpg[0] = unit_of(it, vblk[0]), vpg[1] = unit_of(it, vblk[1]);
    else vpg[0] = page_of(it);
  };
  const auto request_k = [&](int it, int buf) {
    if (it >= rounds) return;
    char* at = lds + buf * TILE + wave * KI * 1024;
    if (EXT && it < npr) {
#pragma unroll
      for (int i = 0; i < KI; ++i) dma16((const char*)A.pool_k + ((int64_t)kpg[2 * i / KI] * 8 * G + g) * D * 2 + koff[i], at + i * 1024);
      return;
    }
    const int off = (jt + it * 64) & (bs - 1), page = __builtin_amdgcn_readfirstlane(kpg[0]);
    const char* base = (const char*)A.k_cache + ((((int64_t)page << A.bs_shift) + off) * G + g) * D * 2;
#pragma unroll
    for (int i = 0; i < KI; ++i) dma16(base + koff[i] + (EXT ? (uint32_t)kblk[i] * 8 * G * D * 2 : 0u), at + i * 1024);
  };
  const auto request_v = [&](int it, int buf) {
    if (it >= rounds) return;
    char* at = lds + buf * TILE + KB + wave * VI * 1024;
    if (EXT && it < npr) {
#pragma unroll
      for (int i = 0; i < VI; ++i) dma16((const char*)A.pool_v + ((int64_t)vpg[i & 1] * G + g) * DV * 16 + voff[i], at + i * 1024);
      return;
    }
    const int off = (jt + it * 64) & (bs - 1), page = __builtin_amdgcn_readfirstlane(vpg[0]);
    const char* base = (const char*)A.v_cache + (((((int64_t)page * G + g) * DV) << A.bs_shift) + off) * 2;
#pragma unroll
    for (int i = 0; i < VI; ++i) {
      const int c = (wave * VI + i) * 8 + (lane >> 3);
      dma16(base + (EXT ? (uint32_t)((c * bs + vblk[i & 1] * 8) * 2) : voff[i]), at + i * 1024);
    }
  };
  // Tokens behind the step's last one lie in the page but belong to nobody: their weight is 0, and their values are made 0 too, since what a
  // page held before may be an infinity. (Pooled rounds: blocks nobody sees, likewise; a round behind the last one: all of it.)
  const auto clear_tail = [&](int it, int buf) {
    if (it < rounds - 1 && !(EXT && it == npr - 1)) return;
    const int live = EXT && it < npr ? nb_last - it * 64 : b_last - (jt + it * 64) + 1;
    if (live >= 64) return;
    char* at = lds + buf * TILE + KB;
    for (int i = tid; i < DV * 64; i += 64 * NW) {
      const int c = i >> 6, t = i & 63;
      if (t >= live) *(bf16_t*)(at + c * 128 + (((t >> 3) ^ ((c >> 1) & 7)) << 4) + (t & 7) * 2) = (bf16_t)0.f;
    }
    __syncthreads();
  };
  const auto arrive = [&] {                         // own requests landed and own reads done; then everybody's
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  lookup_k(0);
  lookup_v(0);
  request_k(0, 0);
  request_v(0, 0);
  lookup_k(1);
  lookup_v(1);

  // ---- queries, while the first tile is on its way: lane holds entries 16 c + 8 hi .. + 7 of query ql, normed, turned and scaled
  const int rel = rel0 + ql, pos = c0 + rel;
  const bool valid = rel < len;
  const int64_t row = (int64_t)row0 + (valid ? rel : len - 1);
  bf16x8_t qb[DC];
  if constexpr (D == 128) {
    const bf16_t* qp = (const bf16_t*)A.q + row * A.q_stride + (int64_t)h * D + 8 * hi;
#pragma unroll
    for (int c = 0; c < DC; ++c) qb[c] = *(const bf16x8_t*)(qp + 16 * c);
    const int pairs = A.rot_dims / 2;
    const bool table = pairs > 0 && BQ * pairs * 8 <= TILE;                     // cos and sin once per position, not once per head
    float2* turn = (float2*)(lds + TILE);
    if (table) {
      for (int i = tid; i < BQ * pairs; i += 64 * NW) {
        const int p = i / pairs, j = i - p * pairs;
        float sn, cs;
        sincosf((float)(b_first + p) * A.rot_freq[j], &sn, &cs);
        turn[i] = make_float2(cs, sn);
      }
      __syncthreads();
    }
    float r = A.scale * query_temp(pos, A.qt_coef, A.qt_every);
    const bf16_t* qw = (const bf16_t*)A.qnorm;
    if (EXT && A.q_row) {
      r *= A.q_row[row];
      qw += (int64_t)h * D;
    } else if (qw) {
      float ss = 0.f;
#pragma unroll
      for (int c = 0; c < DC; ++c)
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += (float)qb[c][e] * (float)qb[c][e];
      ss += other_half(ss);
      r *= rsqrtf(ss / (float)D + A.eps);
    }
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      float w[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) w[e] = 1.f;
      if (qw) ldp<8>(qw + 16 * c + 8 * hi, w);
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const int col = 16 * c + 8 * hi + e;
        float a = (float)qb[c][e] * r * w[e], b = (float)qb[c][e + 1] * r * w[e + 1];
        if (col < A.rot_dims) {                     // the pair (2i, 2i+1) turns by pos * freq[i]
          float sn, cs;
          if (table) {
            const float2 f = turn[(rel - btile * BQ) * pairs + (col >> 1)];
            cs = f.x, sn = f.y;
          } else {
            sincosf((float)pos * A.rot_freq[col >> 1], &sn, &cs);
          }
          turn_pair(a, b, cs, sn);
        }
        qb[c][e] = (bf16_t)a, qb[c][e + 1] = (bf16_t)b;
      }
    }
  } else if constexpr (HEADS != 0) {
    // The product with W_uk,h stands here: a lane's results are its query's operands of the scores as they are. The queries' 128 + 64 entries are requested as they lie, the last 64
    // turn, and through the second tile's place and what lies behind it they become operands. W_uk,h [128][192] comes straight from L2, k-step by k-step two ahead: lane l asks for
    // entries 6 l .. 6 l + 5 of eight rows and turns them by byte permutations, so block j of 32 latent entries holds 6 l + j in row l. A lane then has 24 entries in a row
    // for each a: 48 a + 24 hi + 0 .. 23, units 6 a + 3 hi + t of eight; the key tile's units lie in LDS in that order.
    // As a launch of its own the product reads and writes every head's row once more, 68 us of 14,200 rows and 16 heads (210 MB); here a workgroup's queries take as long as 256 finished
    // entries did (7.2 us: 48 KB of weights a wavefront, 1.5 us of products): window 1,024 68 + 234 -> 246 us, four layers of 14,200 tokens 3,270 -> 3,024.
    constexpr int NOPE = 128, TAIL = 64, ROWS = 32 * (NOPE + TAIL) * 2;
    typedef __attribute__((ext_vector_type(3))) unsigned int u32x3_t;
    const int nu = lane & 15, nr = lane >> 4, tu = lane & 7, tr = lane >> 3, half = A.rot_dims >> 1, apart = half >> 3;
    const bool turns = tu * 8 < A.rot_dims, halves = A.rot_halves != 0, upper = tu >= apart;              // halves: entry i turns with entry i + half, which a lane `apart` units on holds
    const bf16_t* qp = (const bf16_t*)A.q + (int64_t)row0 * A.q_stride + (int64_t)h * (NOPE + TAIL);
    const auto at_row = [&](int r) { return (int64_t)(rel0 + r < len ? rel0 + r : len - 1); };
    const char* wp = (const char*)A.uk + (int64_t)h * NOPE * DV * 2 + hi * 8 * DV * 2 + ql * 12;
    bf16x8_t qn[8], qt[4];
    f32x4_t cs[4][4];
    u32x3_t w[3][8];
    const auto bring = [&](auto step) {
      constexpr int k = decltype(step)::value;
#pragma unroll
      for (int j = 0; j < 8; ++j) __builtin_memcpy(&w[k % 3][j], __builtin_assume_aligned(wp + (k * 16 + j) * DV * 2, 4), 12);
    };
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      qt[i] = *(const bf16x8_t*)(qp + at_row(i * 8 + tr) * A.q_stride + NOPE + tu * 8);
      if (turns) {
        const float2* f = A.turn + (row0 + at_row(i * 8 + tr)) * half + (halves ? (upper ? tu - apart : tu) * 8 : tu * 4);
        cs[i][0] = *(const f32x4_t*)f, cs[i][1] = *(const f32x4_t*)(f + 2);
        if (halves) cs[i][2] = *(const f32x4_t*)(f + 4), cs[i][3] = *(const f32x4_t*)(f + 6);
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) qn[i] = *(const bf16x8_t*)(qp + at_row(i * 4 + nr) * A.q_stride + nu * 8);
    bring(Int<0>{});
    bring(Int<1>{});
    __builtin_amdgcn_sched_barrier(0);
    char* at = lds + TILE + wave * ROWS;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = i * 8 + tr;
      if (halves) {
        const u32x4_t own = __builtin_bit_cast(u32x4_t, qt[i]);
        u32x4_t theirs;
#pragma unroll
        for (int e = 0; e < 4; ++e) theirs[e] = (unsigned)__shfl((int)own[e], upper ? lane - apart : lane + apart, 64);
        const bf16x8_t other = __builtin_bit_cast(bf16x8_t, theirs);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float c = cs[i][e / 2][e % 2 * 2], sn = cs[i][e / 2][e % 2 * 2 + 1], v = (float)qt[i][e], o = (float)other[e];
          qt[i][e] = (bf16_t)((turns ? upper ? v * c + o * sn : v * c - o * sn : v) * A.scale);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          float a = (float)qt[i][e], b = (float)qt[i][e + 1];
          if (turns) {
            const float c = cs[i][e / 4][e % 4], sn = cs[i][e / 4][e % 4 + 1], a2 = a * c - b * sn;
            b = b * c + a * sn, a = a2;
          }
          qt[i][e] = (bf16_t)(a * A.scale), qt[i][e + 1] = (bf16_t)(b * A.scale);
        }
      }
      *(bf16x8_t*)(at + 32 * NOPE * 2 + r * TAIL * 2 + ((tu ^ ((r >> 1) & 7)) << 4)) = qt[i];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = i * 4 + nr;
      *(bf16x8_t*)(at + r * NOPE * 2 + ((nu ^ (r & 15)) << 4)) = qn[i];
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) qn[s] = *(const bf16x8_t*)(at + ql * NOPE * 2 + (((2 * s + hi) ^ (ql & 15)) << 4));
    f32x16_t acc[6];
    static_for<0, 8>([&](auto step) {
      constexpr int k = decltype(step)::value;
      if constexpr (k + 2 < 8) bring(Int<k + 2>{});
      __builtin_amdgcn_sched_barrier(0);
      static_for<0, 6>([&](auto block) {
        constexpr int j = decltype(block)::value;
        u32x4_t x;
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = __builtin_amdgcn_perm(w[k % 3][2 * i + 1][j / 2], w[k % 3][2 * i][j / 2], j % 2 ? 0x07060302u : 0x05040100u);
        const f32x16_t zero = {};
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, x), qn[k], k == 0 ? zero : acc[j], 0, 0, 0);
      });
      __builtin_amdgcn_sched_barrier(0);
    });
    static_for<0, 12>([&](auto index) {
      constexpr int c = decltype(index)::value, a = c / 3, t = c % 3;
      static_for<0, 8>([&](auto entry) {
        constexpr int x = 8 * t + decltype(entry)::value;
        qb[c][x % 8] = (bf16_t)(acc[x % 6][4 * a + x / 6] * A.scale);
      });
    });
#pragma unroll
    for (int c = 0; c < 4; ++c) qb[12 + c] = *(const bf16x8_t*)(at + 32 * NOPE * 2 + ql * TAIL * 2 + (((2 * c + hi) ^ ((ql >> 1) & 7)) << 4));
  } else {
    // Rows are requested as they lie, D / 8 lanes each, and turn into operands by way of the second tile's place, a few rows of every wavefront at a time. (A lane that
    // requests its own query's entries asks for 32 bytes of each of 32 rows; nothing hides that where one workgroup has the compute unit to itself: 12 us of 61 a
    // workgroup, 7.5 so, 14,200 tokens in 9 prompts, 16 heads, window 1,024 / causal 270 / 292 us, 251 / 275 so. 128-wide heads: no
    // difference.)
    constexpr int RL = D / 8, RI = 64 / RL, QI = 32 / RI, PASSES = 4, PR = 32 / PASSES, N = QI / PASSES;        // lanes of a row, rows of a request, requests; rows of a pass
    static_assert(NW * PR * D * 2 <= TILE, "a pass of all wavefronts' rows fits the second tile");
    const int sub = lane % RL, sub_row = lane / RL;
    bf16x8_t qr[QI];
    const bf16_t* qp = (const bf16_t*)A.q + (int64_t)row0 * A.q_stride + (int64_t)h * D + sub * 8;
#pragma unroll
    for (int i = 0; i < QI; ++i) {
      const int r = rel0 + i * RI + sub_row;
      qr[i] = *(const bf16x8_t*)(qp + (int64_t)(r < len ? r : len - 1) * A.q_stride);
    }
    float factor = A.scale * query_temp(pos, A.qt_coef, A.qt_every);
    const bf16_t* qw = (const bf16_t*)A.qnorm;
    const bool own_norm = qw && !(EXT && A.q_row);
    if (EXT && A.q_row) {
      factor *= A.q_row[row];
      qw += (int64_t)h * D;
    }
    const auto finish = [&](float (&v)[8], const float (&w)[8], int col) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = v[e] * factor * w[e];
      if (col >= A.rot_dims) return;
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        if (col + e < A.rot_dims) {                 // the pair (2i, 2i+1) turns by pos * freq[i]
          float sn, cs;
          sincosf((float)pos * A.rot_freq[(col + e) >> 1], &sn, &cs);
          turn_pair(v[e], v[e + 1], cs, sn);
        }
      }
    };
    char* at = lds + TILE + wave * PR * D * 2;
    const int mine = ql % PR;
    static_for<0, PASSES>([&](auto pass) {
      constexpr int p = decltype(pass)::value;
      static_for<0, N>([&](auto index) {
        constexpr int i = decltype(index)::value;
        const int r = i * RI + sub_row;
        *(bf16x8_t*)(at + r * D * 2 + ((sub ^ (r & 15)) << 4)) = qr[p * N + i];
      });
      static_for<0, DC>([&](auto index) {
        constexpr int c = decltype(index)::value;
        const u32x4_t x = *(const u32x4_t*)(at + mine * D * 2 + (((2 * c + hi) ^ (mine & 15)) << 4));
        if constexpr (p == 0) {
          qb[c] = __builtin_bit_cast(bf16x8_t, x);
        } else {
          u32x4_t y = __builtin_bit_cast(u32x4_t, qb[c]);
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = ql / PR == p ? x[e] : y[e];
          qb[c] = __builtin_bit_cast(bf16x8_t, y);
        }
      });
      __builtin_amdgcn_sched_barrier(0);
    });
    if (own_norm) {
      float ss = 0.f;
#pragma unroll
      for (int c = 0; c < DC; ++c)
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += (float)qb[c][e] * (float)qb[c][e];
      factor *= rsqrtf((ss + other_half(ss)) / (float)D + A.eps);
    }
    static_for<0, DC>([&](auto index) {
      constexpr int c = decltype(index)::value;
      float v[8], w[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (float)qb[c][e], w[e] = 1.f;
      if (qw) ldp<8>(qw + 16 * c + 8 * hi, w);
      finish(v, w, 16 * c + 8 * hi);
#pragma unroll
      for (int e = 0; e < 8; ++e) qb[c][e] = (bf16_t)v[e];
    });
  }
  // a sink is a score in the denominator without a value; the sum starts from it (once per query: in the lower half of the lanes). One that weighs
  // nothing beside any score is none: the maximum must lie above that of a round in which the query sees no key
  const float sink = A.sink ? A.sink[h] : -INFINITY;
  const bool none = sink < -1e30f;
  float m = none ? -1e30f : sink, l = none || hi != 0 ? 0.f : 1.f;
  f32x16_t o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[db][i] = 0.f;

  // ---- operands
  const int ktok = 16 * (ql >> 4) + 8 * ((ql >> 2) & 1) + 4 * ((ql >> 3) & 1) + (ql & 3);
  const char* kread = lds + ktok * D * 2;
  const int kswz = (hi ^ (ktok & 15)) * 16;          // unit 2 c + hi, swizzled: (2 c) ^ this
  const char* vread = lds + KB + ql * 128;
  const int vswz = (hi ^ ((ql >> 1) & 7)) * 16;      // unit 2 a + hi
  const auto k_operand = [&](int buf, int kb, int c) { return *(const bf16x8_t*)(kread + buf * TILE + kb * 32 * D * 2 + (kswz ^ (c * 32))); };
  const auto v_operand = [&](int buf, int a, int db) { return *(const bf16x8_t*)(vread + buf * TILE + db * 32 * 128 + (vswz ^ (a * 32))); };
  const auto s_product = [&](f32x16_t& d, const bf16x8_t& k, int c) {
    const f32x16_t zero = {};
    d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k, qb[c], c == 0 ? zero : d, 0, 0, 0);
  };
  const auto o_product = [&](f32x16_t& d, const bf16x8_t& v, const u32x4_t& p) {
    d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v, __builtin_bit_cast(bf16x8_t, p), d, 0, 0, 0);
  };

  // ---- the vector units' part of round `it`, in 13 pieces: caps, masks and maxima of eight scores (0-3), the new maximum (4), four weights (5-12)
  float mx = HIDDEN, alpha = 1.f;
  bool whole = true, moved = false;
  int rlo = 0;
  unsigned rlen = 0u;
  const auto begin = [&](int it) {
    const bool pooled = EXT && it < npr;
    const int j0 = pooled ? it * 64 : jt + it * 64;
    whole = pooled ? j0 + 63 < nb_first : j0 + 63 <= p_first && j0 >= lo_hi;
    if (!whole) {                                   // visible: tokens rlo .. rlo + rlen of the round, counted from this lane's first
      const int top = pooled ? seen_blocks(pos, window, A.pool) - 1 : pos, bottom = pooled ? 0 : vis_lo(pos, window, chunk);
      rlo = top >= bottom ? bottom - j0 - 8 * hi : 0x40000000;
      rlen = top >= bottom ? (unsigned)(top - bottom) : 0u;
    }
  };
  const auto work = [&](auto unit, f32x16_t (&sc)[2], u32x4_t (&pb)[4]) {
    constexpr int u = decltype(unit)::value;
    if constexpr (u < 4) {
      f32x16_t& v = sc[u >> 1];
      if constexpr (u == 0) mx = HIDDEN;
      if (EXT) {
        if (A.softcap > 0.f) {
#pragma unroll
          for (int i = 0; i < 8; ++i) v[(u & 1) * 8 + i] = capped(v[(u & 1) * 8 + i], A.softcap);
        }
      }
      if (!whole) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if ((unsigned)(u * 16 + i - rlo) > rlen) v[(u & 1) * 8 + i] = HIDDEN;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) mx = fmaxf(mx, v[(u & 1) * 8 + i]);
      asm volatile("" : "+v"(mx));                  // (a piece stays where it stands: the compiler would move all of it to where it is used)
    } else if constexpr (u == 4) {
      const float mn = fmaxf(m, fmaxf(mx, other_half(mx)));
      moved = __ballot(mn != m) != 0ull;
      alpha = __builtin_amdgcn_exp2f((m - mn) * LOG2E);
      l *= alpha;
      m = mn;
      asm volatile("" : "+v"(alpha), "+v"(m), "+v"(l));
    } else {
      typedef __attribute__((ext_vector_type(2))) __bf16 b2_t;
      constexpr int i0 = (u - 5) * 4;
      float p[4];                                   // (the maximum is taken off first: as one fused step with its product with log2 e, rounded,
#pragma unroll                                    // rounds with different maxima weigh on different scales; that saves 1-3 % of the kernel's time)
      for (int i = 0; i < 4; ++i) p[i] = __builtin_amdgcn_exp2f((sc[i0 >> 4][(i0 & 15) + i] - m) * LOG2E);
      l += (p[0] + p[1]) + (p[2] + p[3]);
      unsigned w0 = __builtin_bit_cast(unsigned, b2_t{(bf16_t)p[0], (bf16_t)p[1]}), w1 = __builtin_bit_cast(unsigned, b2_t{(bf16_t)p[2], (bf16_t)p[3]});
      asm volatile("" : "+v"(w0), "+v"(w1), "+v"(l));
      pb[i0 >> 3][(i0 & 7) >> 1] = w0;
      pb[i0 >> 3][((i0 & 7) >> 1) + 1] = w1;
    }
  };
  const auto rescale = [&] {
    if (moved) {
#pragma unroll
      for (int db = 0; db < DB; ++db) o[db] *= alpha;
    }
  };
  constexpr int UNITS = 13, AHEAD = 3;              // AHEAD: operands read ahead of their products

  if constexpr (PIPE) {
    f32x16_t sc[2][2];
    u32x4_t pb[2][4];
    // Round it: sums of round it - 1 (V tile in buffer nxt), scores of round it + 1 (K tile in buffer nxt); K tile it + 2 and V tile it come into cur.
    const auto turn = [&](bool first, int it, int cur) {
      arrive();
      if (!first) clear_tail(it - 1, cur ^ 1);
      request_k(it + 2, cur);
      if (!first) request_v(it, cur);
      lookup_k(it + 3);
      if (!first) lookup_v(it + 1);
    };
    const auto round = [&](auto first, int it, auto which) {
      constexpr bool FIRST = decltype(first)::value != 0, WITH_O = !FIRST;
      constexpr int cur = decltype(which)::value, nxt = cur ^ 1, OS = WITH_O ? 4 * DB : 0, SLOTS = OS + 2 * DC;
      turn(FIRST, it, cur);
      begin(it);
      bf16x8_t ring[AHEAD + 1];
      const auto operand = [&](int slot) { return slot < OS ? v_operand(nxt, slot / DB, slot % DB) : k_operand(nxt, (slot - OS) / DC, (slot - OS) % DC); };
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) ring[i] = operand(i);
      static_for<0, SLOTS>([&](auto index) {
        constexpr int slot = decltype(index)::value;
        if constexpr (slot + AHEAD < SLOTS) ring[(slot + AHEAD) % (AHEAD + 1)] = operand(slot + AHEAD);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (slot < OS) o_product(o[slot % DB], ring[slot % (AHEAD + 1)], pb[nxt][slot / DB]);
        else s_product(sc[nxt][(slot - OS) / DC], ring[slot % (AHEAD + 1)], (slot - OS) % DC);
        static_for<slot * UNITS / SLOTS, (slot + 1) * UNITS / SLOTS>([&](auto u) { work(u, sc[cur], pb[cur]); });
        __builtin_amdgcn_sched_barrier(0);
      });
      if (!FIRST && early(it - 1)) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
      }
      if (!FIRST) rescale();
    };
    arrive();
    request_k(1, 1);
    lookup_k(2);
    if (final >= 0) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int c = 0; c < DC; ++c) s_product(sc[0][kb], k_operand(0, kb, c), c);
      round(Int<1>{}, 0, Int<0>{});
    } else {
      turn(true, 0, 0);
    }
    int it = 1;
#pragma unroll 1
    for (; it < rounds && it <= final + 1; it += 2) {       // (in pairs: an odd one at the end is a round that nobody sees)
      round(Int<0>{}, it, Int<1>{});
      if (it > final) {
        ++it;
        break;
      }
      round(Int<0>{}, it + 1, Int<0>{});
    }
#pragma unroll 1
    for (; it <= rounds / 2 * 2; ++it) turn(false, it, it & 1);
    arrive();
    clear_tail(rounds / 2 * 2, 0);
    if (rounds / 2 * 2 <= final) {
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int db = 0; db < DB; ++db) o_product(o[db], v_operand(0, a, db), pb[0][a]);
    }
  } else {
    f32x16_t sc[2];
    u32x4_t pb[4];
    const auto round = [&](int it, int cur) {
      arrive();
      clear_tail(it, cur);
      request_k(it + 1, cur ^ 1);
      request_v(it + 1, cur ^ 1);
      lookup_k(it + 2);
      lookup_v(it + 2);
      if (it > final || early(it)) return;
      begin(it);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int c = 0; c < DC; ++c) s_product(sc[kb], k_operand(cur, kb, c), c);
      static_for<0, UNITS>([&](auto u) { work(u, sc, pb); });
      rescale();
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int db = 0; db < DB; ++db) o_product(o[db], v_operand(cur, a, db), pb[a]);
    };
#pragma unroll 1
    for (int it = 0; it < rounds; ++it) round(it, it & 1);
  }

  // ---- out: lane holds columns 32 db + 8 a + 4 hi .. + 3 of query ql
  if constexpr (D == 128) {
    typedef __attribute__((ext_vector_type(4))) __bf16 b4_t;
    const float inv = 1.f / (l + other_half(l));
    if (!valid) return;
    bf16_t* op = (bf16_t*)A.out + (row * H + h) * DV + 4 * hi;
    const bf16_t* gp = A.gate ? (const bf16_t*)A.gate + row * A.gate_stride + (int64_t)h * A.gate_w : nullptr;
    const auto gated = [](float x, float gv) { return x * sigmoid_hw(gv); };
    const bool wide = gp && A.gate_w != 1;
    const float ginv = gp && !wide ? gated(inv, (float)gp[0]) : inv;
    const bool quads = wide && ((A.gate_stride & 3) == 0) && ((uintptr_t)A.gate & 7) == 0;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      b4_t gv[4];
      if (quads) {
#pragma unroll
        for (int a = 0; a < 4; ++a) gv[a] = *(const b4_t*)(gp + 32 * db + 8 * a + 4 * hi);
      } else if (wide) {
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
          for (int i = 0; i < 4; ++i) gv[a][i] = gp[32 * db + 8 * a + 4 * hi + i];
      }
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        b4_t v;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float x = o[db][4 * a + i] * ginv;
          if (wide) x = gated(x, (float)gv[a][i]);
          v[i] = (bf16_t)x;
        }
        *(b4_t*)(op + 32 * db + 8 * a) = v;
      }
    }
  } else if constexpr (HEADS == 2) {
    // W_uv,h [128][192] times the latent result, which is its operand as it is: a lane holds entries 16 s + 8 hi .. + 7 of its query for each k-step s, since the value tile's columns
    // lie in that order. The weights come in pieces of 32 rows x 64 entries through four places of the wavefront's own, 16-byte unit u of row r at u ^ ((r >> 1) & 7).
    // A launch of its own, which reads the latent results again, takes 34 us for 14,200 rows of 16 heads; four layers of 14,200 tokens 3,024 us with it, 2,899 so (a workgroup's end 4.3 us
    // either way: weights from L2 here, a row 1.5 times as long there).
    constexpr int OUT = 128, PIECE = 32 * 128, PIECES = OUT / 32 * (DV / 64);
    int out_tid = threadIdx.x;                        // (as if new, as below)
    asm volatile("" : "+v"(out_tid));
    const int ol = out_tid & 63, oq = ol & 31, oh = ol >> 5, ow = __builtin_amdgcn_readfirstlane(out_tid >> 6);
    const int live = len - rel0 < 32 ? len - rel0 : 32;
    const float inv = 1.f / (l + other_half(l));
    const bf16_t* gp = A.gate ? (const bf16_t*)A.gate + (int64_t)(row0 + (live > 0 ? rel0 : len - 1)) * A.gate_stride + h : nullptr;      // (nobody's queries: a row that is there)
    const float ginv = gp ? inv * sigmoid_hw((float)gp[(int64_t)(oq < live ? oq : 0) * A.gate_stride]) : inv;
    char* at = lds + ow * 4 * PIECE;
    const char* wbase = (const char*)A.uv + (int64_t)h * OUT * DV * 2;
    const uint32_t wrow = (uint32_t)(ol >> 3) * DV * 2, woff[2] = {wrow + ((ol & 7) ^ (ol >> 4)) * 16, wrow + ((ol & 7) ^ (4 + (ol >> 4))) * 16};
    const auto bring = [&](auto piece) {
      constexpr int p = decltype(piece)::value;
#pragma unroll
      for (int i = 0; i < 4; ++i) dma16(wbase + ((p / 3 * 32 + i * 8) * DV + p % 3 * 64) * 2 + woff[i & 1], at + p % 4 * PIECE + i * 1024);
    };
    bf16x8_t x[12];
#pragma unroll
    for (int s = 0; s < 12; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) x[s][e] = (bf16_t)(o[s / 2][s % 2 * 8 + e] * ginv);
    __syncthreads();                                  // (the tiles have been read)
    static_for<0, 4>(bring);
    f32x16_t y[OUT / 32];
    static_for<0, PIECES>([&](auto piece) {
      constexpr int p = decltype(piece)::value, left = PIECES - 1 - p < 3 ? PIECES - 1 - p : 3;       // pieces that may still be on their way
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0x0F70 + left * 4);  // vmcnt(4 left)
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      bf16x8_t w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = *(const bf16x8_t*)(at + p % 4 * PIECE + oq * 128 + (((2 * j + oh) ^ ((oq >> 1) & 7)) << 4));
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x16_t zero = {};
        y[p / 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[j], x[p % 3 * 4 + j], p % 3 == 0 && j == 0 ? zero : y[p / 3], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (p + 4 < PIECES) bring(Int<p + 4>{});
    });
    typedef __attribute__((ext_vector_type(4))) __bf16 b4_t;
#pragma unroll
    for (int vb = 0; vb < OUT / 32; ++vb)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        b4_t v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (bf16_t)y[vb][4 * a + i];
        *(b4_t*)(at + oq * OUT * 2 + (((4 * vb + a) ^ (oq & 15)) << 4) + oh * 8) = v;
      }
    bf16_t* op = (bf16_t*)A.out + ((int64_t)(row0 + rel0) * H + h) * OUT + (ol & 15) * 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = i * 4 + (ol >> 4);
      const bf16x8_t v = *(const bf16x8_t*)(at + r * OUT * 2 + (((ol & 15) ^ (r & 15)) << 4));
      if (r < live) *(bf16x8_t*)(op + (int64_t)r * H * OUT) = v;
    }
  } else {
    // Through LDS in 32 bits, so that rows (and the gate's) are read and written as they lie, 16 bytes a lane: one workgroup of eight wavefronts has the compute unit to itself, nothing
    // hides what comes behind its rounds (14,200 tokens in 9 prompts, 16 heads, window 1,024 / causal, 251 / 275 us before, 234 / 256 so; 128-wide heads, gated,
    // 323 and 333).
    constexpr int OP = NW * 32 * DV * 4 <= 2 * TILE ? 1 : 2, OC = DV / OP, OU = OC / 8;        // passes; columns of one; units of 8 columns
    static_assert(NW * 32 * OC * 4 <= 2 * TILE && DB % OP == 0 && OC % 32 == 0, "a pass of all wavefronts' rows fits the tiles");
    int out_tid = threadIdx.x;                        // (as if new: addresses of the queries' rows would be kept over the loop otherwise, which has no register left)
    asm volatile("" : "+v"(out_tid));
    const int ol = out_tid & 63, oq = ol & 31, oh = ol >> 5, ow = __builtin_amdgcn_readfirstlane(out_tid >> 6);
    const int live = len - rel0 < 32 ? len - rel0 : 32;                           // (none: a wavefront of nobody's queries)
    const float inv = 1.f / (l + other_half(l));
    const bf16_t* gp = A.gate ? (const bf16_t*)A.gate + (int64_t)(row0 + (live > 0 ? rel0 : len - 1)) * A.gate_stride + (int64_t)h * A.gate_w : nullptr;      // (nobody's queries: a row that is there)
    const bool wide = gp && A.gate_w != 1, units = wide && (A.gate_stride & 7) == 0 && ((uintptr_t)gp & 15) == 0;
    const float ginv = gp && !wide ? inv * sigmoid_hw((float)gp[(int64_t)(oq < live ? oq : 0) * A.gate_stride]) : inv;
    bf16_t* op = (bf16_t*)A.out + ((int64_t)(row0 + rel0) * H + h) * DV;
    char* at = lds + ow * 32 * OC * 4;
    __syncthreads();                                  // (the tiles have been read)
#pragma unroll
    for (int p = 0; p < OP; ++p) {
      bf16x8_t gv[OU / 2];
      if (units) {
#pragma unroll
        for (int i = 0; i < OU / 2; ++i) {
          const int x = i * 64 + ol, r = x / OU, u = x % OU;
          gv[i] = *(const bf16x8_t*)(gp + (int64_t)(r < live ? r : 0) * A.gate_stride + p * OC + u * 8);
        }
      }
#pragma unroll
      for (int db = 0; db < DB / OP; ++db)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          f32x4_t v;
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = o[p * (DB / OP) + db][4 * a + i] * ginv;
          *(f32x4_t*)(at + oq * OC * 4 + (((8 * db + 2 * a + oh) ^ (oq & 7)) << 4)) = v;
        }
#pragma unroll
      for (int i = 0; i < OU / 2; ++i) {
        const int x = i * 64 + ol, r = x / OU, u = x % OU;
        const f32x4_t v0 = *(const f32x4_t*)(at + r * OC * 4 + (((2 * u) ^ (r & 7)) << 4)), v1 = *(const f32x4_t*)(at + r * OC * 4 + (((2 * u + 1) ^ (r & 7)) << 4));
        bf16x8_t y;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float f = e < 4 ? v0[e] : v1[e - 4];
          if (wide) f *= sigmoid_hw((float)(units ? gv[i][e] : gp[(int64_t)(r < live ? r : 0) * A.gate_stride + p * OC + u * 8 + e]));
          y[e] = (bf16_t)f;
        }
        if (r < live) *(bf16x8_t*)(op + (int64_t)r * H * DV + p * OC + u * 8) = y;
      }
    }
  }
}

struct PromptGrid {
  int hw;                                           // heads of a workgroup
  int64_t tiles, rows;                              // query tiles, heads / hw
};
inline PromptGrid prompt_grid(const WindowAttnArgs& a, int nw) {
  const int hpg = a.H / a.G;
  PromptGrid p;
  p.hw = hpg % nw == 0 ? nw : (hpg % 4 == 0 ? 4 : (hpg % 2 == 0 ? 2 : 1));
  p.rows = a.H / p.hw;
  // an upper bound: every portion may end with a partial tile, and every tile holds a token (a workgroup without one takes a live
  // one's place: 64 single tokens, 8 heads over each of two, capped, 38 us with 8 such workgroups behind 256, 26 without)
  p.tiles = a.n / ((nw / p.hw) * 32) + a.nseq;
  if (p.tiles > a.n) p.tiles = a.n;
  return p;
}

template <int D, int DV, int NW, bool EXT, int HEADS = 0>
int launch_prompt(WindowAttnArgs a, hipStream_t stream) {
  const PromptGrid p = prompt_grid(a, NW);
  a.hw = p.hw;
  a.bs_shift = __builtin_ctz(a.block_size);
  constexpr int TILE = 64 * D * 2 + DV * 128, LDS = TILE + (HEADS ? NW * 32 * DV * 2 : TILE);      // (HEADS: queries of 128 + 64 entries, as wide as a value)
  const auto kernel = window_attn_prompt_kernel<D, DV, NW, EXT, HEADS>;
  NVS_LDS_ROOM(kernel, LDS, "nvs_window_attn");
  kernel<<<dim3((unsigned)p.tiles, (unsigned)p.rows), dim3(64 * NW), LDS, stream>>>(a);
  return nvs_check_launch("nvs_window_attn (prompts)");
}

}  // namespace
