// Gated feed-forward activations and routed mixtures of experts.
//
// A routed layer runs as: router (moe_router.hip: 32-bit logits, softmax, choice scores, group limit,
// top-k, weights; past 64 entries a 32-bit library product and the route kernel here) -> plan kernel (pairs (token, choice) sorted by expert into row tiles, every expert's rows padded to a whole
// tile) -> grouped product gate|up with the activation in its epilogue -> grouped product down -> combine kernel (weighted sum
// of a token's choices, pass-through experts, the gated shared expert). Nothing comes back to the host in between, so the
// sequence can be captured in a hipGraph; the order in which pairs land inside an expert's rows is arbitrary but no sum depends
// on it (a row is computed on its own, and a token's choices are added in the order of its choices).
#include "seq_common.h"
#include <type_traits>

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;

constexpr int MAX_EXPERTS = 1024;

// ungated products: mode 2 squares the positive part (the input rows are then gathered by token, as for a gated product)
__device__ __forceinline__ float plain_value(float v, int mode) {
  if (mode != 2) return v;
  v = fmaxf(v, 0.f);
  return v * v;
}

template <typename T>
__global__ void glu_act_kernel(const T* __restrict__ gu, int64_t stride, int ff, int kind, float limit, float alpha, int64_t n,
                               T* __restrict__ out) {
  const int64_t total = n * ff;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = i / ff;
    const int c = (int)(i - t * ff);
    stf(out + i, glu_value(ldf(gu + t * stride + c), kind == 2 ? 0.f : ldf(gu + t * stride + ff + c), kind, limit, alpha));
  }
}

// the same, eight columns per access (ff a multiple of 8, every row aligned for it, fewer than 2^31 accesses)
template <typename T>
__global__ __launch_bounds__(256) void glu_act_rows8_kernel(const T* __restrict__ gu, int64_t stride, int ff8, int kind, float limit, float alpha,
                                                            int total, T* __restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int t = i / ff8, c = (i - t * ff8) * 8;
  float g[8], u[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  ldp<8>(gu + t * stride + c, g);
  if (kind != 2) ldp<8>(gu + t * stride + (int64_t)ff8 * 8 + c, u);
#pragma unroll
  for (int e = 0; e < 8; ++e) g[e] = glu_value(g[e], u[e], kind, limit, alpha);
  stp<8>(out + (int64_t)i * 8, g);
}

// ---- routing without a router: a table row per token id names the token's experts, all with the same weight ----------
__global__ void moe_table_route_kernel(const int64_t* __restrict__ tokens, const int32_t* __restrict__ table, int64_t pairs, int top,
                                       float weight, int32_t* __restrict__ ids, float* __restrict__ wts) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= pairs) return;
  const int64_t t = i / top;
  ids[i] = table[tokens[t] * top + (i - t * top)];
  wts[i] = weight;
}

// ---- routing: one wavefront per token, a lane holds entries lane, lane + 64, ... of the token's scores ---------------
constexpr int ROUTE_PER_LANE = MAX_EXPERTS / 64;

__global__ void moe_route_kernel(const float* __restrict__ z, int64_t z_stride, const float* __restrict__ correction, int total,
                                 int top, int count, int keep, float scale, int score, int renorm, int32_t* __restrict__ ids,
                                 float* __restrict__ wts) {
  const int64_t t = blockIdx.x;
  const int lane = threadIdx.x;
  const int per = total / count;
  float s[ROUTE_PER_LANE], c[ROUTE_PER_LANE];
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < ROUTE_PER_LANE; ++i) {
    const int e = lane + 64 * i;
    s[i] = e < total ? z[t * z_stride + e] : -INFINITY;
    mx = fmaxf(mx, s[i]);
  }
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < ROUTE_PER_LANE; ++i) {
    const int e = lane + 64 * i;
    if (score == 1) s[i] = e < total ? 1.f / (1.f + expf(-s[i])) : 0.f;      // sigmoid: every entry on its own
    else s[i] = e < total ? expf(s[i] - mx) : 0.f;
    sum += s[i];
  }
  sum = score == 1 ? 1.f : wave_sum(sum);
#pragma unroll
  for (int i = 0; i < ROUTE_PER_LANE; ++i) {
    const int e = lane + 64 * i;
    s[i] = s[i] / sum;
    c[i] = e < total ? s[i] + (correction ? correction[e] : 0.f) : -INFINITY;      // the choice score; weights use s
  }
  if (count > 1) {
    // a group's score is its best choice score; entries outside the `keep` best groups cannot be chosen. Lane l holds the
    // score of group l (count <= 64) and ranks it: the number of groups that beat it, a lower index winning a tie.
    float mine = -INFINITY;
    for (int g = 0; g < count; ++g) {
      float v = -INFINITY;
#pragma unroll
      for (int i = 0; i < ROUTE_PER_LANE; ++i) {
        const int e = lane + 64 * i;
        if (e < total && e / per == g) v = fmaxf(v, c[i]);
      }
      v = wave_max(v);
      if (lane == g) mine = v;
    }
    int better = 0;
    for (int g = 0; g < count; ++g) {
      const float v = __shfl(mine, g, 64);
      if (g != lane && (v > mine || (v == mine && g < lane))) ++better;
    }
    const int dropped = better >= keep;
    for (int g = 0; g < count; ++g) {
      if (__shfl(dropped, g, 64) == 0) continue;
#pragma unroll
      for (int i = 0; i < ROUTE_PER_LANE; ++i) {
        const int e = lane + 64 * i;
        if (e < total && e / per == g) c[i] = -INFINITY;
      }
    }
  }
  float chosen_s = 0.f;                             // lane k: the score of choice k
  int chosen_e = 0;
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int at = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < ROUTE_PER_LANE; ++i) {
      const int e = lane + 64 * i;
      if (e < total && (c[i] > best)) best = c[i], at = e;      // (entries of a lane ascend: the first best stays)
    }
    const float wbest = wave_max(best);
    int cand = best == wbest ? at : 0x7fffffff;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const int other = __shfl_xor(cand, o, 64);
      cand = other < cand ? other : cand;
    }
    if (cand == 0x7fffffff) cand = 0;               // (fewer choosable entries than choices: cannot happen with valid sizes)
    float sv = 0.f;
#pragma unroll
    for (int i = 0; i < ROUTE_PER_LANE; ++i) {
      const int e = lane + 64 * i;
      if (e == cand) sv = s[i], c[i] = -INFINITY;
    }
    sv = wave_sum(sv);                              // one lane holds it
    if (lane == k) chosen_s = sv, chosen_e = cand;
  }
  const float denom = renorm ? wave_sum(lane < top ? chosen_s : 0.f) + 1e-20f : 1.f;
  if (lane < top) {
    ids[t * top + lane] = chosen_e;
    wts[t * top + lane] = chosen_s / denom * scale;
  }
}

// ---- plan: one workgroup sorts the pairs by expert --------------------------------------------------------------------
// offs[e] = the rows of the experts before e, each expert's filled up to whole tiles (offs[experts]: all rows); 1,024 threads, an
// expert each (one thread adding 256 experts up took 12 of the plan's 16 us; for up to 16 it is the faster way, 2.6 us a plan of 4
// experts against 3.2)
__device__ __forceinline__ void expert_offsets(const int* counts, int experts, int tm, int* offs, int* sums) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (experts <= 16) {
    if (tid == 0) {
      int o = 0;
      for (int e = 0; e < experts; ++e) {
        offs[e] = o;
        o += (counts[e] + tm - 1) / tm * tm;
      }
      offs[experts] = o;
    }
    __syncthreads();
    return;
  }
  const int own = tid < experts ? (counts[tid] + tm - 1) / tm * tm : 0;
  int v = own;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int up = __shfl_up(v, o, 64);
    if (lane >= o) v += up;
  }
  if (lane == 63) sums[wave] = v;
  __syncthreads();
  for (int k = 0; k < wave; ++k) v += sums[k];
  if (tid < experts) {
    offs[tid] = v - own;
    if (tid == experts - 1) offs[experts] = v;
  }
  __syncthreads();
}

__global__ __launch_bounds__(1024) void moe_plan_kernel(const int32_t* __restrict__ ids, int64_t pairs, int top, int experts, int tm,
                                                        int64_t cap, int32_t* __restrict__ tile_expert, int32_t* __restrict__ row_token,
                                                        int32_t* __restrict__ pair_row) {
  __shared__ int counts[MAX_EXPERTS];
  __shared__ int offs[MAX_EXPERTS + 1], sums[16];
  const int tid = threadIdx.x, nt = blockDim.x;
  for (int e = tid; e < experts; e += nt) counts[e] = 0;
  for (int64_t r = tid; r < cap; r += nt) row_token[r] = -1;
  __syncthreads();
  for (int64_t i = tid; i < pairs; i += nt) {
    const int e = ids[i];
    if (e < experts) atomicAdd(&counts[e], 1);
  }
  __syncthreads();
  expert_offsets(counts, experts, tm, offs, sums);
  for (int64_t tile = tid; tile < cap / tm; tile += nt) {
    const int64_t r = tile * tm;
    int e = -1;
    if (r < offs[experts]) {
      int lo = 0, hi = experts - 1;                 // the last expert whose offset is <= r and who has rows
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (offs[mid] <= r) lo = mid; else hi = mid - 1;
      }
      e = lo;
    }
    tile_expert[tile] = e;
  }
  for (int e = tid; e < experts; e += nt) counts[e] = offs[e];         // now the cursors
  __syncthreads();
  for (int64_t i = tid; i < pairs; i += nt) {
    const int e = ids[i];
    int r = -1;
    if (e < experts) {
      r = atomicAdd(&counts[e], 1);
      row_token[r] = (int32_t)(i / top);
    }
    pair_row[i] = r;
  }
}

// The same by many workgroups, PLAN_PAIRS pairs each: one pass counts (every pair's place among its workgroup's pairs of that expert
// goes to pair_row, the counts to scratch [workgroups][experts]), the next adds up all counts before its own and places its pairs.
// One workgroup is bound by its own few loads in flight and its atomics: 54,200 pairs, 32 experts 33 us, here 7 (256 experts: 45, 10).
constexpr int PLAN_PAIRS = 2048;
__global__ __launch_bounds__(1024) void moe_plan_count_kernel(const int32_t* __restrict__ ids, int64_t pairs, int experts, int64_t cap,
                                                              int32_t* __restrict__ row_token, int32_t* __restrict__ pair_row,
                                                              int32_t* __restrict__ scratch) {
  __shared__ int counts[MAX_EXPERTS];
  const int tid = threadIdx.x;
  for (int e = tid; e < experts; e += 1024) counts[e] = 0;
  const int64_t share = (cap + gridDim.x - 1) / gridDim.x, r1 = (blockIdx.x + 1) * share < cap ? (blockIdx.x + 1) * share : cap;
  for (int64_t r = blockIdx.x * share + tid; r < r1; r += 1024) row_token[r] = -1;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < PLAN_PAIRS / 1024; ++k) {
    const int64_t i = (int64_t)blockIdx.x * PLAN_PAIRS + k * 1024 + tid;
    if (i >= pairs) break;
    const int e = ids[i];
    pair_row[i] = e < experts ? atomicAdd(&counts[e], 1) : -1;
  }
  __syncthreads();
  for (int e = tid; e < experts; e += 1024) scratch[(int64_t)blockIdx.x * experts + e] = counts[e];
}

__global__ __launch_bounds__(1024) void moe_plan_place_kernel(const int32_t* __restrict__ ids, int64_t pairs, int top, int experts, int tm,
                                                              int64_t cap, int32_t* __restrict__ tile_expert, int32_t* __restrict__ row_token,
                                                              int32_t* __restrict__ pair_row, const int32_t* __restrict__ scratch) {
  __shared__ int total[MAX_EXPERTS], before[MAX_EXPERTS], offs[MAX_EXPERTS + 1], sums[16];
  const int tid = threadIdx.x, b = blockIdx.x, blocks = gridDim.x;
  for (int e = tid; e < experts; e += 1024) total[e] = before[e] = 0;
  __syncthreads();
  for (int u = tid; u < blocks * experts; u += 1024) {
    const int o = u / experts, e = u - o * experts, c = scratch[u];
    if (c) {
      atomicAdd(&total[e], c);
      if (o < b) atomicAdd(&before[e], c);
    }
  }
  __syncthreads();
  expert_offsets(total, experts, tm, offs, sums);
  for (int64_t tile = (int64_t)b * 1024 + tid; tile < cap / tm; tile += (int64_t)blocks * 1024) {
    const int64_t r = tile * tm;
    int e = -1;
    if (r < offs[experts]) {
      int lo = 0, hi = experts - 1;                 // the last expert whose offset is <= r and who has rows
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (offs[mid] <= r) lo = mid; else hi = mid - 1;
      }
      e = lo;
    }
    tile_expert[tile] = e;
  }
#pragma unroll
  for (int k = 0; k < PLAN_PAIRS / 1024; ++k) {
    const int64_t i = (int64_t)b * PLAN_PAIRS + k * 1024 + tid;
    if (i >= pairs) break;
    const int e = ids[i];
    if (e >= experts) continue;
    const int r = offs[e] + before[e] + pair_row[i];
    row_token[r] = (int32_t)(i / top);
    pair_row[i] = r;
  }
}

// ---- grouped products --------------------------------------------------------------------------------------------------
// out[r, f] = sum_k X[src(r), k] * W[e(r)][f, k] for the rows r of a tile (all of one expert). GLU: W holds gate rows
// [0, nout) then up rows [nout, 2 nout) and the output is act(gate) * up; src(r) = row_token[r] (the token's input row),
// otherwise src(r) = r. Rows with row_token[r] < 0 are padding.

// plain form, any type and size: a thread owns one row and four features
template <typename T, bool GLU>
__global__ __launch_bounds__(256) void moe_gemm_kernel(const T* __restrict__ X, int64_t ldx, const T* __restrict__ W, int nout, int K,
                                                       const int32_t* __restrict__ tile_expert, const int32_t* __restrict__ row_token,
                                                       int tm, T* __restrict__ out, int64_t ldo, int mode) {
  const int tiles_per = tm / 16;
  const int tile = blockIdx.x / tiles_per;
  const int e = tile_expert[tile];
  if (e < 0) return;
  const int64_t r = (int64_t)blockIdx.x * 16 + (threadIdx.x & 15);
  const int tok = row_token[r];
  if (tok < 0) return;
  const int64_t src = (GLU || mode == 2) ? tok : r;
  const T* xr = X + src * ldx;
  const T* We = W + (int64_t)e * (GLU ? 2 : 1) * nout * K;
  const int f0 = blockIdx.y * 64 + (threadIdx.x >> 4) * 4;
  float ag[4] = {0.f, 0.f, 0.f, 0.f}, au[4] = {0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < K; ++k) {
    const float x = ldf(xr + k);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (f0 + i < nout) {
        ag[i] += x * ldf(We + (int64_t)(f0 + i) * K + k);
        if (GLU) au[i] += x * ldf(We + (int64_t)(nout + f0 + i) * K + k);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (f0 + i < nout) stf(out + r * ldo + f0 + i, GLU ? glu_value(ag[i], au[i], 0, 0.f, 0.f) : plain_value(ag[i], mode));
}

// matrix-core form (bf16, K % 8 == 0, 16-byte aligned rows). Computed transposed, C^T[features x rows] = W X^T with
// v_mfma_f32_16x16x32_bf16: the A operand is 16 weight rows x 32 of k, the B operand 16 input rows x 32 of k, both 16-byte
// loads straight from memory; a lane ends up with four consecutive features of one row (an 8-byte store). A workgroup of four
// wavefronts covers 16 MT rows x 128 features: every wavefront 32 features (FT = 2 blocks) for all the rows.
template <int MT, bool GLU>
__global__ __launch_bounds__(256) void moe_gemm_mfma_kernel(const bf16_t* __restrict__ X, int64_t ldx, const bf16_t* __restrict__ W, int nout,
                                                            int K, const int32_t* __restrict__ tile_expert,
                                                            const int32_t* __restrict__ row_token, bf16_t* __restrict__ out, int64_t ldo, int mode) {
  constexpr int FT = 2, NG = GLU ? 2 : 1;
  const int e = tile_expert[blockIdx.x];
  if (e < 0) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, lk = (lane >> 4) * 8;
  const int64_t row0 = (int64_t)blockIdx.x * (16 * MT);
  const bf16_t* xp[MT];
  bool xok[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int64_t r = row0 + mt * 16 + li;
    const int tok = row_token[r];
    xok[mt] = tok >= 0;
    xp[mt] = X + (xok[mt] ? ((GLU || mode == 2) ? (int64_t)tok : r) : 0) * ldx + lk;
  }
  const bf16_t* We = W + (int64_t)e * NG * nout * K;
  const int fbase = blockIdx.y * (64 * FT) + wave * (16 * FT);
  const bf16_t* wp[FT];
  bool wok[FT];
#pragma unroll
  for (int ft = 0; ft < FT; ++ft) {
    const int f = fbase + ft * 16 + li;
    wok[ft] = f < nout;
    wp[ft] = We + (int64_t)(wok[ft] ? f : 0) * K + lk;
  }
  f32x4_t acc[NG][FT][MT];
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int ft = 0; ft < FT; ++ft)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[g][ft][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const bf16x8_t zero8 = __builtin_bit_cast(bf16x8_t, u32x4_t{0u, 0u, 0u, 0u});
  for (int k0 = 0; k0 < K; k0 += 32) {
    const bool kin = k0 + lk < K;
    bf16x8_t xb[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) xb[mt] = (kin && xok[mt]) ? *(const bf16x8_t*)(xp[mt] + k0) : zero8;
#pragma unroll
    for (int ft = 0; ft < FT; ++ft) {
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const bf16x8_t wa = (kin && wok[ft]) ? *(const bf16x8_t*)(wp[ft] + (int64_t)g * nout * K + k0) : zero8;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[g][ft][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa, xb[mt], acc[g][ft][mt], 0, 0, 0);
      }
    }
  }
  // lane: row li of the tile block, features fbase + 16 ft + 4 (lane >> 4) + 0..3
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    if (!xok[mt]) continue;
    const int64_t r = row0 + mt * 16 + li;
#pragma unroll
    for (int ft = 0; ft < FT; ++ft) {
      const int f = fbase + ft * 16 + (lane >> 4) * 4;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (f + i < nout) {
          const float v = GLU ? glu_value(acc[0][ft][mt][i], acc[NG - 1][ft][mt][i], 0, 0.f, 0.f) : plain_value(acc[0][ft][mt][i], mode);
          out[r * ldo + f + i] = (bf16_t)v;
        }
      }
    }
  }
}

// LDS-tiled matrix-core form for steps with many rows per expert (tiles of 128 rows). A workgroup of four wavefronts computes
// 128 rows x 128 features (GLU: gate and up of the same 64 features; 128 weight rows either way) in steps of 64 along k: all
// threads load the step's operands with 16-byte loads — the NEXT step's loads are issued before the current step is computed —
// into LDS as [row][64 + 8]; a wavefront owns 64 rows x 64 weight rows (4 x 4 MFMA tiles) and reads its operands as 16-byte LDS
// reads: 16 reads for 32 MFMAs per step. The grid is one-dimensional and XCD-aware: workgroups are dealt to the eight XCDs
// round-robin, so workgroup id -> (id % 8) * per_xcd + id / 8 gives every XCD a CONTIGUOUS run of tiles, ordered feature tile
// major / row tile minor: consecutive tiles of an XCD share a weight tile (all row tiles of one expert), which its L2 then serves.
template <bool GLU>
__global__ __launch_bounds__(256) void moe_gemm_tiled_kernel(const bf16_t* __restrict__ X, int64_t ldx, const bf16_t* __restrict__ W, int nout,
                                                             int K, const int32_t* __restrict__ tile_expert,
                                                             const int32_t* __restrict__ row_token, int tiles_m, int tiles_n, int tiles_per,
                                                             bf16_t* __restrict__ out, int64_t ldo, int mode) {
  constexpr int BM = 128, BW = 128, BK = 64, LDK = BK + 8, NG = GLU ? 2 : 1, FB = 4 / NG, BN = BW / NG;   // BN features per tile
  __shared__ __attribute__((aligned(16))) bf16_t Xs[BM][LDK];
  __shared__ __attribute__((aligned(16))) bf16_t Ws[BW][LDK];      // GLU: rows [0, 64) gate, [64, 128) up of the tile's features
  const int per_xcd = gridDim.x / 8;
  const int logical = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (logical >= tiles_m * tiles_n) return;
  const int rt = logical % tiles_m, ft = logical / tiles_m;
  const int e = tile_expert[rt / tiles_per];
  if (e < 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lk = (lane >> 4) * 8;
  const int wm = wave & 1, wn = wave >> 1;
  const int64_t row0 = (int64_t)rt * BM;
  const bf16_t* We = W + (int64_t)e * NG * nout * K;
  // staging: unit u = tid + 256 i -> (row u >> 3, 8 elements of k at (u & 7) * 8); four units of each operand per thread
  const int sk = (tid & 7) * 8, sr = tid >> 3;
  const bf16_t* xsrc[4];
  const bf16_t* wsrc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = sr + 32 * i;
    const int tok = row_token[row0 + r];
    xsrc[i] = tok >= 0 ? X + ((GLU || mode == 2) ? (int64_t)tok : row0 + r) * ldx + sk : nullptr;
    const int g = r / BN, f = ft * BN + r % BN;
    wsrc[i] = f < nout ? We + ((int64_t)g * nout + f) * K + sk : nullptr;
  }
  const u32x4_t zero4 = u32x4_t{0u, 0u, 0u, 0u};
  u32x4_t xr[4], wr[4];
  auto fetch = [&](int k0) {
    const bool kin = k0 + sk < K;
#pragma unroll
    for (int i = 0; i < 4; ++i) xr[i] = (kin && xsrc[i]) ? *(const u32x4_t*)(xsrc[i] + k0) : zero4;
#pragma unroll
    for (int i = 0; i < 4; ++i) wr[i] = (kin && wsrc[i]) ? *(const u32x4_t*)(wsrc[i] + k0) : zero4;
  };
  // accumulators: weight-row block wb of this wavefront's 64 weight rows x row block rb. GLU: a wavefront's 64 weight rows are
  // 32 gate rows and the 32 up rows of the SAME features (wb 0, 1 gate; 2, 3 up), so the activation needs no exchange.
  f32x4_t acc[4][4];
#pragma unroll
  for (int wb = 0; wb < 4; ++wb)
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) acc[wb][rb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  int wrow[4];                                      // LDS row of this lane's operand for weight-row block wb
#pragma unroll
  for (int wb = 0; wb < 4; ++wb) wrow[wb] = GLU ? (wb / FB) * BN + wn * 32 + (wb % FB) * 16 + li : wn * 64 + wb * 16 + li;
  fetch(0);
  for (int k0 = 0; k0 < K; k0 += BK) {
    __syncthreads();                                // the previous step's readers are done
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      *(u32x4_t*)&Xs[sr + 32 * i][sk] = xr[i];
      *(u32x4_t*)&Ws[sr + 32 * i][sk] = wr[i];
    }
    __syncthreads();
    if (k0 + BK < K) fetch(k0 + BK);
#pragma unroll
    for (int kk = 0; kk < BK; kk += 32) {
      bf16x8_t xb[4];
#pragma unroll
      for (int rb = 0; rb < 4; ++rb) xb[rb] = *(const bf16x8_t*)&Xs[wm * 64 + rb * 16 + li][kk + lk];
#pragma unroll
      for (int wb = 0; wb < 4; ++wb) {
        const bf16x8_t wa = *(const bf16x8_t*)&Ws[wrow[wb]][kk + lk];
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) acc[wb][rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa, xb[rb], acc[wb][rb], 0, 0, 0);
      }
    }
  }
  // lane: row li of row block rb; features 16 fb + 4 (lane >> 4) + 0..3 of its wavefront's 64 (GLU: 32)
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) {
    const int64_t r = row0 + wm * 64 + rb * 16 + li;
    if (row_token[r] < 0) continue;
#pragma unroll
    for (int fb = 0; fb < FB; ++fb) {
      const int f = ft * BN + wn * (16 * FB) + fb * 16 + (lane >> 4) * 4;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (f + i < nout) {
          const float v = GLU ? glu_value(acc[fb][rb][i], acc[GLU ? fb + FB : fb][rb][i], 0, 0.f, 0.f) : plain_value(acc[fb][rb][i], mode);
          out[r * ldo + f + i] = (bf16_t)v;
        }
      }
    }
  }
}

// Pipelined matrix-core form (bf16 with K % 64 == 0, 32-bit with K % 32 == 0: rows whose 128-byte pieces are whole). A workgroup of four
// wavefronts computes BM = 16 RB (4 / WN) rows x BW = 16 WB WN weight rows (GLU: gate and up of the same BW / 2 features) in steps of 128
// bytes along k; a wavefront owns 16 RB rows x 16 WB weight rows (WN wavefronts side by side along the weight rows).
//
// The operands go from memory straight into LDS (16 bytes per lane, no registers) through a ring of ST buffers. A step is two halves of
// 64 bytes of k: while a half is multiplied the next half's operands are read from LDS; in the middle of a step every wavefront holds the rest
// of the step's buffer in registers, so behind the one barrier of a step the step ST ahead is requested into it. Requests and reads
// are issued between groups of MFMAs, where the matrix pipe hides them (one wavefront per SIMD has nobody else to). The barrier waits only
// for the requests of the next step. A row's piece is 128 bytes of LDS; 16-byte unit c of row r sits at c ^ ((r >> 1) & 7), so
// the 16 rows an operand read touches lie on 16 different bank quads (the requests fetch the units in that order; the direct path
// could not write padding). The MFMAs are written out with accumulators in the accumulation registers and operands in the vector registers:
// left to itself the compiler moves one or the other between the two files in the loop.
//
// 16-bit tiles of 256 rows are gemm_tiles.h's, but for rows and results that its tiles_fit leaves out; figures of 256 rows below are this kernel's. As many workgroups as fit on the chip at once, and each goes on from tile to tile: the last ST steps of a tile ask for the first ones of the next, whose
// rows were looked up a whole tile earlier, so no tile but the first waits for its plan, its addresses and its operands, and the stores drain behind the next
// tile's first steps. Full tiles of 256 rows x 256 weight rows, us per tile at k = 256 / 1024 / 4096, before and after (the products alone take 5.9 / 23.6 /
// 94): gated 22.4 / 42.2 / 111.8 -> 13.1 / 32.0 / 106.9, plain 20.7 / 41.0 / 111.0 -> 14.7 / 36.8 / 109.0; tiles of 128 rows, gated 12.5 / 22.3 / 62.5 -> 7.3 / 17.4 / 58.3; of
// 64 rows, two at a time 9.7 / 20.5 / 68.0 -> 7.5 / 18.6 / 64.8. Of that the tiles' overlap gives 2 to 3 us; the SiLU of 128 values per lane on the hardware's exponential
// and reciprocal 3 to 5 (it took 30 instructions a value, and no product runs beside it); and the results' way through LDS, so that a store writes whole
// rows of 128 or 256 bytes instead of 32 bytes in each of 16 rows, 2 to 5.
//
// Workgroups go to the eight XCDs round-robin; each XCD takes units of 8 row tiles x 4 feature tiles, whose operands its L2 then serves 4 and
// up to 8 times, and neighbouring units go to different XCDs, so the unused row tiles at the end of the plan cost every XCD the same. The units are counted
// over the tiles alone (a band of 8 row tiles column by column): with holes where the last unit of a band is not full, the same workgroups would be idle in
// every band (ff 768, six feature tiles of gate|up: 203 us, now 171).
//
// Why 128 x 128 per wavefront for many rows: per 32 of k it reads 16 operands for 64 MFMAs, which keeps the LDS pipe (128 bytes a clock for
// four SIMDs) at half of the matrix pipe's time; the 64 x 64 wavefront tile of moe_gemm_tiled_kernel needs all of it. Measured on MI355X, gate|up
// and down of 32 experts: 54,200 rows, width 4096, ff 3072 at tiles of 256 rows 2.27 to 2.38 + 1.32 to 1.41 ms = 1150 to 1200 and 970 to 1030 TFLOP/s (the tiled kernel: 4.05 +
// 2.28 ms). 256 rows (a decode step of 64 sequences, 1.6 + 0.8 GB of weights) at tiles of 16 rows 289 + 141 us = 5.6 TB/s
// (moe_gemm_mfma_kernel 411 + 217); width 1024, ff 768: 20 + 12 us (58 + 27). 32-bit, 1,044 rows, width 1024: 59 + 32 us (moe_gemm_kernel
// 1130 + 763), error against 64-bit sums 9e-7 of the result.
typedef __attribute__((address_space(3))) void lds_void_t;
typedef const __attribute__((address_space(1))) void global_void_t;

__device__ __forceinline__ void dma16(const char* src, char* lds_row) {        // 64 lanes: LDS [lds_row + 16 lane] <- 16 bytes at src
  __builtin_amdgcn_global_load_lds((global_void_t*)src, (lds_void_t*)lds_row, 16, 0, 0);
}

// one weight-row block times RB row blocks, 16 bytes of k per lane: 32 (bf16) or 16 (32-bit) of k
template <typename T, int RB>
__device__ __forceinline__ void mfma_units(f32x4_t (&acc)[RB], const u32x4_t& w, const u32x4_t (&x)[RB]) {
  if constexpr (sizeof(T) == 2) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[rb]) : "v"(w), "v"(x[rb]));
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)                     // (a lane brings the same four entries of k in both operands: any order of k will do)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) asm volatile("v_mfma_f32_16x16x4_f32 %0, %1, %2, %0" : "+a"(acc[rb]) : "v"(w[i]), "v"(x[rb][i]));
  }
}

// bytes of LDS per wavefront beside the ring: one row block of its results (two workgroups per compute unit leave none)
template <typename T, int PER_CU>
constexpr int pipe_turn = sizeof(T) == 2 && PER_CU == 1 ? 4096 : 0;

// silu(g) u. 16-bit results: silu_hw. Results that are not the nearest bfloat16 number to silu(g), in 2^-16 of a million gates in [-20, -10], [-10, -4],
// [-2, 2]: 0.13, 0.25, 0.25; with expf and a division 0.13, 0.13, 0.19; without its two corrections 4.1, 1.6, 0.6.
// They are seven instructions a value while the matrix pipe waits: 14,600 rows, ff 3072, K 1024 184 us without, 197 with them (moe_gemm_pipe_kernel). Eight values side by side take as
// long, and a step of Newton for the reciprocal in the remainder's place (one instruction fewer) leaves 0.38, 0.31, 0.5.
template <typename T>
__device__ __forceinline__ float silu_times(float g, float u) {
  if constexpr (sizeof(T) == 4) return glu_value(g, u, 0, 0.f, 0.f);
  return silu_hw(g) * u;
}

template <typename T, bool GLU, int WN, int WB, int RB, int ST, int PER_CU, bool PLAN>
__global__ __launch_bounds__(256, PER_CU) void moe_gemm_pipe_kernel(const T* __restrict__ X, int64_t ldx, const T* __restrict__ W, int nout, int K,
                                                                    const int32_t* __restrict__ tile_expert,
                                                                    const int32_t* __restrict__ row_token, int tiles_m, int tiles_n,
                                                                    int group, int rows, T* __restrict__ out, int64_t ldo, int mode) {
  constexpr int BM = 16 * RB * (4 / WN), BW = 16 * WB * WN, NG = GLU ? 2 : 1, BN = BW / NG, ROW = 128, UNIT = 16 / sizeof(T);
  constexpr int STAGE = (BM + BW) * ROW, XI = BM >= 32 ? BM / 32 : 1, WI = BW / 32, NR = XI + WI;      // requests of a wavefront per step
  constexpr int FB = WB / NG;                 // feature blocks of a wavefront
  // 16-bit tiles with room beside the ring: two feature blocks lie side by side, so a lane's results are 8 features in a row, and a row
  // block goes through LDS for stores of whole rows (pipe_turn bytes per wavefront)
  constexpr bool PAIR = pipe_turn<T, PER_CU> > 0;
  static_assert(WB % NG == 0 && BW % 32 == 0 && (ST - 2) * NR < 64, "tile");
  // no plan: every tile is expert 0's, and `rows` rows are their own tokens
  const auto expert = [&](int tile) { return PLAN ? tile_expert[tile] : 0; };
  const auto token = [&](int64_t r) { return PLAN ? row_token[r] : (int)r < rows ? (int)r : -1; };
  extern __shared__ __attribute__((aligned(128))) char lds[];
  // tiles in bands of 8 row tiles, a band column by column; this workgroup's: blocks blockIdx.x, blockIdx.x + gridDim.x, ... (the same XCD's)
  int block = blockIdx.x, rt = 0, ft = 0, high = 8;
  const auto find = [&] {
    const int j = block / 8, at = (j / group * 8 + block % 8) * group + j % group;
    const int band = at / (8 * tiles_n), k = at % (8 * tiles_n);
    high = min(8, tiles_m - band * 8);
    if (high <= 0) return false;
    ft = k / high, rt = band * 8 + k % high;
    return ft < tiles_n;
  };
  // tiles without rows are the last row tiles of a plan. In a whole band a workgroup's row tiles only grow: nothing follows the first one
  const auto used = [&](int e) {
    while (e < 0) {
      if (high == 8) return -1;
      block += gridDim.x;
      if (!find()) return -1;
      e = expert(rt);
    }
    return e;
  };
  if (!find()) return;
  int e = used(expert(rt));
  if (e < 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15;
  const int wn = wave % WN, wm = wave / WN;
  // requests: one covers 8 rows; lane l brings unit (l & 7) ^ swizzle of row l >> 3. Padding rows and rows beyond the last feature bring
  // some valid row; what is computed from them is not stored. (Tiles of 16 rows: two wavefronts bring the same rows twice.)
  uint32_t xoff[XI], woff[WI];               // in units of 16 bytes: half the registers of addresses
  static_assert(XI <= RB, "tile");
  int tok[RB];                               // tokens of the rows a lane asks for, near a tile's end of the rows it stores
  const auto look = [&] {
#pragma unroll
    for (int i = 0; i < XI; ++i) tok[i] = token((int64_t)rt * BM + (wave * XI + i) * 8 % BM + (lane >> 3));
  };
  const char* wbase;
  const auto point = [&] {
    int l = lane;
    asm volatile("" : "+v"(l));              // (what follows from the lane alone is worked out here, not kept over the loop)
    wbase = (const char*)(W + (int64_t)e * NG * nout * K);
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int r = (wave * XI + i) * 8 % BM + (l >> 3);
      const uint32_t src = (GLU || mode == 2) ? (tok[i] >= 0 ? tok[i] : 0) : rt * BM + r;
      xoff[i] = src * (uint32_t)(ldx / UNIT) + ((l & 7) ^ ((r >> 1) & 7));
    }
#pragma unroll
    for (int i = 0; i < WI; ++i) {
      const int r = (wave * WI + i) * 8 + (l >> 3), f = ft * BN + r % BN;
      woff[i] = (uint32_t)(r / BN * nout + (f < nout ? f : nout - 1)) * (uint32_t)(K / UNIT) + ((l & 7) ^ (PAIR ? ((r >> 1) & 1) | ((r >> 2) & 6) : (r >> 1) & 7));
    }
  };
  look();
  point();
  const auto request = [&](int i, int at, int step) {                   // request i of a step into the buffer at byte `at`
    if (i < XI) dma16((const char*)X + step * ROW + (uint64_t)xoff[i < XI ? i : 0] * 16, lds + at + (wave * XI + i) * 8 % BM * ROW);
    else dma16(wbase + step * ROW + (uint64_t)woff[i < XI ? 0 : i - XI] * 16, lds + at + (BM + (wave * WI + i - XI) * 8) * ROW);
  };
  f32x4_t acc[WB][RB];
  // operands of a half: weight-row block wb (GLU: the first half gate, the second up of the same features) and row block rb
  struct Operands {
    u32x4_t x[RB], w[WB];
  };
  const int unit0 = ((lane >> 4) ^ ((li >> 1) & 7)) * 16;               // (blocks start at multiples of 16 rows: the swizzle is the lane's)
  const char* xrow = lds + (wm * 16 * RB + li) * ROW;
  const char* wrow = lds + (BM + wn * FB * 16 + (PAIR ? (li >> 2) * 8 + (li & 3) : li)) * ROW;
  const auto load = [&](Operands& o, int g, int at, int half) {         // a WB-th of a half's operands
    const int place = at + (unit0 ^ (half * 64));                       // unit (4 half + (lane >> 4)) ^ swizzle
#pragma unroll
    for (int i = g * RB / WB; i < (g + 1) * RB / WB; ++i) o.x[i] = *(const u32x4_t*)(xrow + place + i * 16 * ROW);
    o.w[g] = *(const u32x4_t*)(wrow + place + (g / FB * BN + (PAIR ? g % FB / 2 * 32 + g % 2 * 4 : g % FB * 16)) * ROW);
  };
  const auto half_step = [&](const Operands& now, Operands& next, int next_at, int next_half, bool ask, int ask_at, int ask_step) {
    constexpr int AG = WB >= 4 ? WB / 2 : WB, PER = (NR + AG - 1) / AG;  // requests go out in the first half of the groups
#pragma unroll
    for (int g = 0; g < WB; ++g) {
      if (ask && g < AG) {
#pragma unroll
        for (int i = g * PER; i < (g + 1) * PER; ++i)
          if (i < NR) request(i, ask_at, ask_step);
      }
      load(next, g, next_at, next_half);
      __builtin_amdgcn_sched_barrier(0);
      mfma_units<T, RB>(acc[g], now.w[g], now.x);
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);      // lgkmcnt(0): what was read ahead is there (the counter is too short to wait for it behind the next reads)
  };
  constexpr int AHEAD = (ST - 2) * NR;       // requests younger than the next step's
  const auto arrive = [&](bool all, bool none) {        // the next step's requests landed (all: every request) and own LDS reads done; then everybody's
    __builtin_amdgcn_sched_barrier(0);
    if (none) __builtin_amdgcn_s_waitcnt(0xC07F);
    else if (all) __builtin_amdgcn_s_waitcnt(0);
    else __builtin_amdgcn_s_waitcnt((AHEAD & 15) | (AHEAD >> 4) << 14);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  const int steps = K / (8 * UNIT);
  Operands a, b;
#pragma unroll
  for (int s = 0; s < ST; ++s) {
    if (s < steps) {
#pragma unroll
      for (int i = 0; i < NR; ++i) request(i, s * STAGE, s);
    }
  }
  arrive(true, false);
#pragma unroll
  for (int g = 0; g < WB; ++g) load(a, g, 0, 0);
  __builtin_amdgcn_s_waitcnt(0xC07F);
  int at = 0;
  const bool whole = ((nout | (int)ldo) & (PAIR ? 7 : 3)) == 0 && ((uintptr_t)out & 15) == 0;
#pragma unroll 1
  for (;;) {
    // what the tile after this one needs is looked up now and used behind the loop
    const int64_t row0 = (int64_t)rt * BM;
    const int f0 = ft * BN;
    block += gridDim.x;
    bool more = find();
    const int e_next = more ? expert(rt) : -1;
    if (more) look();
#pragma unroll
    for (int wb = 0; wb < WB; ++wb)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) acc[wb][rb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    int s = 0;
#pragma unroll 1
    do {
      if (s == (steps > ST ? steps - ST : 0)) {
        if (more) {
          e = used(e_next);
          more = e >= 0;
          if (more && e_next < 0) look();
          if (more) point();
        }
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) tok[rb] = token(row0 + (wm * RB + rb) * 16 + li);
      }
      const int next = at + STAGE == ST * STAGE ? 0 : at + STAGE;
      half_step(a, b, at, 1, false, 0, 0);
      arrive(ST == 2 || (!more && s + ST > steps), s < ST - 1);
      const bool same = s + ST < steps;        // the last ST steps ask for the first ones of the tile that follows
      half_step(b, a, next, 0, same || more, at, same ? s + ST : s + ST - steps);
      at = next;
    } while (++s < steps);
    int l = lane;
    asm volatile("" : "+v"(l));
    const int wi = l & 15;
    asm volatile("s_nop 15\n\ts_nop 15");      // the last products are written before they are read: every read depends on one of
#pragma unroll                             // these statements, and volatile ones keep their order
    for (int wb = 0; wb < WB; ++wb)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) asm volatile("" : "+a"(acc[wb][rb]));
    __builtin_amdgcn_s_waitcnt(0x0F70);        // the requests for the next tile are there: its first ST - 1 steps need not wait behind the stores
    // lane: row li of row block rb; features 16 fb + 4 (lane >> 4) + 0..3 of its wavefront's, or 32 fb + 8 (lane >> 4) + 0..7 of a pair's
    constexpr int RUN = PAIR ? 8 : 4, RUNS = FB * 4 / RUN;
    const auto value = [&](int rb, int i) {    // number i of a lane's results of a row block
      const float y = acc[i / 4][rb][i % 4];
      if constexpr (GLU) return (T)silu_times<T>(y, acc[i / 4 + FB][rb][i % 4]);
      else return (T)plain_value(y, mode);
    };
    const int first = f0 + wn * FB * 16;       // the wavefront's features
    if (PAIR && whole) {
      constexpr int UNITS = PAIR ? RUNS * 4 : 4, PER = 64 / UNITS;       // 16-byte units of a row, rows of a store
      u32x4_t* turn = (u32x4_t*)(lds + ST * STAGE + wave * pipe_turn<T, PER_CU>);
      const auto place = [&](int r, int u) { return r * UNITS + (u ^ ((UNITS == 16 ? r : r >> 1) & (UNITS - 1))); };
      const int f = first + l % UNITS * 8, sub = l / UNITS;
      T* to = out + (row0 + wm * RB * 16 + sub) * ldo + f;
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const uint32_t live = (uint32_t)__ballot(tok[rb] >= 0);
#pragma unroll
        for (int u = 0; u < RUNS; ++u) {
          union { T v[RUN]; u32x4_t q; } o;
#pragma unroll
          for (int i = 0; i < RUN; ++i) o.v[i] = value(rb, u * RUN + i);
          turn[place(wi, u * 4 + (l >> 4))] = o.q;
        }
#pragma unroll
        for (int p = 0; p < 16 / PER; ++p) {
          const u32x4_t q = turn[place(p * PER + sub, l % UNITS)];
          if ((live >> (p * PER + sub) & 1) && f < nout) *(u32x4_t*)(to + (int64_t)(rb * 16 + p * PER) * ldo) = q;
        }
      }
    } else {
      const int mine = first + (l >> 4) * RUN;
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        T* to = out + (row0 + (wm * RB + rb) * 16 + wi) * ldo + mine;
        if (tok[rb] < 0) continue;
#pragma unroll
        for (int u = 0; u < RUNS; ++u) {
          typedef __attribute__((ext_vector_type(4))) T t4_t;
          if (!PAIR && whole) {
            if (mine + u * RUN * 4 < nout) *(t4_t*)(to + u * RUN * 4) = t4_t{value(rb, u * RUN), value(rb, u * RUN + 1), value(rb, u * RUN + 2), value(rb, u * RUN + 3)};
          } else {
#pragma unroll
            for (int i = 0; i < RUN; ++i)
              if (mine + u * RUN * 4 + i < nout) to[u * RUN * 4 + i] = value(rb, u * RUN + i);
          }
        }
      }
    }
    if (!more) break;
  }
}

template <typename T, bool GLU, int WN, int WB, int RB, int ST, int PER_CU, bool PLAN = true>
int launch_pipe(const void* X, int64_t ldx, const void* W, int nout, int K, const int32_t* tile_expert, const int32_t* row_token, int64_t cap,
                void* out, int64_t ldo, int mode, hipStream_t st, int rows = 0) {
  constexpr int BM = 16 * RB * (4 / WN), BW = 16 * WB * WN, BN = GLU ? BW / 2 : BW, LDS = ST * (BM + BW) * 128 + 4 * pipe_turn<T, PER_CU>;
  const int64_t tiles_m = cap / BM, tiles_n = (nout + BN - 1) / BN;
  // Tiles of a group share an L2. Few tiles go to the XCDs in smaller groups, so that each of them brings its share of the weights
  const int64_t tiles = tiles_m * tiles_n;
  const int group = tiles >= 256 ? 32 : 8;
  int64_t blocks = (tiles + 8 * group - 1) / (8 * group) * (8 * group);
  NVS_REQUIRE(blocks < (1ll << 31), "nvs_moe_gemm: step too large");
  const auto kernel = moe_gemm_pipe_kernel<T, GLU, WN, WB, RB, ST, PER_CU, PLAN>;
  NVS_LDS_ROOM(kernel, LDS, "nvs_moe_gemm");
  // the ring goes on over the tiles of a workgroup if every stage holds a step of every tile
  if (K / (128 / (int)sizeof(T)) >= ST && blocks > 256 * PER_CU) blocks = 256 * PER_CU;
  kernel<<<dim3((unsigned)blocks), dim3(256), LDS, st>>>((const T*)X, ldx, (const T*)W, nout, K, tile_expert, row_token, (int)tiles_m, (int)tiles_n,
                                                         group, rows, (T*)out, ldo, mode);
  return nvs_check_launch("nvs_moe_gemm (matrix cores, pipelined)");
}

#include "gemm_tiles.h"

// ---- combine: one workgroup per token ------------------------------------------------------------------------------------
template <typename T, int VEC>
__global__ void moe_combine_kernel(const T* __restrict__ rows, int64_t ldr, const int32_t* __restrict__ pair_row,
                                   const float* __restrict__ wts, int top, const T* __restrict__ h, int64_t ldh,
                                   const T* __restrict__ shared, const float* __restrict__ shared_gate, int64_t gate_stride, int width,
                                   float* __restrict__ res, T* __restrict__ out) {
  const int64_t t = blockIdx.x;
  float sg = 0.f;
  if (shared) sg = shared_gate ? 1.f / (1.f + expf(-shared_gate[t * gate_stride])) : 1.f;      // no gate: the shared expert is added as it is
  for (int c = (blockIdx.y * blockDim.x + threadIdx.x) * VEC; c < width; c += gridDim.y * blockDim.x * VEC) {
    float acc[VEC], v[VEC];
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] = 0.f;
    for (int k = 0; k < top; ++k) {
      const int r = pair_row[t * top + k];
      ldv<VEC>(r >= 0 ? rows + (int64_t)r * ldr + c : h + t * ldh + c, v);      // no row: a pass-through expert
      const float w = wts[t * top + k];
#pragma unroll
      for (int i = 0; i < VEC; ++i) acc[i] += w * v[i];
    }
    if (shared) {
      ldv<VEC>(shared + t * width + c, v);
#pragma unroll
      for (int i = 0; i < VEC; ++i) acc[i] += sg * v[i];
    }
    if (res) {                                      // the residual add is taken along: out is the new residual row, rounded
      ldv<VEC>(res + t * width + c, v);
#pragma unroll
      for (int i = 0; i < VEC; ++i) acc[i] += v[i];
      stv<VEC>(res + t * width + c, acc);
    }
    if (out) stv<VEC>(out + t * width + c, acc);
  }
}

}  // namespace

static int g_moe_plain = 0;
extern "C" void nvs_moe_force_plain(int on) { g_moe_plain = on; }

extern "C" int nvs_glu_act(const void* gu, int64_t stride, int dtype, int ff, int kind, float limit, float alpha, int64_t n, void* out,
                           void* stream) {
  NVS_REQUIRE(gu && out && ff > 0 && stride >= (kind == 2 ? 1 : 2) * (int64_t)ff && kind >= 0 && kind <= 2 && n >= 0, "nvs_glu_act: ff %d stride %lld kind %d",
              ff, (long long)stride, kind);
  if (n == 0) return NVS_OK;
  const int64_t units = n * (ff / 8);
  if (ff % 8 == 0 && stride % 8 == 0 && ((uintptr_t)gu | (uintptr_t)out) % 32 == 0 && units < (1ll << 31) - 256) {
    NVS_DISPATCH(dtype, glu_act_rows8_kernel<T><<<dim3((unsigned)((units + 255) / 256)), dim3(256), 0, (hipStream_t)stream>>>(
                            (const T*)gu, stride, ff / 8, kind, limit, alpha, (int)units, (T*)out));
    return nvs_check_launch("nvs_glu_act (eight columns per access)");
  }
  int64_t blocks = (n * ff + 255) / 256;
  if (blocks > 65535 * 16) blocks = 65535 * 16;
  NVS_DISPATCH(dtype, glu_act_kernel<T><<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>((const T*)gu, stride, ff, kind, limit,
                                                                                                    alpha, n, (T*)out));
  return nvs_check_launch("nvs_glu_act");
}

extern "C" int nvs_moe_route(const float* z, int64_t z_stride, const float* correction, int64_t n, int total, int top, int count, int keep,
                             float scale, int score, int renorm, int32_t* ids, float* wts, void* stream) {
  NVS_REQUIRE(z && ids && wts && n >= 0 && (score == 0 || score == 1), "nvs_moe_route: bad argument");
  NVS_REQUIRE(total > 0 && total <= MAX_EXPERTS && z_stride >= total && top > 0 && top <= 64 && count > 0 && count <= 64 && total % count == 0 &&
                  keep > 0 && keep <= count && (int64_t)keep * (total / count) >= top,
              "nvs_moe_route: %d entries, %d choices, %d of %d groups", total, top, keep, count);
  if (n == 0) return NVS_OK;
  moe_route_kernel<<<dim3((unsigned)n), dim3(64), 0, (hipStream_t)stream>>>(z, z_stride, correction, total, top, count, keep, scale, score, renorm, ids, wts);
  return nvs_check_launch("nvs_moe_route");
}

extern "C" int nvs_moe_table_route(const int64_t* tokens, const int32_t* table, int64_t n, int top, float weight, int32_t* ids, float* wts,
                                   void* stream) {
  NVS_REQUIRE(tokens && table && ids && wts && n >= 0 && top > 0 && top <= 64, "nvs_moe_table_route: bad argument (%d choices)", top);
  if (n == 0) return NVS_OK;
  const int64_t pairs = n * top;
  moe_table_route_kernel<<<dim3((unsigned)((pairs + 255) / 256)), dim3(256), 0, (hipStream_t)stream>>>(tokens, table, pairs, top, weight, ids, wts);
  return nvs_check_launch("nvs_moe_table_route");
}

extern "C" int64_t nvs_moe_rows(int64_t pairs, int experts, int tm) { return (pairs + (int64_t)experts * (tm - 1) + tm - 1) / tm * tm; }

extern "C" int nvs_moe_plan(const int32_t* ids, int64_t n, int top, int experts, int tm, int32_t* tile_expert, int32_t* row_token,
                            int32_t* pair_row, void* stream) {
  NVS_REQUIRE(ids && tile_expert && row_token && pair_row && n >= 0 && top > 0, "nvs_moe_plan: null argument");
  NVS_REQUIRE(experts > 0 && experts <= MAX_EXPERTS && (tm == 16 || tm == 64 || tm == 128 || tm == 256), "nvs_moe_plan: %d experts, tiles of %d rows", experts, tm);
  if (n == 0) return NVS_OK;
  const int64_t cap = nvs_moe_rows(n * top, experts, tm);
  NVS_REQUIRE(cap < (1ll << 31), "nvs_moe_plan: step too large");
  moe_plan_kernel<<<dim3(1), dim3(1024), 0, (hipStream_t)stream>>>(ids, n * top, top, experts, tm, cap, tile_expert, row_token, pair_row);
  return nvs_check_launch("nvs_moe_plan");
}

extern "C" int64_t nvs_moe_plan_scratch(int64_t pairs, int experts) {
  // (one workgroup / many, us: 4,096 pairs 5.6 / 6.5 with 32 experts, 7.0 / 7.1 with 256; 8,192: 7.8 / 6.4, 10.0 / 7.2)
  return pairs >= 6144 ? (pairs + PLAN_PAIRS - 1) / PLAN_PAIRS * experts : 0;
}

extern "C" int nvs_moe_plan_wide(const int32_t* ids, int64_t n, int top, int experts, int tm, int32_t* tile_expert, int32_t* row_token,
                                 int32_t* pair_row, int32_t* scratch, int64_t scratch_ints, void* stream) {
  const int64_t pairs = n * top, need = nvs_moe_plan_scratch(pairs, experts);
  if (!scratch || need == 0) return nvs_moe_plan(ids, n, top, experts, tm, tile_expert, row_token, pair_row, stream);
  NVS_REQUIRE(ids && tile_expert && row_token && pair_row && n >= 0 && top > 0, "nvs_moe_plan_wide: null argument");
  NVS_REQUIRE(experts > 0 && experts <= MAX_EXPERTS && (tm == 16 || tm == 64 || tm == 128 || tm == 256), "nvs_moe_plan_wide: %d experts, tiles of %d rows",
              experts, tm);
  const int64_t cap = nvs_moe_rows(pairs, experts, tm);
  NVS_REQUIRE(cap < (1ll << 31) && need < (1ll << 31), "nvs_moe_plan_wide: step too large");
  NVS_REQUIRE(scratch_ints >= need, "nvs_moe_plan_wide: scratch of %lld entries is too small", (long long)scratch_ints);
  const dim3 grid((unsigned)((pairs + PLAN_PAIRS - 1) / PLAN_PAIRS));
  moe_plan_count_kernel<<<grid, dim3(1024), 0, (hipStream_t)stream>>>(ids, pairs, experts, cap, row_token, pair_row, scratch);
  moe_plan_place_kernel<<<grid, dim3(1024), 0, (hipStream_t)stream>>>(ids, pairs, top, experts, tm, cap, tile_expert, row_token, pair_row, scratch);
  return nvs_check_launch("nvs_moe_plan_wide");
}

extern "C" int nvs_moe_gemm(const void* X, int64_t ldx, const void* W, int dtype, int mode, int nout, int K, const int32_t* tile_expert,
                            const int32_t* row_token, int64_t cap, int tm, void* out, int64_t ldo, void* stream) {
  NVS_REQUIRE(X && W && tile_expert && row_token && out && mode >= 0 && mode <= 2, "nvs_moe_gemm: bad argument");
  const int glu = mode == 1;
  NVS_REQUIRE(nout > 0 && K > 0 && ldx >= K && ldo >= nout && (tm == 16 || tm == 64 || tm == 128 || tm == 256) && cap >= 0 && cap % tm == 0,
              "nvs_moe_gemm: %d x %d, %lld rows in tiles of %d", nout, K, (long long)cap, tm);
  if (cap == 0) return NVS_OK;
  hipStream_t st = (hipStream_t)stream;
  const bool matrix_cores = dtype == NVS_BF16 && K % 8 == 0 && ldx % 8 == 0 && !g_moe_plain;
  const int64_t size = dtype == NVS_BF16 ? 2 : 4, reach = 16ll << 32;      // (its offsets are 32 bits of 16-byte units: rows and an expert's weights up to 64 GiB)
  const bool whole = cap * ldx * size < reach && 2ll * nout * K * size < reach &&
                     (K % (dtype == NVS_BF16 ? 64 : 32) == 0) && ldx % (dtype == NVS_BF16 ? 8 : 4) == 0 && (((uintptr_t)X | (uintptr_t)W) & 15) == 0;
  if (whole && !g_moe_plain) {
#define NVS_PIPE(...)                                                                                                       \
  (dtype == NVS_BF16                                                                                                        \
       ? (glu ? launch_pipe<bf16_t, true, __VA_ARGS__>(X, ldx, W, nout, K, tile_expert, row_token, cap, out, ldo, mode, st) \
              : launch_pipe<bf16_t, false, __VA_ARGS__>(X, ldx, W, nout, K, tile_expert, row_token, cap, out, ldo, mode, st)) \
       : (glu ? launch_pipe<float, true, __VA_ARGS__>(X, ldx, W, nout, K, tile_expert, row_token, cap, out, ldo, mode, st)  \
              : launch_pipe<float, false, __VA_ARGS__>(X, ldx, W, nout, K, tile_expert, row_token, cap, out, ldo, mode, st)))
    if (tm == 256 && dtype == NVS_BF16 && tiles_fit(ldx, cap, nout, K, (glu ? 2ll : 1ll) * nout * K, out, ldo)) {
      const auto launch = glu ? launch_tiles<1, true> : mode ? launch_tiles<2, true> : launch_tiles<0, true>;
      return launch(X, ldx, W, nout, K, tile_expert, row_token, cap, out, ldo, st, "nvs_moe_gemm (matrix cores, tiles of 256 rows)", 0, nullptr);
    }
    if (tm == 256) return NVS_PIPE(2, 8, 8, 2, 1);
    if (tm == 128) return NVS_PIPE(2, 8, 4, 3, 1);
    if (tm == 64) return NVS_PIPE(4, 4, 4, 2, 2);
    return NVS_PIPE(4, 2, 1, 4, 2);
#undef NVS_PIPE
  }
  if (matrix_cores && tm >= 128) {
    const int bn = glu ? 64 : 128;                  // features per tile
    const int tiles_m = (int)(cap / 128), tiles_n = (nout + bn - 1) / bn;
    const int64_t blocks = ((int64_t)tiles_m * tiles_n + 7) / 8 * 8;
    NVS_REQUIRE(blocks < (1ll << 31), "nvs_moe_gemm: step too large");
    if (glu)
      moe_gemm_tiled_kernel<true><<<dim3((unsigned)blocks), dim3(256), 0, st>>>((const bf16_t*)X, ldx, (const bf16_t*)W, nout, K, tile_expert,
                                                                                row_token, tiles_m, tiles_n, tm / 128, (bf16_t*)out, ldo, mode);
    else
      moe_gemm_tiled_kernel<false><<<dim3((unsigned)blocks), dim3(256), 0, st>>>((const bf16_t*)X, ldx, (const bf16_t*)W, nout, K, tile_expert,
                                                                                 row_token, tiles_m, tiles_n, tm / 128, (bf16_t*)out, ldo, mode);
    return nvs_check_launch("nvs_moe_gemm (matrix cores, LDS tiles)");
  }
  if (matrix_cores) {
    const dim3 grid((unsigned)(cap / tm), (unsigned)((nout + 127) / 128));
#define NVS_MOE_CASE(MT, GLU)                                                                                                        \
  moe_gemm_mfma_kernel<MT, GLU><<<grid, dim3(256), 0, st>>>((const bf16_t*)X, ldx, (const bf16_t*)W, nout, K, tile_expert, row_token,  \
                                                            (bf16_t*)out, ldo, mode)
    if (tm == 64) {
      if (glu) NVS_MOE_CASE(4, true); else NVS_MOE_CASE(4, false);
    } else {
      if (glu) NVS_MOE_CASE(1, true); else NVS_MOE_CASE(1, false);
    }
#undef NVS_MOE_CASE
    return nvs_check_launch("nvs_moe_gemm (matrix cores)");
  }
  const dim3 grid((unsigned)(cap / 16), (unsigned)((nout + 63) / 64));
  if (glu) {
    NVS_DISPATCH(dtype, moe_gemm_kernel<T, true><<<grid, dim3(256), 0, st>>>((const T*)X, ldx, (const T*)W, nout, K, tile_expert, row_token, tm,
                                                                            (T*)out, ldo, mode));
  } else {
    NVS_DISPATCH(dtype, moe_gemm_kernel<T, false><<<grid, dim3(256), 0, st>>>((const T*)X, ldx, (const T*)W, nout, K, tile_expert, row_token,
                                                                             tm, (T*)out, ldo, mode));
  }
  return nvs_check_launch("nvs_moe_gemm");
}

// silu(g) u of [g | u] = X W^T: the tiles of the grouped product with one expert and no plan. The library's product and the activation behind it write and read
// [n, 2 ff] once more than this: 14,600 rows, ff 3072, K 1024 202 us, here 155; which of them is taken is the caller's choice (measured there).
extern "C" int nvs_silu_linear(const void* X, int64_t ldx, const void* W, int ff, int K, int64_t n, int tm, void* out, int64_t ldo, void* stream) {
  if (n == 0) return NVS_OK;
  NVS_REQUIRE(X && W && out && ff > 0 && K > 0 && K % 64 == 0 && n > 0 && ldx >= K && ldx % 8 == 0 && ldo >= ff && (((uintptr_t)X | (uintptr_t)W) & 15) == 0,
              "nvs_silu_linear: %lld rows, %d x %d", (long long)n, ff, K);
  NVS_REQUIRE((tm == 64 || tm == 256) && n < (1ll << 31) - 256 && (n + 255) * ldx < (8ll << 32) && 2ll * ff * K < (8ll << 32), "nvs_silu_linear: step too large");
  const int64_t cap = (n + tm - 1) / tm * tm;
  if (tm == 256 && tiles_fit(ldx, n, ff, K, 2ll * ff * K, out, ldo)) return launch_tiles<1, false>(X, ldx, W, ff, K, nullptr, nullptr, n, out, ldo, (hipStream_t)stream, "nvs_silu_linear", (int)n);
  if (tm == 256) return launch_pipe<bf16_t, true, 2, 8, 8, 2, 1, false>(X, ldx, W, ff, K, nullptr, nullptr, cap, out, ldo, 1, (hipStream_t)stream, (int)n);
  return launch_pipe<bf16_t, true, 4, 4, 4, 2, 2, false>(X, ldx, W, ff, K, nullptr, nullptr, cap, out, ldo, 1, (hipStream_t)stream, (int)n);
}

// X W^T (+ bias) of many rows
extern "C" int nvs_linear_tiles(const void* X, int64_t ldx, const void* W, const void* bias, int nout, int K, int64_t n, void* out, int64_t ldo, void* stream) {
  if (n == 0) return NVS_OK;
  NVS_REQUIRE(X && W && out && nout > 0 && n > 0 && ldx >= K && ldx % 8 == 0 && ldo >= nout && (((uintptr_t)X | (uintptr_t)W | (uintptr_t)bias) & 15) == 0 &&
                  n < (1ll << 31) - 256 && tiles_fit(ldx, n, nout, K, (int64_t)nout * K, out, ldo),
              "nvs_linear_tiles: %lld rows, %d x %d", (long long)n, nout, K);
  if (bias) return launch_tiles<3, false>(X, ldx, W, nout, K, nullptr, nullptr, n, out, ldo, (hipStream_t)stream, "nvs_linear_tiles", (int)n, bias);
  return launch_tiles<0, false>(X, ldx, W, nout, K, nullptr, nullptr, n, out, ldo, (hipStream_t)stream, "nvs_linear_tiles", (int)n);
}

extern "C" int nvs_moe_combine(const void* rows, int64_t ldr, const int32_t* pair_row, const float* wts, int top, const void* h, int64_t ldh,
                               const void* shared, const float* shared_gate, int64_t gate_stride, int dtype, int64_t n, int width, float* res,
                               void* out, void* stream) {
  NVS_REQUIRE(rows && pair_row && wts && h && (out || res) && top > 0 && width > 0 && n >= 0,
              "nvs_moe_combine: bad argument");
  if (n == 0) return NVS_OK;
  // four columns per access where every row starts aligned for it; wide rows of few tokens are spread over several workgroups
  const uintptr_t al = (uintptr_t)rows | (uintptr_t)h | (uintptr_t)shared | (uintptr_t)res | (uintptr_t)out;
  const bool vec = width % 4 == 0 && ldr % 4 == 0 && ldh % 4 == 0 && al % 16 == 0;
  const int per = vec ? width / 4 : width, threads = per >= 256 ? 256 : (per >= 128 ? 128 : 64);
  const dim3 grid((unsigned)n, n <= 512 ? (unsigned)((per + threads - 1) / threads) : 1u);
#define NVS_COMBINE(VEC)                                                                                                              \
  NVS_DISPATCH(dtype, moe_combine_kernel<T, VEC><<<grid, dim3(threads), 0, (hipStream_t)stream>>>(                                      \
                          (const T*)rows, ldr, pair_row, wts, top, (const T*)h, ldh, (const T*)shared, shared_gate, gate_stride, width, \
                          res, (T*)out))
  if (vec) NVS_COMBINE(4);
  else NVS_COMBINE(1);
#undef NVS_COMBINE
  return nvs_check_launch("nvs_moe_combine");
}
