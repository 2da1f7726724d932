// The norm before a linear layer and the layer in one kernel, for up to 16 rows (a decode step of few sequences).
//
// Such a step is a chain of launches whose weights are read in 1-3 us each; the add + norm between two of them (two per layer) was a launch of its own, 2.4 us and
// the gap before it, for a few KB. Here every workgroup of the linear layer norms the rows again: they are asked for first, the workgroup's weights
// right behind, so the rows' sums, norm and way through LDS lie under the weights' way from memory. A workgroup takes 16 columns (SiLU: and their partners);
// eight wavefronts share the reduction, each with a ring of two pieces (128 bytes of k per row, 16-byte unit c of row r at c ^ ((r >> 1) & 7): the 16 rows
// of an operand read lie on 16 different bank quads), filled straight from memory, and the sums meet in LDS. Workgroup 0
// writes the new residual, into a tensor of its own: the others still read the old one.
// x may be the fp32 slabs of a reduction split over workgroups (nvl_linear_decode mode 2): with few rows the down and out projections have too few columns to
// fill the chip otherwise (1024 x 3072, one row: 3.6 us in four slabs, 5.2 whole).
//   v = x + residual (slabs: v = bf16(sum) + residual);  residual' = bf16(v);  h = bf16(v rsqrt(mean v^2 + eps) w);  out = h W^T, or silu(gate) * up of its halves
// MI355X, one row, traced: 4096 x 1024 with the norm 4.3 us (norm 2.4, product 3.6, and a gap), 6144 x 1024 with norm and SiLU 5.7 (2.4 + 5.3); a step of one
// sequence through 28 layers 954 -> 925 us. The rows are normed by every workgroup, so more and wider ones lose what the launch gives: layers.py calls
// this for up to 8 rows of width 1,024, with the figures beside it.
#include "common.h"

namespace {

typedef __attribute__((address_space(3))) void lds_void_t;
typedef const __attribute__((address_space(1))) void global_void_t;

__device__ __forceinline__ float silu_f32(float g) { return g / (1.f + __expf(-g)); }

constexpr int kNormWaves = 8, kNormDepth = 2, kNormMaxK = 2048;

// S slabs of x (0: x is bf16), CH chunks of 8 entries of a row per lane
template <bool SILU, int S, int CH>
__global__ __launch_bounds__(64 * kNormWaves) void norm_linear_kernel(const void* __restrict__ x, int64_t slab, const bf16_t* __restrict__ residual,
                                                                      const bf16_t* __restrict__ norm_w, float eps, const bf16_t* __restrict__ w,
                                                                      bf16_t* __restrict__ out, bf16_t* __restrict__ residual_out, int M, int N, int K) {
  constexpr int NT = SILU ? 2 : 1, ROW = 128, STAGE = NT * 16 * ROW, NR = NT * 2, SL = S > 0 ? S : 1;
  extern __shared__ __attribute__((aligned(128))) unsigned char smem_raw[];        // rings; normed rows [piece][16][128]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, lq = lane >> 4;
  const int f0 = blockIdx.x * 16, pieces = K / 64, chunks = K / 8;
  unsigned char* ring = smem_raw + wave * (kNormDepth * STAGE);
  unsigned char* rows = smem_raw + kNormWaves * kNormDepth * STAGE;
  // row `wave` (and then wave + 8): asked for before the weights (what has landed is counted in order)
  struct Row {
    u32x4_t x[CH], r[CH];
    f32x4_t p[CH][SL][2];
  } row;
  u32x4_t wr[CH];
  const auto ask = [&](int m) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int ch = lane + 64 * c;
      if (ch >= chunks) continue;
      if constexpr (S > 0) {
#pragma unroll
        for (int k = 0; k < S; ++k) {
          const float* p = (const float*)x + k * slab + (int64_t)m * K + ch * 8;
          row.p[c][k][0] = *reinterpret_cast<const f32x4_t*>(p), row.p[c][k][1] = *reinterpret_cast<const f32x4_t*>(p + 4);
        }
      } else {
        row.x[c] = *reinterpret_cast<const u32x4_t*>((const bf16_t*)x + (int64_t)m * K + ch * 8);
      }
      if (residual != nullptr) row.r[c] = *reinterpret_cast<const u32x4_t*>(residual + (int64_t)m * K + ch * 8);
    }
  };
  if (wave < M) {
    ask(wave);
#pragma unroll
    for (int c = 0; c < CH; ++c)
      if (lane + 64 * c < chunks) wr[c] = *reinterpret_cast<const u32x4_t*>(norm_w + (lane + 64 * c) * 8);
  }
  __builtin_amdgcn_sched_barrier(0);
  const bf16_t* src[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int r = i * 8 + (lane >> 3), f = f0 + r % 16;
    src[i] = w + ((int64_t)(r / 16) * N + (f < N ? f : N - 1)) * K + ((lane & 7) ^ ((r >> 1) & 7)) * 8;
  }
  const int mine = (pieces - wave + kNormWaves - 1) / kNormWaves;
  const auto request = [&](int s) {
#pragma unroll
    for (int i = 0; i < NR; ++i)
      __builtin_amdgcn_global_load_lds((global_void_t*)(src[i] + (int64_t)(s * kNormWaves + wave) * 64),
                                       (lds_void_t*)(ring + s % kNormDepth * STAGE + i * 1024), 16, 0, 0);
  };
#pragma unroll
  for (int s = 0; s < kNormDepth; ++s)
    if (s < mine) request(s);
#pragma unroll 1
  for (int m = wave; m < M; m += kNormWaves) {
    if (m != wave) ask(m);
    float v[CH][8], ss = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      if (lane + 64 * c >= chunks) continue;
      if constexpr (S > 0) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          f32x4_t p = row.p[c][0][h];
#pragma unroll
          for (int k = 1; k < SL; ++k) p += row.p[c][k][h];
#pragma unroll
          for (int i = 0; i < 4; ++i) v[c][h * 4 + i] = round_bf16(p[i]);
        }
      } else {
        unpack8(row.x[c], v[c]);
      }
      if (residual != nullptr) {
        float r[8];
        unpack8(row.r[c], r);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[c][i] += r[i];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) ss += v[c][i] * v[c][i];
    }
    const float rstd = rsqrtf(wave_allreduce_sum(ss) / (float)K + eps);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int ch = lane + 64 * c;
      if (ch >= chunks) continue;
      if (blockIdx.x == 0) *reinterpret_cast<u32x4_t*>(residual_out + (int64_t)m * K + ch * 8) = pack8(v[c]);
      float wf[8];
      unpack8(wr[c], wf);
#pragma unroll
      for (int i = 0; i < 8; ++i) wf[i] *= v[c][i] * rstd;
      *reinterpret_cast<u32x4_t*>(rows + (ch >> 3) * (16 * ROW) + m * ROW + (((ch & 7) ^ ((m >> 1) & 7)) << 4)) = pack8(wf);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0xC07F);              // lgkmcnt(0): the rows are written (and the weights keep coming)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  f32x4_t acc[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) acc[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int unit0 = (lq ^ ((li >> 1) & 7)) * 16;
#pragma unroll 1
  for (int s = 0; s < mine; ++s) {
    __builtin_amdgcn_sched_barrier(0);
    if (s + kNormDepth <= mine) __builtin_amdgcn_s_waitcnt(0x0F70 | (kNormDepth - 1) * NR);        // this piece landed
    else __builtin_amdgcn_s_waitcnt(0x0F70);
    __builtin_amdgcn_sched_barrier(0);
    const unsigned char* at = ring + s % kNormDepth * STAGE + li * ROW;
    const unsigned char* xat = rows + (s * kNormWaves + wave) * (16 * ROW) + li * ROW;             // (rows beyond M hold anything: their results are not stored)
    bf16x8_t wf[2][NT], xf[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      xf[h] = *reinterpret_cast<const bf16x8_t*>(xat + (unit0 ^ (h * 64)));
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) wf[h][nt] = *reinterpret_cast<const bf16x8_t*>(at + nt * 16 * ROW + (unit0 ^ (h * 64)));
    }
    if (s + kNormDepth < mine) {
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0xC07F);
      __builtin_amdgcn_sched_barrier(0);
      request(s + kNormDepth);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h][nt], xf[h], acc[nt], 0, 0, 0);
  }
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) *reinterpret_cast<f32x4_t*>(ring + (nt * 64 + lane) * 16) = acc[nt];
  __syncthreads();
  if (wave != 0) return;
  f32x4_t v[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    v[nt] = *reinterpret_cast<const f32x4_t*>(smem_raw + (nt * 64 + lane) * 16);
#pragma unroll
    for (int ww = 1; ww < kNormWaves; ++ww) v[nt] += *reinterpret_cast<const f32x4_t*>(smem_raw + ww * (kNormDepth * STAGE) + (nt * 64 + lane) * 16);
  }
  const int f = f0 + lq * 4;
  if (li >= M || f >= N) return;
  if constexpr (SILU) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[0][i] = silu_f32(round_bf16(v[0][i])) * round_bf16(v[NT - 1][i]);
  }
  *reinterpret_cast<u32x2_t*>(out + (int64_t)li * N + f) = u32x2_t{pack_bf16x2(v[0][0], v[0][1]), pack_bf16x2(v[0][2], v[0][3])};
}

template <bool SILU, int S, int CH>
int launch_norm_linear(const void* x, const void* residual, const void* norm_w, float eps, const void* w, void* out, void* residual_out, int64_t m, int n,
                       int k, hipStream_t s) {
  constexpr int ring = kNormWaves * kNormDepth * (SILU ? 2 : 1) * 2048;
  static bool attr_done[NVL_MAX_DEVICES] = {};
  bool& attr_set = attr_done[nvl_device_slot()];
  if (!attr_set) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&norm_linear_kernel<SILU, S, CH>), hipFuncAttributeMaxDynamicSharedMemorySize,
                            ring + CH * 512 * 32) != hipSuccess) {
      nvl_set_error("nvl_norm_linear: cannot reserve LDS");
      return NVL_ELAUNCH;
    }
    attr_set = true;
  }
  hipLaunchKernelGGL((norm_linear_kernel<SILU, S, CH>), dim3((unsigned)((n + 15) / 16)), dim3(64 * kNormWaves), ring + k * 32, s, x, m * k,
                     (const bf16_t*)residual, (const bf16_t*)norm_w, eps, (const bf16_t*)w, (bf16_t*)out, (bf16_t*)residual_out, (int)m, n, k);
  return nvl_check_launch("nvl_norm_linear");
}

}  // namespace

extern "C" int nvl_norm_linear(const void* x, int slabs, const void* residual, const void* norm_weight, float eps, const void* weight, void* out,
                               void* residual_out, int64_t m, int n, int k, int silu, void* stream) {
  NVL_REQUIRE(m >= 0 && m <= 16 && n > 0 && n % 4 == 0 && k > 0 && k % 64 == 0 && k <= kNormMaxK && (slabs == 0 || slabs == 1 || slabs == 2 || slabs == 4),
              "nvl_norm_linear: %lld x %d x %d, %d slabs (up to 16 rows, n %% 4 == 0, k %% 64 == 0 up to %d, 0, 1, 2 or 4 slabs)", (long long)m, n, k, slabs,
              kNormMaxK);
  if (m == 0) return NVL_OK;
  NVL_REQUIRE(x && norm_weight && weight && out && residual_out && residual_out != residual, "nvl_norm_linear: null pointer, or the residual in place");
  NVL_REQUIRE(((uintptr_t)x | (uintptr_t)residual | (uintptr_t)norm_weight | (uintptr_t)weight | (uintptr_t)out | (uintptr_t)residual_out) % 16 == 0,
              "nvl_norm_linear: pointers must be 16-byte aligned");
#define NVL_NORM_LINEAR(S)                                                                                                                              \
  (k <= 1024 ? (silu ? launch_norm_linear<true, S, 2>(x, residual, norm_weight, eps, weight, out, residual_out, m, n, k, (hipStream_t)stream)           \
                     : launch_norm_linear<false, S, 2>(x, residual, norm_weight, eps, weight, out, residual_out, m, n, k, (hipStream_t)stream))         \
             : (silu ? launch_norm_linear<true, S, 4>(x, residual, norm_weight, eps, weight, out, residual_out, m, n, k, (hipStream_t)stream)           \
                     : launch_norm_linear<false, S, 4>(x, residual, norm_weight, eps, weight, out, residual_out, m, n, k, (hipStream_t)stream)))
  switch (slabs) {
    case 0: return NVL_NORM_LINEAR(0);
    case 1: return NVL_NORM_LINEAR(1);
    case 2: return NVL_NORM_LINEAR(2);
    default: return NVL_NORM_LINEAR(4);
  }
#undef NVL_NORM_LINEAR
}
