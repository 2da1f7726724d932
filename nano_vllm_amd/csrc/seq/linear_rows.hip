// Linear layers of few rows: out[M, N] = x[M, K] . W[N, K]^T (+ bias), bf16 or 32-bit, sums in 32-bit, with a gated activation where one
// follows: the products of a decode step (a row per running sequence) and of short prompts.
//
// What bounds them: the weights are read once, so large ones are bound by memory; small ones (2-12 MB, most layers of width 1,024) by how long one
// chain "request, wait, multiply, add up, store" takes and by what a compute unit can take in (about 50 bytes a clock). So the split is
// for parallel requests and few bytes per unit, not for reuse: a workgroup computes 16 NT weight rows x 16 MT rows of x, its NW wavefronts
// share the reduction (every wavefront every NW-th piece of 128 bytes of k, so that together they read whole neighbouring rows'
// kilobytes), each with a ring of its own of D pieces in LDS, filled from memory without registers: no barrier until the partial sums meet in LDS.
// A row's piece is 128 bytes; its 16-byte unit c sits at c ^ ((row >> 1) & 7), so the 16 rows of an operand read lie on 16
// different bank quads (the requests fetch the units in that order).
//
// Measured on MI355X, weights from memory, graph replay, 64 rows in bf16: 4096 x 1024 4.5 us (the library's product 8.6), 1024 x 2048 4.3 (8.3), 1024 x 1024 3.6
// (8.6), 4096 x 12288 24 (30; the read alone 17 to 21). A decode step of 54 launches, 17 of them library products and 4 activations behind one: 596 us, now 478.
#include "seq_common.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;
typedef __attribute__((address_space(3))) void lds_void_t;
typedef const __attribute__((address_space(1))) void global_void_t;

struct RowsArgs {
  const char *x, *w, *bias;
  char* out;
  int64_t ldx, ldo;                 // bytes, elements
  int M, N, K, tiles_n, tiles_m;    // N: output columns
  int act;
  float limit, alpha;
};

// 16 bytes of k per lane of NT weight-row blocks and MT row blocks: 32 (bf16) or 16 (32-bit) of k. (32-bit: a lane brings the same four
// entries of k in both operands, any order of k will do; products of one sum stay apart, each waits for the one before)
template <typename T, int NT, int MT>
__device__ __forceinline__ void mfma_units(f32x4_t (&acc)[NT][MT], const u32x4_t (&w)[NT], const u32x4_t (&x)[MT]) {
#pragma unroll
  for (int i = 0; i < (sizeof(T) == 2 ? 1 : 4); ++i)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        if constexpr (sizeof(T) == 2)
          acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w[nt]), __builtin_bit_cast(bf16x8_t, x[mt]), acc[nt][mt], 0, 0, 0);
        else
          acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(f32x4_t, w[nt])[i], __builtin_bit_cast(f32x4_t, x[mt])[i], acc[nt][mt], 0, 0, 0);
      }
}

// GLU: a gated activation of glu_value (W: N gate rows, then N up rows), otherwise the sums (+ bias), with act 2 their GELU
template <typename T, int NT, int MT, int NW, int D, bool GLU>
__global__ __launch_bounds__(NW * 64) void linear_rows_kernel(RowsArgs a) {
  constexpr int NG = GLU ? 2 : 1, FT = NT / NG, ROW = 128, STAGE = (NT + MT) * 16 * ROW, NR = (NT + MT) * 2;
  static_assert(NT % NG == 0 && (D - 1) * NR < 64 && NT * MT * 1024 <= D * STAGE, "tile");
  extern __shared__ __attribute__((aligned(128))) char lds[];
  // the row groups of one column tile share its weights: they go to the same XCD (workgroups are dealt round-robin to eight)
  const int j = blockIdx.x / 8, ct = j / a.tiles_m * 8 + blockIdx.x % 8, rt = j % a.tiles_m;
  if (ct >= a.tiles_n) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15;
  const int f0 = ct * FT * 16, r0 = rt * MT * 16;
  const int64_t wrow = (int64_t)a.K * sizeof(T);
  // requests: one covers 8 rows; lane l brings unit (l & 7) ^ swizzle of row l >> 3. Rows beyond the last bring that one's: what is
  // computed from them is not stored.
  const char* src[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int r = i * 8 + (lane >> 3), u = ((lane & 7) ^ ((r >> 1) & 7)) * 16;
    if (i < NT * 2) {
      const int g = r / (FT * 16), f = f0 + r % (FT * 16);
      src[i] = a.w + ((int64_t)g * a.N + (f < a.N ? f : a.N - 1)) * wrow + u;
    } else {
      const int m = r0 + r - NT * 16;
      src[i] = a.x + (int64_t)(m < a.M ? m : a.M - 1) * a.ldx + u;
    }
  }
  char* ring = lds + wave * (D * STAGE);
  const int pieces = (int)(wrow / ROW), mine = (pieces - wave + NW - 1) / NW;
  const auto request = [&](int s) {
    const int64_t k = (int64_t)(s * NW + wave) * ROW;
#pragma unroll
    for (int i = 0; i < NR; ++i)
      __builtin_amdgcn_global_load_lds((global_void_t*)(src[i] + k), (lds_void_t*)(ring + s % D * STAGE + i * 8 * ROW), 16, 0, 0);
  };
  f32x4_t acc[NT][MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < D; ++s)
    if (s < mine) request(s);
  const int unit0 = ((lane >> 4) ^ ((li >> 1) & 7)) * 16;
  const char* op = ring + li * ROW;
#pragma unroll 1
  for (int s = 0; s < mine; ++s) {
    __builtin_amdgcn_sched_barrier(0);
    if (D > 1 && s + D <= mine) __builtin_amdgcn_s_waitcnt(0x0F70 | ((D - 1) * NR & 15) | ((D - 1) * NR >> 4) << 14);   // this piece landed
    else __builtin_amdgcn_s_waitcnt(0x0F70);
    __builtin_amdgcn_sched_barrier(0);
    const char* at = op + s % D * STAGE;
    u32x4_t w[2][NT], x[2][MT];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) w[h][nt] = *(const u32x4_t*)(at + nt * 16 * ROW + (unit0 ^ (h * 64)));
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) x[h][mt] = *(const u32x4_t*)(at + (NT + mt) * 16 * ROW + (unit0 ^ (h * 64)));
    }
    if (s + D < mine) {
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0xC07F);            // the reads of this piece are done: its place can be filled again
      __builtin_amdgcn_sched_barrier(0);
      request(s + D);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) mfma_units<T, NT, MT>(acc, w[h], x[h]);
  }
  // the wavefronts' sums meet: each leaves its own in its ring (nobody else's requests or reads touch it)
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) *(f32x4_t*)(ring + ((nt * MT + mt) * 64 + lane) * 16) = acc[nt][mt];
  __syncthreads();
  typedef __attribute__((ext_vector_type(4))) T t4_t;
  const bool quads = ((a.N | (int)a.ldo) & 3) == 0 && ((uintptr_t)a.out & 15) == 0;
#pragma unroll
  for (int item = tid; item < FT * MT * 64; item += NW * 64) {
    const int tile = item >> 6, ft = tile / MT, mt = tile % MT, l = item & 63;
    f32x4_t v[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const char* p = lds + (((g * FT + ft) * MT + mt) * 64 + l) * 16;
      v[g] = *(const f32x4_t*)p;
#pragma unroll
      for (int ww = 1; ww < NW; ++ww) v[g] += *(const f32x4_t*)(p + ww * (D * STAGE));
    }
    const int f = f0 + ft * 16 + (l >> 4) * 4, m = r0 + mt * 16 + (l & 15);
    if (m >= a.M) continue;
    T* o = (T*)a.out + (int64_t)m * a.ldo + f;
    t4_t t;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (GLU) t[i] = (T)glu_value(v[0][i], v[NG - 1][i], a.act, a.limit, a.alpha);
      else {
        const float z = a.bias && f + i < a.N ? v[0][i] + ldf((const T*)a.bias + f + i) : v[0][i];
        t[i] = (T)(a.act == 2 ? gelu_tanhf_(z) : z);
      }
    }
    if (quads) {
      if (f < a.N) *(t4_t*)o = t;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (f + i < a.N) o[i] = t[i];
    }
  }
}

template <typename T, int NT, int MT, int NW, int D, bool GLU>
int launch_rows(RowsArgs a, hipStream_t st) {
  constexpr int LDS = NW * D * (NT + MT) * 2048, FT = GLU ? NT / 2 : NT;
  a.tiles_n = (a.N + FT * 16 - 1) / (FT * 16), a.tiles_m = (a.M + MT * 16 - 1) / (MT * 16);
  const int64_t blocks = ((int64_t)a.tiles_n + 7) / 8 * 8 * a.tiles_m;
  NVS_REQUIRE(blocks < (1ll << 31), "nvs_linear_rows: product too large");
  const auto kernel = linear_rows_kernel<T, NT, MT, NW, D, GLU>;
  NVS_LDS_ROOM(kernel, LDS, "nvs_linear_rows");
  kernel<<<dim3((unsigned)blocks), dim3(NW * 64), LDS, st>>>(a);
  return nvs_check_launch("nvs_linear_rows");
}

// Clocks of the busiest compute unit for a tile of nt x mt blocks, per 1,024 of k: its workgroups, times the matrix pipe's (a block is 128
// clocks in bf16, 2,048 in 32-bit) and the requests' (16 rows at 50 bytes a clock). It orders the tiles as measured: us, bf16, 64 rows, weights
// of 4096 x 1024 at 1x1 / 2x1 / 2x2 / 2x4 blocks 5.1 / 4.9 / 4.5 / 5.8, 1024 x 1024 3.6 / 3.9 / 4.3 / 5.4, 2048 x 2048 5.6 / 5.3 / 5.6 / 7.4; 256 rows,
// 4096 x 1024, 2x2 / 2x4 / 4x4 9.3 / 9.5 / 7.5; 32-bit, 330 rows, 4096 x 1024 at 2x2 / 2x3 / 2x4 / 4x3 38.5 / 39.7 / 36.3 / 33.6, 1024 x 1024 16.4 / 10.3 / 12.5 / 17.
float tile_clocks(bool wide_type, int nt, int mt, int64_t tiles_n, int64_t tiles_m) {
  const float units = (float)((tiles_n * tiles_m + 255) / 256);
  return wide_type ? units * (2048.f * nt * mt + 1310.f * (nt + mt)) : units * (128.f * nt * mt + 655.f * (nt + mt));
}

template <typename T, bool GLU>
int choose_rows(const RowsArgs& a, hipStream_t st) {
  constexpr bool WIDE = sizeof(T) == 4;
  int best = -1;
  float least = 0.f;
  static constexpr int tile[8][2] = {{1, 1}, {2, 1}, {2, 2}, {2, 4}, {4, 4}, {4, 2}, {2, 3}, {4, 3}};
  for (int i = GLU ? 1 : 0; i < (WIDE ? 8 : 6); ++i) {
    const int ft = 16 * (GLU ? tile[i][0] / 2 : tile[i][0]), rows = 16 * tile[i][1];
    const float c = tile_clocks(WIDE, tile[i][0], tile[i][1], (a.N + ft - 1) / ft, (a.M + rows - 1) / rows);
    if (best < 0 || c < least) best = i, least = c;
  }
  switch (best) {
    case 0: if constexpr (!GLU) return launch_rows<T, 1, 1, 8, 2, GLU>(a, st);
    case 1: return launch_rows<T, 2, 1, 8, 2, GLU>(a, st);
    case 2: return launch_rows<T, 2, 2, 4, WIDE ? 1 : 2, GLU>(a, st);
    case 3: return launch_rows<T, 2, 4, 4, WIDE ? 1 : 2, GLU>(a, st);
    case 4: return launch_rows<T, 4, 4, WIDE ? 4 : 8, 1, GLU>(a, st);
    case 5: return launch_rows<T, 4, 2, 4, WIDE ? 1 : 2, GLU>(a, st);
  }
  if constexpr (WIDE) return best == 6 ? launch_rows<T, 2, 3, 4, 1, GLU>(a, st) : launch_rows<T, 4, 3, 4, 2, GLU>(a, st);
  return NVS_EINVAL;
}

}  // namespace

extern "C" int nvs_linear_rows(const void* x, int64_t ldx, const void* w, const void* bias, int dtype, int64_t m, int n, int k, int act, float limit,
                               float alpha, void* out, int64_t ldo, void* stream) {
  if (m == 0) return NVS_OK;
  NVS_REQUIRE(x && w && out && (dtype == NVS_BF16 || dtype == NVS_F32) && act >= -1 && act <= 2 && (act < 0 || act == 2 || !bias), "nvs_linear_rows: bad argument");
  const int64_t esize = dtype == NVS_BF16 ? 2 : 4;
  NVS_REQUIRE(m > 0 && m < (1ll << 24) && n > 0 && n < (1 << 24) && k > 0 && ldx >= k && ldo >= n, "nvs_linear_rows: %lld x %d x %d", (long long)m, n, k);
  NVS_REQUIRE(k * esize % 128 == 0 && ldx * esize % 16 == 0 && (((uintptr_t)x | (uintptr_t)w) & 15) == 0,
              "nvs_linear_rows: rows of whole 128-byte pieces on 16-byte boundaries (k %d, stride %lld)", k, (long long)ldx);
  const RowsArgs a{(const char*)x, (const char*)w, (const char*)bias, (char*)out, ldx * esize, ldo, (int)m, n, k, 0, 0, act, limit, alpha};
  hipStream_t st = (hipStream_t)stream;
  if (act == 0 || act == 1) return dtype == NVS_BF16 ? choose_rows<bf16_t, true>(a, st) : choose_rows<float, true>(a, st);
  return dtype == NVS_BF16 ? choose_rows<bf16_t, false>(a, st) : choose_rows<float, false>(a, st);
}
