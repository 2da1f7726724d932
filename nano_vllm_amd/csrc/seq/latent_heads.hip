// Latent attention's products per head: y[t, a, :] = W_a x[t, a, :]. In front of the attention W_uk,a^T takes a head's unrotated query part into the latent space, and
// the rotated part goes behind it in the same pass; behind the attention W_uv,a takes its output back out.
//
// Bound by memory: a head's weights are 48 KB (128 x 192), a row's entries are read once and written once. A workgroup of four wavefronts keeps one head's
// weights in LDS ([N][K]; W_uk is stored [K][N] and turned on the way in, 8 x 8 entries per lane) for all its rows; a wavefront takes 32 rows at a time, which it
// loads straight into the registers the matrix instruction reads (lane: row lane & 15, 8 entries of k) a tile ahead of their use, so nobody waits for anybody. The
// results of 16 rows go through LDS so that a store writes whole rows. Heads follow the workgroup number, so an XCD meets the same few heads' weights. About 512
// workgroups: two fit on a compute unit, and fewer rows per workgroup would only load the weights more often.
//
// MI355X, 14,000 rows, 16 heads, 128 -> 192 + 64 turned entries: 57 us (a batched product and the rotation 95); 192 -> 128:
// 29 us (46).
#include "seq_common.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2_t;

struct LatentArgs {
  const bf16_t *x, *w;
  bf16_t* y;
  const float2* turn;      // [n][rot_dims / 2]: cos and sin of a row's pairs
  int64_t n, ldx, ldy;     // entries from row to row
  int xh, yh, rows;        // entries from head to head; rows of a workgroup
  int H, tail, rot_dims, halves;      // tail: entries behind x's K that go behind y's N
  int lanes_log;
};

// 16-byte unit u of row r of [rows][units] sits at u ^ swizzle(r): 16 rows of one unit lie on 16 different bank quads
template <int UNITS>
__device__ __forceinline__ int place(int r, int u) {
  return r * UNITS + (u ^ (UNITS % 16 == 0 ? r & 15 : (r >> 1) & 7));
}

// the part behind of 32 rows: its leading rot_dims entries turn. A lane keeps one pair (2^p.lanes_log lanes per row) and asks for 8 rows' at once
__device__ __forceinline__ void turn_tail(const LatentArgs& p, const bf16_t* from, bf16_t* to, int64_t at, int64_t end, int lane) {
  const int per = 64 >> p.lanes_log, half = p.rot_dims >> 1, pairs = p.tail >> 1, rows = (int)min<int64_t>(32, end - at);
  for (int c = lane & ((1 << p.lanes_log) - 1); c < pairs; c += 64) {
    const bool turns = c < half, apart = turns && p.halves;
    const int f = apart ? c : 2 * c, s = apart ? c + half : 2 * c + 1;
#pragma unroll 1
    for (int r0 = lane >> p.lanes_log; r0 < rows; r0 += 8 * per) {
      bf16_t u[8], v[8];                     // (16-bit accesses: pairs side by side as one of 32 bits and a choice between the two took 61 us for 57)
      float2 cs[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int64_t t = at + min(r0 + j * per, rows - 1);
        u[j] = from[t * p.ldx + f];
        v[j] = from[t * p.ldx + s];
        if (turns) cs[j] = p.turn[t * half + c];
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float a = (float)u[j], b = (float)v[j];
        if (turns) u[j] = (bf16_t)(a * cs[j].x - b * cs[j].y), v[j] = (bf16_t)(b * cs[j].x + a * cs[j].y);
        if (r0 + j * per < rows) {
          bf16_t* row = to + (at + r0 + j * per) * p.ldy;
          row[f] = u[j];
          row[s] = v[j];
        }
      }
    }
  }
}

template <int K, int N, bool TURNED>
__global__ __launch_bounds__(256) void latent_heads_kernel(LatentArgs p) {
  constexpr int KS = K / 32, NB = N / 16, KU = K / 8, NU = N / 8;
  extern __shared__ __attribute__((aligned(128))) char lds[];
  u32x4_t* wl = (u32x4_t*)lds;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, q = lane >> 4;
  u32x4_t* mine = (u32x4_t*)(lds + K * N * 2) + wave * 16 * NU;
  const int a = blockIdx.x % p.H;
  const int64_t begin = (int64_t)(blockIdx.x / p.H) * p.rows, end = min(begin + p.rows, p.n);
  const bf16_t* xa = p.x + (int64_t)a * p.xh;
  bf16_t* ya = p.y + (int64_t)a * p.yh;
  u32x4_t x[KS][2];
  const auto bring = [&](int64_t at) {
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const int64_t r = min(at + rb * 16 + li, end - 1);                // (rows behind the last one: that one again, nobody stores it)
#pragma unroll
      for (int s = 0; s < KS; ++s) x[s][rb] = *(const u32x4_t*)(xa + r * p.ldx + s * 32 + q * 8);
    }
  };
  int64_t at = begin + wave * 32;
  if (at < end) bring(at);
  const bf16_t* wa = p.w + (int64_t)a * K * N;
  if constexpr (TURNED) {
    for (int i = tid; i < KU * NU; i += 256) {                          // 8 x 8 entries: 8 rows of k, 8 features
      const int f8 = i % NU, k8 = i / NU;
      union { u32x4_t q; uint16_t h[8]; } in[8], out;
#pragma unroll
      for (int j = 0; j < 8; ++j) in[j].q = *(const u32x4_t*)(wa + (k8 * 8 + j) * N + f8 * 8);
#pragma unroll
      for (int f = 0; f < 8; ++f) {
#pragma unroll
        for (int j = 0; j < 8; ++j) out.h[j] = in[j].h[f];
        wl[place<KU>(f8 * 8 + f, k8)] = out.q;
      }
    }
  } else {
    for (int i = tid; i < KU * N; i += 256) wl[place<KU>(i / KU, i % KU)] = *(const u32x4_t*)(wa + i * 8);
  }
  __syncthreads();
#pragma unroll 1
  for (; at < end; at += 128) {
    f32x4_t acc[NB][2];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb][0] = acc[nb][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const bf16x8_t w = __builtin_bit_cast(bf16x8_t, wl[place<KU>(nb * 16 + li, s * 4 + q)]);
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
          acc[nb][rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, __builtin_bit_cast(bf16x8_t, x[s][rb]), acc[nb][rb], 0, 0, 0);
      }
    if (at + 128 < end) bring(at + 128);
    // lane: row li of a block, features 16 nb + 4 q + 0..3
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        union { bf16_t h[4]; u32x2_t d; } o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o.h[i] = (bf16_t)acc[nb][rb][i];
        ((u32x2_t*)(mine + place<NU>(li, nb * 2 + (q >> 1))))[q & 1] = o.d;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int j = 0; j < NU / 4; ++j) {
        const int v = j * 64 + lane, r = v / NU, u = v % NU;
        const u32x4_t o = mine[place<NU>(r, u)];
        if (at + rb * 16 + r < end) *(u32x4_t*)(ya + (at + rb * 16 + r) * p.ldy + u * 8) = o;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    if (TURNED && p.tail) turn_tail(p, xa + K, ya + N, at, end, lane);
  }
}

template <int K, int N, bool TURNED>
int launch_heads(LatentArgs p, hipStream_t st) {
  constexpr int LDS = K * N * 2 + 4 * 16 * N * 2;
  const auto kernel = latent_heads_kernel<K, N, TURNED>;
  NVS_LDS_ROOM(kernel, LDS, "nvs_latent_heads");
  const int64_t tiles = (p.n + 127) / 128, chunks = 512 / p.H > 0 ? 512 / p.H : 1;
  p.rows = (int)((tiles + chunks - 1) / chunks) * 128;
  const int64_t blocks = (p.n + p.rows - 1) / p.rows * p.H;
  NVS_REQUIRE(blocks < (1ll << 31), "nvs_latent_heads: step too large");
  kernel<<<dim3((unsigned)blocks), dim3(256), LDS, st>>>(p);
  return nvs_check_launch("nvs_latent_heads");
}

template <bool TURNED>
int heads_of(const LatentArgs& p, int K, int N, hipStream_t st) {
#define NVS_HEADS(k, n) \
  if (K == k && N == n) return launch_heads<k, n, TURNED>(p, st)
#define NVS_HEADS_N(k) NVS_HEADS(k, 64); NVS_HEADS(k, 128); NVS_HEADS(k, 192); NVS_HEADS(k, 256)
  NVS_HEADS_N(64);
  NVS_HEADS_N(128);
  NVS_HEADS_N(192);
  NVS_HEADS_N(256);
#undef NVS_HEADS_N
#undef NVS_HEADS
  NVS_REQUIRE(false, "nvs_latent_heads: heads of %d -> %d", K, N);
}

}  // namespace

extern "C" int nvs_latent_heads(const void* x, int64_t ldx, int xh, const void* w, int turned, int K, int N, void* y, int64_t ldy, int yh, int H, int tail,
                                int rot_dims, int rot_halves, const void* turn, int64_t n, void* stream) {
  if (n == 0) return NVS_OK;
  NVS_REQUIRE(x && w && y && n > 0 && n < (1ll << 31) && H > 0 && K > 0 && N > 0 && tail >= 0 && tail % 2 == 0 && (turned || tail == 0), "nvs_latent_heads: bad argument");
  NVS_REQUIRE(xh >= K + tail && yh >= N + tail && ldx >= (int64_t)(H - 1) * xh + K + tail && ldy >= (int64_t)(H - 1) * yh + N + tail &&
                  ((ldx | xh | ldy | yh) & 7) == 0 && (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15) == 0,
              "nvs_latent_heads: %d heads of %d -> %d in rows of %lld and %lld", H, K, N, (long long)ldx, (long long)ldy);
  NVS_REQUIRE(rot_dims >= 0 && rot_dims % 2 == 0 && rot_dims <= tail && (rot_dims == 0 || (turn && ((uintptr_t)turn & 7) == 0)), "nvs_latent_heads: rotation of %d of %d entries",
              rot_dims, tail);
  LatentArgs p{(const bf16_t*)x, (const bf16_t*)w, (bf16_t*)y, (const float2*)turn, n, ldx, ldy, xh, yh, 0, H, tail, rot_dims, rot_halves, 0};
  while (p.lanes_log < 6 && (2 << p.lanes_log) < tail) ++p.lanes_log;
  return turned ? heads_of<true>(p, K, N, (hipStream_t)stream) : heads_of<false>(p, K, N, (hipStream_t)stream);
}
