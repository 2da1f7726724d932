// The gates of the real-gated linear recurrence, up to what its scan reads. Per block of 128 channels r = R u + b_r, i = I u + b_i with 32-bit u and matrices, then
// per token and channel log a = -c sigmoid(r) softplus(lam) and the added term sqrt(1 - a^2) sigmoid(i) u, as pairs [n][channels][2].
//
// The products run on the 16-bit matrix instructions without giving up the 32 bits: a 32-bit number is exactly the sum of three bfloat16 numbers, products of those are exact
// in 32 bits, and the instruction adds them in 32. Matrices that came from a 16-bit checkpoint are their first part alone: three products, a fifth of the
// 32-bit instructions' time. Others (a workgroup sees that when it cuts its matrices up) take eight, all that reach the last place of the sum.
//
// A workgroup of eight wavefronts keeps the parts of 64 channels' two matrices in LDS (96 KB, [part][128 features][128]); a wavefront takes 32 rows at a time, loads them
// straight into the order the instruction reads, a pass ahead, and splits them there. Lane: a token, four neighbouring channels of both gates, so the gates'
// arithmetic happens where the sums are and a token's 16 channels leave as one 128-byte line.
//
// An infinity is its first part alone, but its products with another number's parts that are 0 are not numbers: where the matrices or a pass's rows hold one, results that
// are no numbers are summed up again in 32 bits as they stand.
//
// What bounds it: the gates' arithmetic (two sigmoids, an exponential, 1 - a^2 and its root: about 70 vector instructions per value, 140 us of 57 million values) beside
// 690 MB of traffic (135 us) and 75 us of products. 13,550 tokens, 4,096 channels: 230 to 250 us; a library product in 32 bits with the bias copied in
// front of it took 595, and both passes of the scan did the arithmetic again (213 + 307 us; reading pairs 80 + 153).
#include "seq_common.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;

constexpr int BW = 128, SLICE = 64, PARTS = 3, PART_BYTES = 2 * SLICE * BW * 2;

struct Split {
  bf16x8_t part[PARTS];
};
__device__ __forceinline__ Split split8(const f32x4_t& lo, const f32x4_t& hi) {
  Split s;
#pragma unroll
  for (int i = 0; i < 8; ++i) {                     // 8 bits of the significand each; an infinity is its first part alone
    float v = i < 4 ? lo[i & 3] : hi[i & 3];
#pragma unroll
    for (int k = 0; k < PARTS; ++k) {
      const uint32_t bits = __builtin_bit_cast(uint32_t, v) & 0xffff0000u;
      const float p = __builtin_bit_cast(float, bits);
      s.part[k][i] = __builtin_bit_cast(__bf16, (uint16_t)(bits >> 16));
      v = k == 0 && v == p ? 0.f : v - p;
    }
  }
  return s;
}

template <typename T>
__global__ __launch_bounds__(512) void rglru_gates_kernel(const float* __restrict__ u, const float* __restrict__ w, const float* __restrict__ bias,
                                                          const T* __restrict__ lam, float c, int channels, int blocks, int64_t n, int rows,
                                                          float* __restrict__ pairs) {
  extern __shared__ __attribute__((aligned(128))) char lds[];
  __shared__ int more, odd;                         // some entry is more than its first part; some entry is not finite
  __shared__ float plus[SLICE];                     // softplus(lam)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, q = lane >> 4;
  const int slices = blocks * (BW / SLICE), slice = blockIdx.x % slices, blk = slice / (BW / SLICE), half = slice % (BW / SLICE);
  const int64_t begin = (int64_t)(blockIdx.x / slices) * rows, end = begin + rows < n ? begin + rows : n;
  const float* ub = u + blk * BW;
  f32x4_t x[4][2][2];
  const auto bring = [&](int64_t at) {
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const int64_t r = at + rb * 16 + li < end ? at + rb * 16 + li : end - 1;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const f32x4_t* from = (const f32x4_t*)(ub + r * channels + s * 32 + q * 8);
        x[s][rb][0] = from[0];
        x[s][rb][1] = from[1];
      }
    }
  };
  int64_t at = begin + wave * 32;
  if (at < end) bring(at);
  // feature row f (gate r: f < 64) of a part: 16-byte unit k8 at k8 ^ (f & 15)
  if (tid == 0) more = odd = 0;
  if (tid < SLICE) plus[tid] = softplusf_(ldf(lam + blk * BW + half * SLICE + tid));
  __syncthreads();
  const float* wb = w + (int64_t)blk * BW * 2 * BW + half * SLICE;
  bool mine = false;
  float odd_entries = 0.f;
  constexpr int ITEMS = 2 * SLICE * BW / 8 / 512;
  const int f = tid % (2 * SLICE);
  f32x4_t lo[ITEMS], hi[ITEMS];                     // (asked for together: their way here is most of a decode step's time)
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const float* from = wb + (int64_t)(tid + i * 512) / (2 * SLICE) * 8 * 2 * BW + f / SLICE * BW + f % SLICE;
#pragma unroll
    for (int j = 0; j < 4; ++j) lo[i][j] = from[j * 2 * BW], hi[i][j] = from[(j + 4) * 2 * BW];
  }
#pragma unroll
  for (int i = 0; i < ITEMS; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) odd_entries += lo[i][j] * 0.f + hi[i][j] * 0.f;
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int k8 = (tid + i * 512) / (2 * SLICE);
    const Split s = split8(lo[i], hi[i]);
#pragma unroll
    for (int k = 0; k < PARTS; ++k) {
      const u32x4_t bits = __builtin_bit_cast(u32x4_t, s.part[k]);
      *(u32x4_t*)(lds + k * PART_BYTES + f * BW * 2 + ((k8 ^ (f & 15)) << 4)) = bits;
      if (k > 0) mine |= ((bits[0] | bits[1] | bits[2] | bits[3]) & 0x7fff7fffu) != 0;
    }
  }
  if (mine) more = 1;
  if (odd_entries != 0.f) odd = 1;
  __syncthreads();
  const bool whole = more == 0, odd_matrices = odd != 0;
  const int c0 = blk * BW + half * SLICE + q * 4;   // this lane's channels: c0 + 16 fb + 0..3
  float sp[4][4];
#pragma unroll
  for (int fb = 0; fb < 4; ++fb)
#pragma unroll
    for (int i = 0; i < 4; ++i) sp[fb][i] = plus[q * 4 + fb * 16 + i];
  const float* br = bias + (int64_t)blk * 2 * BW + half * SLICE + q * 4;
#pragma unroll 1
  for (; at < end; at += 256) {
    f32x4_t acc[8][2];
#pragma unroll
    for (int fb = 0; fb < 8; ++fb) acc[fb][0] = acc[fb][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    bool strange = odd_matrices;
    if (!whole) {
      f32x4_t odd_rows = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) odd_rows += (x[s][0][0] * 0.f + x[s][0][1] * 0.f) + (x[s][1][0] * 0.f + x[s][1][1] * 0.f);
      strange |= __ballot(odd_rows[0] + odd_rows[1] + odd_rows[2] + odd_rows[3] != 0.f) != 0;
    }
    const auto operand = [&](int part, int fb, int s) {
      return *(const bf16x8_t*)(lds + part * PART_BYTES + (fb * 16 + li) * BW * 2 + (((s * 4 + q) ^ li) << 4));
    };
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      __builtin_amdgcn_sched_barrier(0);              // (moved together, the splits of all steps need registers that are not there)
      const Split a = split8(x[s][0][0], x[s][0][1]), b = split8(x[s][1][0], x[s][1][1]);
#pragma unroll
      for (int fb = 0; fb < 8; ++fb) {
        const bf16x8_t w0 = operand(0, fb, s);
#pragma unroll
        for (int k = PARTS - 1; k >= 0; --k) {
          acc[fb][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0, a.part[k], acc[fb][0], 0, 0, 0);
          acc[fb][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0, b.part[k], acc[fb][1], 0, 0, 0);
        }
      }
      if (!whole) {
#pragma unroll
        for (int fb = 0; fb < 8; ++fb)
#pragma unroll
          for (int p = 1; p < PARTS; ++p) {
            const bf16x8_t wp = operand(p, fb, s);
#pragma unroll
            for (int k = PARTS - p; k >= 0; --k) {
              acc[fb][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wp, a.part[k], acc[fb][0], 0, 0, 0);
              acc[fb][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wp, b.part[k], acc[fb][1], 0, 0, 0);
            }
          }
      }
    }
    const int64_t now = at;
    if (at + 256 < end) bring(at + 256);
#pragma unroll
    for (int fb = 0; fb < 4; ++fb) {
      __builtin_amdgcn_sched_barrier(0);
      const f32x4_t b_r = *(const f32x4_t*)(br + fb * 16), b_i = *(const f32x4_t*)(br + BW + fb * 16);
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        const int64_t t = now + rb * 16 + li;
        if (t >= end) continue;
        const f32x4_t uv = *(const f32x4_t*)(u + t * channels + c0 + fb * 16);
        f32x4_t out[2];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const RglruTerms v = rglru_terms(acc[fb][rb][i] + b_r[i], acc[fb + 4][rb][i] + b_i[i], uv[i], sp[fb][i], c);
          out[i >> 1][(i & 1) * 2] = v.la;
          out[i >> 1][(i & 1) * 2 + 1] = v.add;
        }
        f32x4_t* to = (f32x4_t*)(pairs + (t * channels + c0 + fb * 16) * 2);
        to[0] = out[0];
        to[1] = out[1];
      }
    }
    if (strange) {                                  // this lane's results again, those that are no numbers
#pragma unroll 1
      for (int j = 0; j < 32; ++j) {
        const int64_t t = now + (j >> 4) * 16 + li;
        const int ch = c0 + (j >> 2 & 3) * 16 + (j & 3), in_block = ch - blk * BW;
        if (t >= end) continue;
        float* to = pairs + (t * channels + ch) * 2;
        if (to[0] == to[0] && to[1] == to[1]) continue;
        const float* col = w + (int64_t)blk * BW * 2 * BW + in_block;
        const float* bs = bias + (int64_t)blk * 2 * BW + in_block;
        float gr = 0.f, gi = 0.f;
#pragma unroll 1
        for (int k = 0; k < BW; ++k) {
          const float uk = ub[t * channels + k];
          gr = fmaf(col[k * 2 * BW], uk, gr), gi = fmaf(col[k * 2 * BW + BW], uk, gi);
        }
        const RglruTerms v = rglru_terms(gr + bs[0], gi + bs[BW], u[t * channels + ch], plus[in_block - half * SLICE], c);
        to[0] = v.la;
        to[1] = v.add;
      }
    }
  }
}

}  // namespace

extern "C" int nvs_rglru_gates(const float* u, const float* w, const float* bias, const void* lam, int dtype, float c, int channels, int blocks, int64_t n,
                               float* pairs, void* stream) {
  if (n == 0) return NVS_OK;
  NVS_REQUIRE(u && w && bias && lam && pairs && n > 0 && blocks > 0 && channels == blocks * BW, "nvs_rglru_gates: %d channels in %d blocks", channels, blocks);
  NVS_REQUIRE((((uintptr_t)u | (uintptr_t)bias | (uintptr_t)pairs) & 15) == 0 && ((uintptr_t)w & 3) == 0, "nvs_rglru_gates: addresses");
  const int64_t slices = (int64_t)blocks * (BW / SLICE), passes = (n + 255) / 256, wanted = slices < 256 ? 256 / slices : 1;
  const int64_t rows = (passes + wanted - 1) / wanted * 256, grid = (n + rows - 1) / rows * slices;
  NVS_REQUIRE(grid < (1ll << 31) && rows < (1ll << 31), "nvs_rglru_gates: step too large");
  NVS_DISPATCH(dtype, {
    const auto kernel = rglru_gates_kernel<T>;
    NVS_LDS_ROOM(kernel, PARTS * PART_BYTES, "nvs_rglru_gates");
    kernel<<<dim3((unsigned)grid), dim3(512), PARTS * PART_BYTES, (hipStream_t)stream>>>(u, w, bias, (const T*)lam, c, channels, blocks, n, (int)rows, pairs);
  });
  return nvs_check_launch("nvs_rglru_gates");
}
