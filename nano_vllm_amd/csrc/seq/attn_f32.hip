// Windowed attention over the paged cache in full precision (32-bit, 128-wide heads or latent rows of 256 with values of 192), on v_mfma_f32_16x16x4_f32. Masks,
// sink, temperature, norms, rotation, gate, caps and pooled blocks mean what they mean in attn_window.hip's scalar kernel, which takes every other size.
//
// The scalar kernel gives a wavefront to every (token, head): a lane reads its key's row alone and the values' columns one key after the other, 112 us for 331
// tokens of 16 heads (keys of 100 tokens on average). Here a workgroup takes 16 query columns, the heads of a kv head (up to 16) times
// as many positions as fill them, and its four wavefronts every fourth tile of 16 keys; operands come from memory as 16-byte loads (a lane brings the same four
// entries of the contraction in both operands: any order will do), the next tile's before this one is multiplied. Everything is computed
// transposed: S^T = K Q^T, O^T += V^T P^T; a lane owns one column (lane & 15) and the weights of its four keys are its operand of the second product as they are.
// What bounds it: per tile of 16 x 16 and wavefront 64 products of 32 clocks and the latency of its loads; us, scalar kernel and here: 331
// tokens in three portions, 16 heads over 8 kv heads 137 and 31, 2,000 9,090 and 360, 64 single tokens behind 200 to 1,500 504 and 125; latent rows, 16 heads, 331 tokens
// 209 and 28. Eight wavefronts instead of four spill (38, 385, 161, 58).
//
// Values of keys that a column does not see weigh 0; where a tile holds values that are not finite, its products are made key by key for the columns that
// see them, so that they reach no other.
#include "attn_window_core.h"

int window_attn_f32(const WindowAttnArgs& a, hipStream_t stream);

namespace {

constexpr float HIDDEN = -3e38f;                  // a masked score: its weight is 0 whatever the maximum is

template <int D, int DV, int NW>
__global__ __launch_bounds__(64 * NW) void window_attn_f32_kernel(const WindowAttnArgs A) {
  constexpr int DC = D / 16, DB = DV / 16;
  extern __shared__ __attribute__((aligned(16))) char parts[];        // outputs [wavefront][DB][64][4], maxima and sums [wavefront][16]
  float2(*ml)[16] = (float2(*)[16])(parts + NW * DB * 1024);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, lq = lane >> 4;
  const int H = A.H, G = A.G, hpg = H / G, hp = A.hw, np = 16 / hp, groups = (hpg + hp - 1) / hp, window = A.window, chunk = A.chunk, bs = A.block_size;
  const int g = blockIdx.y / groups, h0 = g * hpg + blockIdx.y % groups * hp, heads = (g + 1) * hpg - h0 < hp ? (g + 1) * hpg - h0 : hp;
  // the portion of this workgroup's columns: 64 portions at a time, their tile counts summed over the lanes
  int tile = blockIdx.x, s = 0, len = 0, row0 = 0;
  for (int base = 0;; base += 64) {
    const int i = base + lane;
    const int first = i <= A.nseq ? A.cu_q[i] : 0, n_i = i < A.nseq ? A.cu_q[i + 1] - first : 0, tiles = (n_i + np - 1) / np;
    int sum = tiles;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(sum, d, 64);
      sum += lane >= d ? up : 0;
    }
    const uint64_t in = __ballot(tile < sum);
    if (in != 0) {
      const int at = __builtin_ctzll(in);
      s = base + at;
      len = __builtin_amdgcn_readlane(n_i, at);
      row0 = __builtin_amdgcn_readlane(first, at);
      tile -= __builtin_amdgcn_readlane(sum - tiles, at);
      break;
    }
    tile -= __builtin_amdgcn_readlane(sum, 63);
    if (base + 64 >= A.nseq) return;                // the whole workgroup leaves
  }
  tile = (len + np - 1) / np - 1 - tile;            // the last columns of a portion, which see the most, go first
  const int c0 = __builtin_amdgcn_readfirstlane(A.ctx0[s]);
  const int32_t* __restrict__ bt = A.block_tables + (int64_t)s * A.bt_stride;
  const int rel = tile * np + li / hp;
  const bool valid = li / hp < np && li % hp < heads && rel < len;
  const int rel_ok = rel < len && li / hp < np ? rel : len - 1, pos = c0 + rel_ok, h = h0 + (li % hp < heads ? li % hp : 0);
  const int64_t row = (int64_t)row0 + rel_ok;
  const int b_first = c0 + tile * np, b_last = c0 + (tile * np + np < len ? tile * np + np : len) - 1;
  // tiles: [0, npr) hold 16 pooled blocks each, the others 16 tokens, the first from a multiple of 16 on
  const int nb_last = seen_blocks(b_last, window, A.pool), npr = (nb_last + 15) >> 4;
  const int first = vis_lo(b_first, window, chunk) >> 4, tiles = npr + (b_last >> 4) - first + 1;
  f32x4_t kf[DC], vf[DB], kn[DC], vn[DB];
  const auto page_of = [&](int i) { return i >= npr && i < tiles ? bt[((first + i - npr) * 16) >> A.bs_shift] : 0; };
  const auto load = [&](int i, int64_t page, f32x4_t (&k)[DC], f32x4_t (&v)[DB]) {
    const float *kp, *vp;
    int64_t vc;                                     // elements between value columns
    if (i < npr) {
      const int most = (nb_last - 1) >> 3, uk = 2 * i + (li >> 3), uv = 2 * i + (lq >> 1);
      kp = (const float*)A.pool_k + (((int64_t)pool_unit(uk < most ? uk : most, A.pool, bs, bt) * 8 + (li & 7)) * G + g) * D;
      vp = (const float*)A.pool_v + ((int64_t)pool_unit(uv < most ? uv : most, A.pool, bs, bt) * G + g) * DV * 8 + (lq & 1) * 4;
      vc = 8;
    } else {
      const int j0 = (first + i - npr) * 16, off = j0 & (bs - 1);
      kp = (const float*)A.k_cache + (((page << A.bs_shift) + off + li) * G + g) * D;
      vp = (const float*)A.v_cache + (((page * G + g) * DV) << A.bs_shift) + off + lq * 4;
      vc = bs;
    }
#pragma unroll
    for (int c = 0; c < DC; ++c) k[c] = *(const f32x4_t*)(kp + 16 * c + 4 * lq);
#pragma unroll
    for (int db = 0; db < DB; ++db) v[db] = *(const f32x4_t*)(vp + (16 * db + li) * vc);
  };
  int page = page_of(wave);                         // looked up a tile before the loads that use it
  if (wave < tiles) load(wave, page, kn, vn);
  page = page_of(wave + NW);

  // ---- queries: lane holds entries 16 c + 4 lq .. + 3 of its column, normed and turned
  f32x4_t q[DC];
  {
    const float* qp = (const float*)A.q + row * A.q_stride + (int64_t)h * D + 4 * lq;
    const float* qw = (const float*)A.qnorm;
#pragma unroll
    for (int c = 0; c < DC; ++c) q[c] = *(const f32x4_t*)(qp + 16 * c);
    float r = 1.f;
    if (A.q_row) {
      r = A.q_row[row], qw += (int64_t)h * D;       // norm over the whole projection: weights of every head
    } else if (qw) {
      float ss = 0.f;
#pragma unroll
      for (int c = 0; c < DC; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) ss += q[c][e] * q[c][e];
      ss += __shfl_xor(ss, 16, 64), ss += __shfl_xor(ss, 32, 64);
      r = rsqrtf(ss / (float)D + A.eps);
    }
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      if (qw) q[c] *= r * *(const f32x4_t*)(qw + 16 * c + 4 * lq);
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        const int col = 16 * c + 4 * lq + e;
        if (col < A.rot_dims) {                     // the pair (2i, 2i+1) turns by pos * freq[i]
          float sn, cs;
          sincosf((float)pos * A.rot_freq[col >> 1], &sn, &cs);
          const float x = q[c][e], y = q[c][e + 1];
          q[c][e] = x * cs - y * sn, q[c][e + 1] = y * cs + x * sn;
        }
      }
    }
  }
  const float scale = A.scale * query_temp(pos, A.qt_coef, A.qt_every);
  const int nb = seen_blocks(pos, window, A.pool), lo = vis_lo(pos, window, chunk);
  // a sink is a score in the denominator without a value: the first wavefront's sum starts from it (one that weighs nothing beside any score is none)
  const float sink = A.sink && wave == 0 ? A.sink[h] : -INFINITY;
  const bool none = sink < -1e30f;
  float m = none ? -1e30f : sink, l = none || lq != 0 ? 0.f : 1.f;
  f32x4_t o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int i = wave; i < tiles; i += NW) {
#pragma unroll
    for (int c = 0; c < DC; ++c) kf[c] = kn[c];
#pragma unroll
    for (int db = 0; db < DB; ++db) vf[db] = vn[db];
    if (i + NW < tiles) load(i + NW, page, kn, vn);
    page = page_of(i + 2 * NW);
    f32x4_t even = f32x4_t{0.f, 0.f, 0.f, 0.f}, odd = even;
#pragma unroll
    for (int c = 0; c < DC; ++c)
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        even = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[c][e], q[c][e], even, 0, 0, 0);
        odd = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[c][e + 1], q[c][e + 1], odd, 0, 0, 0);
      }
    const bool pooled = i < npr;
    const int j0 = (pooled ? i : first + i - npr) * 16 + 4 * lq, bottom = pooled ? 0 : lo, top = pooled ? nb - 1 : pos;
    float p[4], mx = HIDDEN;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      p[r] = (even[r] + odd[r]) * scale;
      if (A.softcap > 0.f) p[r] = A.softcap * tanhf(p[r] / A.softcap);
      if (j0 + r < bottom || j0 + r > top) p[r] = HIDDEN;
      mx = fmaxf(mx, p[r]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    const float mn = fmaxf(m, fmaxf(mx, __shfl_xor(mx, 32, 64)));
    if (__ballot(mn != m) != 0ull) {
      const float alpha = expf(m - mn);
      l *= alpha;
      m = mn;
#pragma unroll
      for (int db = 0; db < DB; ++db) o[db] *= alpha;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      p[r] = expf(p[r] - m);
      l += p[r];
    }
    if (pooled ? (i + 1) * 16 > nb_last : j0 - 4 * lq + 15 > b_last) {      // what lies behind the last one is nobody's
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (j0 + r > (pooled ? nb_last - 1 : b_last)) {
#pragma unroll
          for (int db = 0; db < DB; ++db) vf[db][r] = 0.f;
        }
    }
    float odd_values = 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r = 0; r < 4; ++r) odd_values += vf[db][r] * 0.f;
    if (__ballot(odd_values != 0.f) == 0ull) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int db = 0; db < DB; ++db) o[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[db][r], p[r], o[db], 0, 0, 0);
    } else {                                        // key by key: column 16 db + 4 lq + r's value is in lane (its column & 15) + 16 (key >> 2)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        for (int k4 = 0; k4 < 4; ++k4) {
          const float w = __shfl(p[r], k4 * 16 + li, 64);
          const int key = (pooled ? i : first + i - npr) * 16 + 4 * k4 + r;
          const bool seen = key >= bottom && key <= top;
#pragma unroll
          for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float v = __shfl(vf[db][r], k4 * 16 + 4 * lq + e, 64);
              if (seen) o[db][e] += w * v;
            }
        }
    }
  }

  // ---- the wavefronts' parts meet in LDS
  l += __shfl_xor(l, 16, 64), l += __shfl_xor(l, 32, 64);
  if (lq == 0) ml[wave][li] = make_float2(m, l);
#pragma unroll
  for (int db = 0; db < DB; ++db) *(f32x4_t*)(parts + ((wave * DB + db) * 64 + lane) * 16) = o[db];
  __syncthreads();
  if (!valid) return;
  float most = -INFINITY, sum = 0.f, f[NW];
#pragma unroll
  for (int w = 0; w < NW; ++w) most = fmaxf(most, ml[w][li].x);
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    f[w] = expf(ml[w][li].x - most);
    sum += f[w] * ml[w][li].y;
  }
  const float inv = 1.f / sum;
  float* op = (float*)A.out + (row * H + h) * DV;
  const float* gp = A.gate ? (const float*)A.gate + row * A.gate_stride + (int64_t)h * A.gate_w : nullptr;
  for (int db = wave; db < DB; db += NW) {
    f32x4_t v = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) v += f[w] * *(const f32x4_t*)(parts + ((w * DB + db) * 64 + lane) * 16);
    const int c = 16 * db + 4 * lq;
    v *= inv;
    if (gp) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] *= 1.f / (1.f + expf(-gp[A.gate_w == 1 ? 0 : c + e]));
    }
    *(f32x4_t*)(op + c) = v;
  }
}

template <int D, int DV, int NW>
int launch_f32(const WindowAttnArgs& a, dim3 grid, hipStream_t stream) {
  constexpr int LDS = NW * (DV / 16 * 1024 + 128);
  const auto kernel = window_attn_f32_kernel<D, DV, NW>;
  NVS_LDS_ROOM(kernel, LDS, "nvs_window_attn");
  kernel<<<grid, dim3(64 * NW), LDS, stream>>>(a);
  return nvs_check_launch("nvs_window_attn (32-bit tiles)");
}

}  // namespace

int window_attn_f32(const WindowAttnArgs& args, hipStream_t stream) {
  WindowAttnArgs a = args;
  const int hpg = a.H / a.G;
  a.hw = hpg < 16 ? hpg : 16;
  a.bs_shift = __builtin_ctz(a.block_size);
  int64_t tiles = a.n / (16 / a.hw) + a.nseq;       // an upper bound: every portion may end with a partial tile, and every tile holds a token
  if (tiles > a.n) tiles = a.n;
  const dim3 grid((unsigned)tiles, (unsigned)(a.G * ((hpg + a.hw - 1) / a.hw)));
  return a.d == 128 ? launch_f32<128, 128, 4>(a, grid, stream) : launch_f32<256, 192, 4>(a, grid, stream);
}
