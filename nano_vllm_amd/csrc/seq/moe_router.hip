// The router of a mixture of experts in one kernel: logits of up to 64 entries (the shared expert's gate among them) in 32 bits, scores, group limit,
// choices and weights. As passes of their own (a 32-bit copy of the rows, the library's 32-bit product of 33 columns, the route kernel of moe.hip) that
// was 138 us for 13,550 rows of 4,096 (here 30) and 58 of 1,024 (14), and for 64 rows of 1,024 three launches in a chain, 17 us (9).
//
// What bounds it: many rows by reading them (111 MB at 5.1 TB/s, 22 us), few by one chain of requests and by how fast a compute unit takes the router's rows in;
// long reductions of few rows are therefore shared by up to eight workgroups and chosen from by a second launch (64 rows of 4,096: 17 -> 13 us). A workgroup takes 16 MT rows and all entries; its eight
// wavefronts share the reduction as in linear_rows.hip (rings of one piece of 128 bytes of the rows and the same k of the router's rows, straight into
// LDS), the sums meet in LDS, and 4 or 16 lanes per row choose.
//
// bf16 rows times 32-bit weights on the bf16 matrix instructions: a weight is the sum of three bf16 numbers exactly (its leading 8 bits, the next 8 and
// the last 8, each cut off the rest), their products with bf16 entries are exact in 32 bits, and only sums are rounded, as in a 32-bit product; the
// 32-bit instructions take 256 clocks for the 48 of the three. The second and third parts have sums of their own, which are
// added once; where the first part's sum is not finite (an infinity in a row meets zeros in the other parts) it stands alone.
#include "seq_common.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;
typedef __attribute__((address_space(3))) void lds_void_t;
typedef const __attribute__((address_space(1))) void global_void_t;

struct RouterArgs {
  const char* x;
  const float *w, *bias, *correction;
  int64_t ldx;                      // bytes
  int n, K, entries, total, top, count, keep, score, renorm;
  float scale;
  int32_t* ids;
  float *wts, *gate, *parts;        // parts [splits][n][16 NT]: where the reduction is split over workgroups, their sums
  int splits;
};

constexpr int NW = 8, MAX_ROUTER = 64;

// the leading 8 bits of 8 weights as a bf16 operand, and the rest of each
__device__ __forceinline__ u32x4_t cut(float (&v)[8]) {
  u32x4_t out;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const unsigned lo = __builtin_bit_cast(unsigned, v[2 * i]), hi = __builtin_bit_cast(unsigned, v[2 * i + 1]);
    out[i] = __builtin_amdgcn_perm(hi, lo, 0x07060302);               // the upper halves of both
    v[2 * i] -= __builtin_bit_cast(float, lo & 0xffff0000u), v[2 * i + 1] -= __builtin_bit_cast(float, hi & 0xffff0000u);
  }
  return out;
}

constexpr int LD = MAX_ROUTER + 1;                    // logits in LDS: [row][entry]

// the value of a lane N further in the same 16 (or, of four lanes a row, of lane ^ N): plain VALU moves, no LDS
template <int LANES, int N>
__device__ __forceinline__ int other(int v) {
  return __builtin_amdgcn_update_dpp(0, v, LANES == 16 ? 0x120 + N : N == 1 ? 0xB1 : 0x4E, 0xf, 0xf, false);
}
template <int LANES, int N>
__device__ __forceinline__ float other(float v) { return __builtin_bit_cast(float, other<LANES, N>(__builtin_bit_cast(int, v))); }
template <int LANES>
__device__ __forceinline__ float row_max(float v) {
  if constexpr (LANES == 16) v = fmaxf(v, other<LANES, 8>(v)), v = fmaxf(v, other<LANES, 4>(v));
  v = fmaxf(v, other<LANES, 2>(v));
  return fmaxf(v, other<LANES, 1>(v));
}
template <int LANES>
__device__ __forceinline__ float row_sum(float v) {     // (the same number in every lane: additions commute)
  if constexpr (LANES == 16) v += other<LANES, 8>(v), v += other<LANES, 4>(v), v += other<LANES, 2>(v), v += other<LANES, 1>(v);
  else v += other<LANES, 1>(v), v += other<LANES, 2>(v);
  return v;
}
struct Choice {
  float c, s;
  int at;
};
template <int LANES, int N>
__device__ __forceinline__ void better_of(Choice& a) {  // the better choice score; a lower index wins a tie
  const float c = other<LANES, N>(a.c), s = other<LANES, N>(a.s);
  const int at = other<LANES, N>(a.at);
  if (c > a.c || (c == a.c && at < a.at)) a = Choice{c, s, at};
}

// Choices and weights of row r0 + row (row < rows) from its logits in LDS: LANES lanes, lane p of them holds entries p, p + LANES, ... What they tell each other goes
// by moves between lanes; through LDS it took 0.5 us a choice. 16 lanes a row are the shorter chain, four the fewer instructions: 33 entries, four choices, us, four by way of LDS /
// 16 by moves, 64 rows of 1,024 9.5 / 8.1, of 4,096 13.9 / 10.1; 14,200 rows of 1,024, four by way of LDS / 16 / four by moves 14.9 / 16.0 / 14.5.
template <int NT, int LANES>
__device__ __forceinline__ void route_row(const RouterArgs& a, float* z, int r0, int row, int rows) {
  constexpr int PER = NT * 16 / LANES;
  const int lane = threadIdx.x & 63, p = lane & (LANES - 1), p0 = lane & (64 - LANES);
  if (row >= rows || r0 + row >= a.n) return;         // (the row's lanes together)
  float s[PER], c[PER];
  float* zr = z + row * LD;
  float mx = -INFINITY, sum_s = 0.f;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = p + LANES * i;
    s[i] = e < a.total ? zr[e] : -INFINITY;
    mx = fmaxf(mx, s[i]);
  }
  if (a.gate && a.entries > a.total && p == 0) a.gate[r0 + row] = zr[a.total];
  mx = row_max<LANES>(mx);
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = p + LANES * i;
    if (a.score == 1) s[i] = e < a.total ? 1.f / (1.f + expf(-s[i])) : 0.f;
    else s[i] = e < a.total ? expf(s[i] - mx) : 0.f;
    sum_s += s[i];
  }
  sum_s = a.score == 1 ? 1.f : row_sum<LANES>(sum_s);
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = p + LANES * i;
    s[i] = s[i] / sum_s;
    c[i] = e < a.total ? s[i] + (a.correction ? a.correction[e] : 0.f) : -INFINITY;
  }
  if (a.count > 1) {                                // a group's score is its best choice score; entries outside the `keep` best groups cannot be chosen
    const int per = a.total / a.count, inverse = (65536 + per - 1) / per;      // (e * inverse >> 16 is e / per: e < 64)
    float own[PER];                                 // lane p: the scores of groups p, p + LANES, ... (a group has an entry at least: no more of them than entries)
    int better[PER], group[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) group[i] = (p + LANES * i) * inverse >> 16;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      own[j] = -INFINITY, better[j] = 0;
      for (int l = 0; l < LANES && j * LANES + l < a.count; ++l) {
        float v = -INFINITY;
#pragma unroll
        for (int i = 0; i < PER; ++i)
          if (group[i] == j * LANES + l) v = fmaxf(v, c[i]);
        v = row_max<LANES>(v);
        if (p == l) own[j] = v;
      }
    }
#pragma unroll
    for (int j = 0; j < PER; ++j)
      for (int l = 0; l < LANES && j * LANES + l < a.count; ++l) {
        const float v = __shfl(own[j], p0 + l, 64);
#pragma unroll
        for (int i = 0; i < PER; ++i)               // (the number of groups that beat one, a lower index winning a tie)
          if (LANES * i < a.count) better[i] += v > own[i] || (v == own[i] && j * LANES + l < p + LANES * i);
      }
    unsigned long long dropped = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (LANES * j < a.count) dropped |= (__ballot(p + LANES * j < a.count && better[j] >= a.keep) >> p0 & ((1ull << LANES) - 1)) << (LANES * j);
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (dropped >> (group[i] & 63) & 1) c[i] = -INFINITY;      // (entries behind the last one are out anyway)
  }
  float denom = 0.f;                                // lane p holds choices p, p + LANES, ...: written as they come, divided at the end
  for (int k = 0; k < a.top; ++k) {
    Choice best = {-INFINITY, 0.f, 0x7fffffff};
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (c[i] > best.c) best = Choice{c[i], s[i], p + LANES * i};            // (entries of a lane ascend: the first best stays)
    if constexpr (LANES == 16) better_of<LANES, 8>(best), better_of<LANES, 4>(best);
    better_of<LANES, 2>(best), better_of<LANES, 1>(best);
    if (best.at == 0x7fffffff) {                    // nothing that can be chosen (scores that are not numbers): entry 0
      best.at = 0;
      best.s = __shfl(s[0], p0, 64);
    }
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (p + LANES * i == best.at) c[i] = -INFINITY;
    denom += best.s;
    if ((k & (LANES - 1)) == p) {
      a.ids[(int64_t)(r0 + row) * a.top + k] = best.at;
      if (a.renorm) zr[k] = best.s;                 // (the row's logits are no longer read)
      else a.wts[(int64_t)(r0 + row) * a.top + k] = best.s * a.scale;
    }
  }
  if (a.renorm) {
    denom += 1e-20f;
    for (int k = p; k < a.top; k += LANES) a.wts[(int64_t)(r0 + row) * a.top + k] = zr[k] / denom * a.scale;
  }
}

template <typename T, int NT, int MT>
__global__ __launch_bounds__(NW * 64) void moe_router_kernel(RouterArgs a) {
  constexpr bool SPLIT = sizeof(T) == 2;
  constexpr int WROW = SPLIT ? 256 : 128, UNITS = WROW / 16, XB = MT * 16 * 128, WB = NT * 16 * WROW, RING = XB + WB;
  constexpr int XR = MT * 2, WR = WB / 1024, WPR = 1024 / WROW;         // requests, router rows a request covers
  static_assert(NT * MT * 1024 <= RING && NW * RING <= 160 * 1024, "tile");
  extern __shared__ __attribute__((aligned(256))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, lq = lane >> 4;
  const int r0 = blockIdx.x * MT * 16;
  char* ring = lds + wave * RING;
  const char *xs[XR], *ws[WR];                      // rows and entries beyond the last bring the last one's: their results are not read
#pragma unroll
  for (int i = 0; i < XR; ++i) {
    const int r = i * 8 + (lane >> 3), m = r0 + r;
    xs[i] = a.x + (int64_t)(m < a.n ? m : a.n - 1) * a.ldx + ((lane & 7) ^ ((r >> 1) & 7)) * 16;
  }
#pragma unroll
  for (int i = 0; i < WR; ++i) {
    const int r = i * WPR + lane / UNITS, swizzle = SPLIT ? r & 15 : (r >> 1) & 7;
    ws[i] = (const char*)(a.w + (int64_t)(r < a.entries ? r : a.entries - 1) * a.K) + ((lane % UNITS) ^ swizzle) * 16;
  }
  f32x4_t acc[NT][MT], rest[SPLIT ? NT : 1][SPLIT ? MT : 1];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      acc[nt][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if constexpr (SPLIT) rest[nt][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
  const int pieces = a.K / (128 / (int)sizeof(T));
#pragma unroll 1
  for (int s = blockIdx.y * NW + wave; s < pieces; s += NW * a.splits) {
#pragma unroll
    for (int i = 0; i < XR; ++i)
      __builtin_amdgcn_global_load_lds((global_void_t*)(xs[i] + (int64_t)s * 128), (lds_void_t*)(ring + i * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < WR; ++i)
      if (i * WPR < a.entries)                       // (entries that nobody brings are not read either)
        __builtin_amdgcn_global_load_lds((global_void_t*)(ws[i] + (int64_t)s * WROW), (lds_void_t*)(ring + XB + i * 1024), 16, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0F70);              // vmcnt(0): the piece landed
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      u32x4_t x[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) x[mt] = *(const u32x4_t*)(ring + (mt * 16 + li) * 128 + (((h * 4 + lq) ^ ((li >> 1) & 7)) * 16));
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const char* wr = ring + XB + (nt * 16 + li) * WROW;
        if constexpr (SPLIT) {
          const f32x4_t w0 = *(const f32x4_t*)(wr + ((h * 8 + lq * 2) ^ li) * 16), w1 = *(const f32x4_t*)(wr + ((h * 8 + lq * 2 + 1) ^ li) * 16);
          float v[8] = {w0[0], w0[1], w0[2], w0[3], w1[0], w1[1], w1[2], w1[3]};
          const bf16x8_t first = __builtin_bit_cast(bf16x8_t, cut(v)), second = __builtin_bit_cast(bf16x8_t, cut(v)), third = __builtin_bit_cast(bf16x8_t, cut(v));
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            const bf16x8_t xb = __builtin_bit_cast(bf16x8_t, x[mt]);
            acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(first, xb, acc[nt][mt], 0, 0, 0);
            rest[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(second, xb, rest[nt][mt], 0, 0, 0);
            rest[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(third, xb, rest[nt][mt], 0, 0, 0);
          }
        } else {
          const f32x4_t w0 = *(const f32x4_t*)(wr + ((h * 4 + lq) ^ ((li >> 1) & 7)) * 16);
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
              acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(w0[i], __builtin_bit_cast(f32x4_t, x[mt])[i], acc[nt][mt], 0, 0, 0);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);              // lgkmcnt(0): the piece is read, its place can be filled again
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      f32x4_t v = acc[nt][mt];
      if constexpr (SPLIT) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = fabsf(v[i]) < INFINITY ? v[i] + rest[nt][mt][i] : v[i];
      }
      *(f32x4_t*)(ring + ((nt * MT + mt) * 64 + lane) * 16) = v;
    }
  __syncthreads();
  constexpr int ITEMS = NT * MT * 64, HELD = (ITEMS + NW * 64 - 1) / (NW * 64);
  f32x4_t sum[HELD];
#pragma unroll
  for (int i = 0; i < HELD; ++i) {
    const int item = tid + i * NW * 64;
    if (item < ITEMS) {
      sum[i] = *(const f32x4_t*)(lds + item * 16);
#pragma unroll
      for (int ww = 1; ww < NW; ++ww) sum[i] += *(const f32x4_t*)(lds + ww * RING + item * 16);
    }
  }
  if (a.parts) {
#pragma unroll
    for (int i = 0; i < HELD; ++i) {
      const int item = tid + i * NW * 64, tile = item >> 6, l = item & 63, nt = tile / MT, m = r0 + tile % MT * 16 + (l & 15);
      if (item < ITEMS && m < a.n) *(f32x4_t*)(a.parts + ((int64_t)blockIdx.y * a.n + m) * (NT * 16) + nt * 16 + (l >> 4) * 4) = sum[i];
    }
    return;
  }
  __syncthreads();
  float* z = (float*)lds;
#pragma unroll
  for (int i = 0; i < HELD; ++i) {
    const int item = tid + i * NW * 64, tile = item >> 6, l = item & 63, nt = tile / MT, mt = tile % MT;
    if (item < ITEMS) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int e = nt * 16 + (l >> 4) * 4 + k;
        z[(mt * 16 + (l & 15)) * LD + e] = sum[i][k] + (a.bias && e < a.entries ? a.bias[e] : 0.f);
      }
    }
  }
  __syncthreads();
  constexpr int LANES = MT <= 2 ? 16 : 4;
  static_assert(MT * 16 * LANES <= NW * 64, "a row's lanes");
  route_row<NT, LANES>(a, z, r0, tid / LANES, MT * 16);
}

// the sums of a split reduction, added in order, and their choices: 16 rows per workgroup
template <int NT>
__global__ __launch_bounds__(256) void moe_router_parts_kernel(RouterArgs a) {
  __shared__ float z[16 * LD];
  const int r0 = blockIdx.x * 16;
  for (int u = threadIdx.x; u < 16 * NT * 4; u += 256) {
    const int row = u / (NT * 4), e = u % (NT * 4) * 4;
    if (r0 + row >= a.n) break;
    const float* p = a.parts + (int64_t)(r0 + row) * (NT * 16) + e;
    f32x4_t v = *(const f32x4_t*)p;
    for (int s = 1; s < a.splits; ++s) v += *(const f32x4_t*)(p + (int64_t)s * a.n * (NT * 16));
#pragma unroll
    for (int k = 0; k < 4; ++k) z[row * LD + e + k] = v[k] + (a.bias && e + k < a.entries ? a.bias[e + k] : 0.f);
  }
  __syncthreads();
  route_row<NT, 16>(a, z, r0, threadIdx.x / 16, 16);
}

template <typename T, int NT, int MT>
int launch_router(const RouterArgs& a, hipStream_t st) {
  constexpr int LDS = NW * (MT * 16 * 128 + NT * 16 * (sizeof(T) == 2 ? 256 : 128));
  static_assert(LDS >= MT * 16 * LD * 4, "logits");
  const auto kernel = moe_router_kernel<T, NT, MT>;
  NVS_LDS_ROOM(kernel, LDS, "nvs_moe_router");
  kernel<<<dim3((unsigned)((a.n + MT * 16 - 1) / (MT * 16)), (unsigned)a.splits), dim3(NW * 64), LDS, st>>>(a);
  if (a.parts) moe_router_parts_kernel<NT><<<dim3((unsigned)((a.n + 15) / 16)), dim3(256), 0, st>>>(a);
  return nvs_check_launch("nvs_moe_router");
}

template <typename T>
int choose_router(const RouterArgs& a, hipStream_t st) {
  const int nt = (a.entries + 15) / 16;
#define NVS_ROUTER(MT, MT4)                                                    \
  (nt == 1 ? launch_router<T, 1, MT>(a, st) : nt == 2 ? launch_router<T, 2, MT>(a, st) \
                                            : nt == 3 ? launch_router<T, 3, MT>(a, st) : launch_router<T, 4, MT4>(a, st))
  // 16 rows a workgroup until the chip is full, then as few workgroups as fill it: each reads the whole router (from L2)
  if (a.n <= 4096) return NVS_ROUTER(1, 1);
  if (a.n <= 8192) return NVS_ROUTER(2, 2);
  return NVS_ROUTER(4, 2);
#undef NVS_ROUTER
}

}  // namespace

// How many workgroups share a row block's reduction: two launches then, the second one chooses.
static int router_splits(int64_t n, int k, int dtype) {
  const int pieces = k / (dtype == NVS_BF16 ? 64 : 32);
  const int64_t blocks = (n + 15) / 16;
  int splits = 1;
  while (splits < 8 && pieces > 2 * NW * splits && blocks * splits * 2 <= 256) splits *= 2;
  return splits;
}

extern "C" int64_t nvs_moe_router_workspace(int64_t n, int entries, int k, int dtype) {
  const int splits = n > 0 && k > 0 ? router_splits(n, k, dtype) : 1;
  return splits > 1 ? splits * n * ((entries + 15) / 16 * 16) : 0;
}

extern "C" int nvs_moe_router(const void* x, int64_t ldx, int dtype, const float* router, const float* bias, int entries, int k, const float* correction,
                              int64_t n, int total, int top, int count, int keep, float scale, int score, int renorm, int32_t* ids, float* wts,
                              float* gate, float* ws, int64_t ws_floats, void* stream) {
  NVS_REQUIRE(n >= 0 && n < (1ll << 31) - 64 && (dtype == NVS_BF16 || dtype == NVS_F32) && (score == 0 || score == 1), "nvs_moe_router: bad argument");
  if (n == 0) return NVS_OK;
  NVS_REQUIRE(x && router && ids && wts, "nvs_moe_router: null argument");
  NVS_REQUIRE(total > 0 && (entries == total || (entries == total + 1 && gate)) && entries <= MAX_ROUTER && top > 0 && top <= 64 && count > 0 && count <= 64 &&
                  total % count == 0 && keep > 0 && keep <= count && (int64_t)keep * (total / count) >= top,
              "nvs_moe_router: %d entries, %d choices, %d of %d groups", total, top, keep, count);
  const int64_t esize = dtype == NVS_BF16 ? 2 : 4;
  NVS_REQUIRE(k > 0 && k * esize % 128 == 0 && ldx >= k && ldx * esize % 16 == 0 && (((uintptr_t)x | (uintptr_t)router) & 15) == 0,
              "nvs_moe_router: rows of whole 128-byte pieces on 16-byte boundaries (k %d, stride %lld)", k, (long long)ldx);
  const int64_t need = nvs_moe_router_workspace(n, entries, k, dtype);
  const int splits = ws && need ? router_splits(n, k, dtype) : 1;      // (no workspace: one launch)
  NVS_REQUIRE(splits == 1 || (ws_floats >= need && ((uintptr_t)ws & 15) == 0), "nvs_moe_router: workspace of %lld floats is too small", (long long)ws_floats);
  const RouterArgs a{(const char*)x, router, bias, correction, ldx * esize, (int)n, k, entries, total, top, count, keep, score, renorm, scale, ids, wts, gate, splits > 1 ? ws : nullptr, splits};
  return dtype == NVS_BF16 ? choose_router<bf16_t>(a, (hipStream_t)stream) : choose_router<float>(a, (hipStream_t)stream);
}
