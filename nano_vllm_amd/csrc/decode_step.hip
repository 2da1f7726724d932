// All layers of a decode step of up to four sequences in one launch (Qwen3-0.6B's shape: width 1,024, two query heads over a kv head).
//
// As launches of their own the layers' parts (norm + qkv, attention, merge + o, norm + gate|up, down) are 140 dependent ones of 4 to 8 us: 31 MB of weights a
// layer are read in 6, and the rest is the way from one launch to the next and its first requests' way to memory. Here 256 workgroups stay, and a phase's outputs go to the
// next one's readers as words that say of themselves whether they have been written: the exchange memory starts as kEmpty everywhere (a NaN that is never
// stored), a reader asks for the words it needs until none is empty. No flag, no fence, no cache write-back lies between the two: words are stored and loaded
// past the caches that are not shared (relaxed, agent scope), each is read for itself, and every word is written once a step. The weights of later phases are requested before the
// wait of an earlier one. A phase that does nothing but hand 8 KB on takes 1.7 us this way, one with 32 KB of weights a workgroup 2.6 (a launch 3.3 and more).
//
// Forward progress. Items (a phase's shares) have an order, and an item waits for items before it alone. When all 256 workgroups are seen to run at once (they count themselves
// at the start), each takes the item of its own number in every phase. When they are not all there in time (other launches hold their places), the step's mode becomes
// "dealt": items are taken in order from a counter, so whoever holds the first unfinished one can go on, with any number of workgroups on the chip. One word, changed once by
// compare-and-swap, holds the decision for all. Waits are bounded all the same: a reader that has asked in vain as often as its caller allows says so, in a sync word and in the
// caller's, and then goes on with what is there, a NaN, which makes the rows it is part of NaN. Such a key or value of the new token is not stored once the sync word is set: it is
// looked at behind the words that the row is made of, and set in front of everything that a reader who gave up leads to.
//
// A workgroup is eight wavefronts that multiply and four that fetch. A matrix is cut into 256 shares of 16 operand rows: 16 output features of the whole reduction (qkv), or 8
// features in halves of the reduction (gate|up, 4 + 4 features a tile, three tiles), or 4 features in quarters (o, down); the other operand's columns are (row, part of
// the reduction), so 16 x 16 products of which those on the diagonal count cover four rows. The wavefronts share the reduction, their sums meet in LDS.
//   v = residual + bf16(y) stays in 32 bits on its way into a norm, the residual is bf16(v), as in linear_norm.hip; attention as in attn_decode.hip, but the weights of
//   the values stay in 32 bits.
// What bounds it: six hand-overs a layer of 1.2 us and the work between them (attention 1.9 us, a product 0.5, a norm 0.3); 31 MB of weights are under way meanwhile. MI355X,
// Qwen3-0.6B, whole steps with the output head's 75 us, launches apart / here, one sequence of 30, 700, 2,047 and 4,000 tokens 748 810 871 914 / 486 497 533 604 us; two of
// 450 and 900 842 / 544; three of 700, 1,000 and 1,500 910 / 653; four of 60, 2,000, 4,000 810 961 1094 / 557 830 1033 (keys and values alone are 370 us of it).
#include "rope_common.h"

namespace {

constexpr unsigned int kEmpty = 0xFFFFFFFFu;
constexpr int kGroups = 256, kMulWaves = 8, kFetchWaves = 4, kThreads = 64 * (kMulWaves + kFetchWaves);
constexpr int kMaxLayers = 40, kWidth = 1024, kMaxFf = 3072, kMaxParts = 32;
constexpr int kChunk = 32;                       // keys the multiplying wavefronts take at once: four each
constexpr int kHeld = 4;                         // chunks requested ahead
constexpr float kNegBig = -1.0e30f, kHidden = -3e38f;
// Pauses before a phase's words are first asked for, about 100 clocks each. An answer "empty" takes 0.7 us as any other does, and 256 workgroups that ask without a pause keep the
// few channels the words lie on busy: a phase that hands 8 KB on took 2.2 us so and 1.6 with 1,300 clocks between handing on and asking. 14 to 26 for 20, 35 to 65 for 50
// and 45 to 80 for 60 are the same step within 1 %; gate|up with 14, 20, 26: 503, 497, 492 us a step.
constexpr int kPause = 20, kPauseGateUp = 28, kPauseMerge = 50, kPauseMerged = 16, kPauseParts = 60, kPauseIdle = 20;

struct StepLayer {
  const bf16_t *norm1, *wqkv, *qn, *kn, *wo, *norm2, *wgu, *wd;
  bf16_t *kc, *vc;
};

struct StepArgs {
  StepLayer layer[kMaxLayers];
  const float* cos_sin;
  const int32_t *tables, *ctx;
  unsigned int* ws;                              // sync words [64]; then the layers' exchange words; then v of the step's input
  float* hidden;
  bf16_t* residual;
  int32_t* gave_up;
  int64_t bt_stride, max_pos;
  float eps, scale_log2e;
  int layers, rows, hq, hkv, ff, block_size, parts, asks;
};

// words of a layer's exchange, in order
struct Exchange {
  int qkv, po, ml, att, v1, act, v2, total;      // offsets
  __host__ __device__ Exchange(int rows, int hq, int hkv, int ff, int parts) {
    qkv = 0;
    po = qkv + rows * (hq + 2 * hkv) * 64;
    ml = po + rows * hq * parts * 128;
    att = ml + rows * hq * parts * 2;
    v1 = att + rows * hq * 64;
    act = v1 + rows * kWidth;
    v2 = act + rows * ff / 2;
    total = v2 + rows * kWidth;
  }
};
// sync words: [0] workgroups that have come, [1] the mode (0 open, 1 fixed, 2 dealt), [2] the next share, [3] looks before the mode is dealt, [4] whether a wait gave up; and the
// contexts' cut: keys of a row's parts, and parts of the rows before it
constexpr int kSyncWords = 64, kCutKeys = 8, kCutBefore = 16;

// The contexts' cut into parts of whole chunks, rows * parts of them at most in all; the new token is the last key of its row's last part, a row of no context has one part too.
// Contexts about alike get `parts` each. Where the longest one's would be longer by more than a chunk than parts of one length that cut all contexts, it is those (at most kMaxParts of a
// context). Us a step, launches apart / `parts` each / parts of one length, contexts of 4,000 and three of 100 960 / 971 / 685, of 4,000 and three of 1,000 976 / 1008 / 803, of 3,000,
// 1,500, 700 and 50 943 / 890 / 731; of 1,500, 1,000 and 700 910 / 653 / 670, of three of 1,100 and one of 1,431 - / 712 / 720: chunks behind the four held ahead are what the parts wait for.
// (By the launch before the step: in the step itself it took four rows 12 to 20 us, for what it left of the registers.)
__device__ void cut_contexts(unsigned int* ws, const int32_t* ctx, int rows, int parts) {
  const auto chunks = [&](int b) { return (max(ctx[b], 0) + kChunk - 1) / kChunk; };
  int sum = 0, most = 0;
  for (int b = 0; b < rows; ++b) sum += chunks(b), most = max(most, chunks(b));
  const int all = rows * parts, longest = (most + parts - 1) / parts;
  int c = max((sum + all - 1) / all, (most + kMaxParts - 1) / kMaxParts);
  for (; c < longest; ++c) {                     // (rows' last parts may be short)
    int n = 0;
    for (int b = 0; b < rows; ++b) n += max((chunks(b) + c - 1) / c, 1);
    if (n <= all) break;
  }
  ws[kCutBefore] = 0;
  for (int b = 0, n = 0; b < rows; ++b) {
    const int of = max(longest <= c + 1 ? (chunks(b) + parts - 1) / parts : c, 1);
    ws[kCutKeys + b] = of * kChunk;
    ws[kCutBefore + b + 1] = n += max((chunks(b) + of - 1) / of, 1);
  }
}

__device__ __forceinline__ void group_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0xC07F);            // lgkmcnt(0): what went to LDS is there (requests to memory stay on their way)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void hand(unsigned int* p, unsigned int w) {
  __hip_atomic_store(p, w == kEmpty ? 0x7FFF7FFFu : w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);        // (a NaN either way)
}
__device__ __forceinline__ void hand(unsigned int* p, float v) { hand(p, __float_as_uint(v)); }
__device__ __forceinline__ bool there(const u32x4_t& w) { return w[0] != kEmpty && w[1] != kEmpty && w[2] != kEmpty && w[3] != kEmpty; }
__device__ __forceinline__ bool there(const u32x2_t& w) { return w[0] != kEmpty && w[1] != kEmpty; }
__device__ __forceinline__ __amdgpu_buffer_rsrc_t words(const unsigned int* p, int n) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, n * 4, 0x00020000);        // (beyond n: zeros)
}
constexpr int kPastCaches = 16;                  // sc1: agent scope

// lanes l, l ^ 16, l ^ 32, l ^ 48
__device__ __forceinline__ float rows_sum(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
__device__ __forceinline__ float rows_max(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

template <int MR>
struct __attribute__((aligned(128))) StepShared {
  static constexpr int kRow = kMaxFf * 2 + 64;   // bytes of a row of the products' right operand
  unsigned char act[MR * kRow];
  float red[kMulWaves * 3 * 2 * 4 * 8 > 2048 ? kMulWaves * 3 * 2 * 4 * 8 : 2048];        // the wavefronts' sums: a matrix's, or the attention's [8][2][128]
  float ml[kMulWaves][2][2];
  unsigned int head[4][64];                      // attention: two rotated queries, the new key and value
  float res[4][4], ss[4][4], den;
  int item, mode;
};

template <int MR>
struct Step {
  const StepArgs& a;
  StepShared<MR>& sh;
  const Exchange ex;
  int tid, lane, wave, l4;                       // l4: lane among the fetching wavefronts
  bool broken = false;
  u32x4_t wa[4], wo[2], wg[3][2], wd[3], kr[kHeld], vr[kHeld];
  u32x2_t n1, n2;

  __device__ __forceinline__ Step(const StepArgs& args, StepShared<MR>& s)
      : a(args), sh(s), ex(args.rows, args.hq, args.hkv, args.ff, args.parts), tid(threadIdx.x), lane(threadIdx.x & 63),
        wave(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)), l4(threadIdx.x - 64 * kMulWaves) {}
  // The lane's numbers as if new: addresses made of them would be kept in registers over the layers otherwise, more of them than there are, and what goes to scratch memory
  // comes back behind the weights on their way (a step of 700 tokens took 690 us with 27 registers spilled).
  __device__ __forceinline__ void afresh() {
    asm volatile("" : "+v"(tid));
    lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l4 = tid - 64 * kMulWaves;
  }
  __device__ __forceinline__ bool multiplies() const { return wave < kMulWaves; }
  __device__ __forceinline__ unsigned int* slot(int l) const { return a.ws + kSyncWords + (int64_t)l * ex.total; }
  // v in front of layer l: the step's input behind all layers' words, or the second sum of the layer before
  __device__ __forceinline__ unsigned int* v_in(int l) const { return l == 0 ? slot(a.layers) : slot(l - 1) + ex.v2; }

  // ---- shares -----------------------------------------------------------------------------------------------------
  __device__ __forceinline__ int shares_qkv() const { return (a.hq + 2 * a.hkv) * 8; }
  __device__ __forceinline__ int shares_attention() const { return a.rows * a.hkv * a.parts; }
  __device__ __forceinline__ int shares_merge() const { return a.rows * a.hq; }

  // (32-bit offsets from a base in scalar registers: a matrix has less than 4 GB)
  __device__ __forceinline__ static u32x4_t weight(const bf16_t* m, uint32_t at) {
    return *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const unsigned char*>(m) + at);
  }
  template <int FROM, int TO>
  __device__ __forceinline__ void load_qkv(int l, int item) {
    afresh();
    const uint32_t at = ((item * 16 + (lane & 15)) * kWidth + wave * 128 + (lane >> 4) * 8) * 2u;
#pragma unroll
    for (int s = FROM; s < TO; ++s) wa[s] = weight(a.layer[l].wqkv, at + s * 64u);
  }
  // four features of a reduction of K in quarters
  template <int N>
  __device__ __forceinline__ void load_quarters(u32x4_t (&w)[N], const bf16_t* m, int K, int item) {
    afresh();
    const int S = K / 1024;
    const uint32_t at = ((item * 4 + (lane & 3)) * K + ((lane >> 2) & 3) * (K / 4) + wave * S * 32 + (lane >> 4) * 8) * 2u;
#pragma unroll
    for (int s = 0; s < N; ++s) w[s] = weight(m, at + (s < S ? s : 0) * 64u);        // (without a branch: registers that may be left as they are count as held)
  }
  __device__ __forceinline__ void load_gate_up(int l, int item) {
    afresh();
    const int T = a.ff / 1024, j = lane & 7;
    const uint32_t at = (((j < 4 ? 0 : a.ff) + item * T * 4 + (j & 3)) * kWidth + ((lane >> 3) & 1) * 512 + wave * 64 + (lane >> 4) * 8) * 2u;
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
      for (int s = 0; s < 2; ++s) wg[t][s] = weight(a.layer[l].wgu + (t < T ? t : 0) * 4 * kWidth, at + s * 64u);
  }

  // ---- fetching ---------------------------------------------------------------------------------------------------
  __device__ __forceinline__ void give_up() {
    if (!broken && lane == 0) {
      __hip_atomic_store(a.ws + 4, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (a.gave_up) __hip_atomic_store(a.gave_up, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    broken = true;
    __builtin_amdgcn_s_waitcnt(0x0F70);          // vmcnt(0): the words are there before the barrier behind which this phase's results are handed on
  }
  // N units of 16 bytes a lane, `units` in all; and one more, at byte `at` of another place
  template <int N, bool ONE>
  __device__ __forceinline__ void fetch(const unsigned int* src, int units, u32x4_t (&v)[N], const unsigned int* one, int at, u32x4_t& w) {
    const auto rs = words(src, units * 4);
    const auto r1 = words(one, ONE ? a.rows * kWidth : 0);
    for (int asks = 0;; ++asks) {
      asm volatile("" ::: "memory");
#pragma unroll
      for (int i = 0; i < N; ++i) v[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, (l4 + 256 * i) * 16, 0, kPastCaches);
      if constexpr (ONE) w = __builtin_amdgcn_raw_buffer_load_b128(r1, at, 0, kPastCaches);
      bool ok = true;
#pragma unroll
      for (int i = 0; i < N; ++i) ok = ok && there(v[i]);
      if constexpr (ONE) ok = ok && there(w);
      if (__all(ok)) break;
      if (broken || asks >= a.asks) {
        give_up();
        break;
      }
    }
  }

  // the rows of v, normed, as the products' right operand
  __device__ __forceinline__ void fetch_normed(const unsigned int* v, const u32x2_t& nw) {
    u32x4_t w[MR], none;
    fetch<MR, false>(v, a.rows * 256, w, nullptr, 0, none);
    float ss[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) s += __uint_as_float(w[m][i]) * __uint_as_float(w[m][i]);
      ss[m] = wave_allreduce_sum(s);
    }
    if (lane == 0) {
#pragma unroll
      for (int m = 0; m < MR; ++m) sh.ss[m][wave - kMulWaves] = ss[m];
    }
    group_barrier();
    const float g[4] = {bf16lo_to_f32(nw[0]), bf16hi_to_f32(nw[0]), bf16lo_to_f32(nw[1]), bf16hi_to_f32(nw[1])};
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      const f32x4_t s = *reinterpret_cast<const f32x4_t*>(sh.ss[m]);
      const float rstd = rsqrtf(((s[0] + s[1]) + (s[2] + s[3])) / (float)kWidth + a.eps);
      float o[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = g[i] * (__uint_as_float(w[m][i]) * rstd);
      *reinterpret_cast<u32x2_t*>(sh.act + m * StepShared<MR>::kRow + l4 * 8) = u32x2_t{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
    }
  }
  // rows of 16-bit words (units of 16 bytes a row), and the residual beside the share's features
  template <int N>
  __device__ __forceinline__ void fetch_rows(const unsigned int* src, int row_units, const unsigned int* v, int item) {
    u32x4_t w[N], r;
    fetch<N, true>(src, a.rows * row_units, w, v, (l4 * kWidth + item * 4) * 4, r);        // (lanes beyond the rows: zeros)
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int u = l4 + 256 * i, m = u / row_units;
      if (m < a.rows) *reinterpret_cast<u32x4_t*>(sh.act + m * StepShared<MR>::kRow + (u - m * row_units) * 16) = w[i];
    }
    if (l4 < a.rows) {
#pragma unroll
      for (int i = 0; i < 4; ++i) sh.res[l4][i] = round_bf16(__uint_as_float(r[i]));
    }
  }
  __device__ __forceinline__ bf16x8_t operand(int m, int k) const {
    return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(sh.act + (m < MR ? m : MR - 1) * StepShared<MR>::kRow + k * 2));
  }
  __device__ __forceinline__ static f32x4_t mul(const u32x4_t& w, const bf16x8_t& x, const f32x4_t& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w), x, c, 0, 0, 0);
  }

  // ---- phases -----------------------------------------------------------------------------------------------------
  __device__ __forceinline__ void qkv_fetch(int l) {
    afresh();
    fetch_normed(v_in(l), n1);
    group_barrier();
    group_barrier();
    group_barrier();
  }
  __device__ __forceinline__ void qkv(int l, int item) {
    afresh();
    group_barrier();
    group_barrier();
    const int col = lane & 15, kg = lane >> 4;
    f32x4_t c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) c = mul(wa[s], operand(col, wave * 128 + s * 32 + kg * 8), c);
    if (col < MR) *reinterpret_cast<f32x4_t*>(&sh.red[(wave * 4 + col) * 16 + kg * 4]) = c;
    group_barrier();
    const int p = tid & 7, f = (tid >> 3) & 15, m = tid >> 7;            // a wavefront's sum, a feature, a row
    const float y = half8_allreduce_sum(sh.red[(p * 4 + (m < MR ? m : 0)) * 16 + f]);
    const float other = row16_ror8(y);
    if (m < a.rows && p == 0 && !(f & 1)) hand(slot(l) + ex.qkv + m * (a.hq + 2 * a.hkv) * 64 + item * 8 + f / 2, pack_bf16x2(y, other));
    group_barrier();
  }

  // the sum of four features' quarters: lanes of one (row, feature) hold the eight wavefronts' shares
  template <int N>
  __device__ __forceinline__ float quarters(const u32x4_t (&w)[N], int K, int& m, int& j) {
    const int col = lane & 15, kg = lane >> 4, S = K / 1024, q = col >> 2;
    f32x4_t c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < N; ++s)
      if (s < S) c = mul(w[s], operand(col & 3, q * (K / 4) + (wave * S + s) * 32 + kg * 8), c);
    if (q == kg && (col & 3) < MR) *reinterpret_cast<f32x4_t*>(&sh.red[((wave * 4 + q) * 4 + (col & 3)) * 4]) = c;
    group_barrier();
    const int p = tid & 7;
    j = (tid >> 3) & 3, m = tid >> 5;                                    // (rows 0 .. 3: the first two wavefronts)
    float y = 0.f;
    if (m < MR) {
#pragma unroll
      for (int i = 0; i < 4; ++i) y += sh.red[((p * 4 + i) * 4 + m) * 4 + j];
    }
    return half8_allreduce_sum(y);
  }

  __device__ __forceinline__ void out_fetch(int l, int item) {
    afresh();
    fetch_rows<MR>(slot(l) + ex.att, a.hq * 16, v_in(l), item);
    group_barrier();
    group_barrier();
    group_barrier();
  }
  __device__ __forceinline__ void out_projection(int l, int item) {
    afresh();
    group_barrier();
    int m, j;
    const float y = quarters(wo, a.hq * 128, m, j);
    if (m < a.rows && (tid & 7) == 0) hand(slot(l) + ex.v1 + m * kWidth + item * 4 + j, round_bf16(y) + sh.res[m][j]);
    group_barrier();
  }

  __device__ __forceinline__ void gate_up_fetch(int l) {
    afresh();
    fetch_normed(slot(l) + ex.v1, n2);
    group_barrier();
    group_barrier();
    group_barrier();
  }
  __device__ __forceinline__ void gate_up(int l, int item) {
    afresh();
    group_barrier();
    group_barrier();
    const int col = lane & 15, kg = lane >> 4, T = a.ff / 1024, half = (col >> 2) & 1;
    f32x4_t c[3];
#pragma unroll
    for (int t = 0; t < 3; ++t) c[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const bf16x8_t x = operand(col & 3, half * 512 + wave * 64 + s * 32 + kg * 8);
#pragma unroll
      for (int t = 0; t < 3; ++t)
        if (t < T) c[t] = mul(wg[t][s], x, c[t]);
    }
    // operand rows 4 kg ..: half kg / 2, features 4 (kg & 1) .. (0: of the gate, 1: of up)
    if (col < 8 && half == kg >> 1 && (col & 3) < MR) {
#pragma unroll
      for (int t = 0; t < 3; ++t)
        if (t < T) *reinterpret_cast<f32x4_t*>(&sh.red[(((wave * 3 + t) * 2 + half) * 4 + (col & 3)) * 8 + (kg & 1) * 4]) = c[t];
    }
    group_barrier();
    const int p = tid & 3, j = (tid >> 2) & 7, r = tid >> 5, t = r % 3, m = r / 3;        // two wavefronts' halves each; a feature; a tile; a row
    float y = 0.f;
    if (m < MR && t < T) {
#pragma unroll
      for (int i = 0; i < 4; ++i) y += sh.red[((((p * 2 + (i >> 1)) * 3 + t) * 2 + (i & 1)) * 4 + m) * 8 + j];
    }
    y += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(y), 0xB1, 0xf, 0xf, false));        // quad_perm [1,0,3,2]
    y += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(y), 0x4E, 0xf, 0xf, false));        // quad_perm [2,3,0,1]
    y = round_bf16(y);
    const float up = __shfl_xor(y, 16, 64);
    const float z = y / (1.f + __expf(-y)) * up;
    const float next = __shfl_xor(z, 4, 64);
    if (m < a.rows && t < T && p == 0 && j < 4 && !(j & 1))
      hand(slot(l) + ex.act + m * (a.ff / 2) + (item * T + t) * 2 + j / 2, pack_bf16x2(z, next));
    group_barrier();
  }

  __device__ __forceinline__ void down_fetch(int l, int item) {
    afresh();
    fetch_rows<(3 * MR + 1) / 2>(slot(l) + ex.act, a.ff / 8, slot(l) + ex.v1, item);
    group_barrier();
    group_barrier();
    group_barrier();
  }
  __device__ __forceinline__ void down(int l, int item) {
    afresh();
    group_barrier();
    int m, j;
    const float y = round_bf16(quarters(wd, a.ff, m, j));
    if (m < a.rows && (tid & 7) == 0) {
      const int at = m * kWidth + item * 4 + j;
      if (l + 1 < a.layers) {
        hand(slot(l) + ex.v2 + at, y + sh.res[m][j]);
      } else {                                   // the last norm adds them
        a.hidden[at] = y;
        a.residual[at] = (bf16_t)sh.res[m][j];
      }
    }
    group_barrier();
  }

  // ---- attention --------------------------------------------------------------------------------------------------
  struct Place {                                 // a share of the attention: a kv head of part `at` of all
    int b, h, at, per, first, end, len;          // keys first .. end - 1, of `per`
    bool last, whole;                            // the context's last part; its only one
  };
  __device__ __forceinline__ int word(int i) const { return __builtin_amdgcn_readfirstlane((int)a.ws[i]); }      // of the cut (scalar: a branch on others would wait for the weights on their way)
  __device__ __forceinline__ int before(int b) const { return word(kCutBefore + b); }
  __device__ __forceinline__ int parts(int b) const { return before(b + 1) - before(b); }
  __device__ __forceinline__ Place place(int item) const {
    const int at = item / a.hkv;
    int b = 0;
    while (b + 1 < a.rows && at >= before(b + 1)) ++b;
    const int part = at - before(b), n = parts(b), len = a.ctx[b], per = word(kCutKeys + b), first = part * per;
    return Place{b, item - at * a.hkv, at, per, first, min(max(len, 0), first + per), len, part == n - 1, n == 1};
  }
  // element of a layer's cache where this lane's 16 bytes of token `key` lie (inside the cache whatever the context is)
  __device__ __forceinline__ int64_t row_of(const Place& at, int key) const {
    key = max(0, min(key, at.len - 1));
    const int blk = max(a.tables[at.b * a.bt_stride + key / a.block_size], 0);
    return (((int64_t)blk * a.hkv + at.h) * a.block_size + key % a.block_size) * 128 + (lane & 15) * 8;
  }
  __device__ __forceinline__ void first_keys(const Place& at, int64_t (&from)[kHeld]) const {
#pragma unroll
    for (int i = 0; i < kHeld; ++i)              // (keys that are not the part's: its last one again)
      from[i] = row_of(at, min(at.first + i * kChunk + wave * 4 + (lane >> 4), at.end - 1));
  }
  __device__ __forceinline__ void load_kv(int l, const int64_t (&at)[kHeld], int keys) {
#pragma unroll
    for (int i = 0; i < kHeld; ++i)
      if (i == 0 || keys > i * kChunk) {
        kr[i] = *reinterpret_cast<const u32x4_t*>(a.layer[l].kc + at[i]);
        vr[i] = *reinterpret_cast<const u32x4_t*>(a.layer[l].vc + at[i]);
      }
  }

  struct Online {
    float m[2], l[2], o[2][8];
  };
  // keys in registers: lane group g of wavefront w holds key 32 i + 4 w + g, 8 dims a lane
  template <int N>
  __device__ __forceinline__ void attend(Online& x, const float (&q)[2][8], const u32x4_t* k, const u32x4_t* v, const bool* seen) const {
    float s[N][2];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      float f[8];
      unpack8(k[i], f);
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        float d = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) d += q[g][e] * f[e];
        s[i][g] = seen[i] ? row16_allreduce_sum(d) * a.scale_log2e : kHidden;
      }
    }
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      float top = x.m[g];
#pragma unroll
      for (int i = 0; i < N; ++i) top = fmaxf(top, s[i][g]);
      const float r = __builtin_amdgcn_exp2f(x.m[g] - top);
      x.m[g] = top;
      x.l[g] *= r;
#pragma unroll
      for (int e = 0; e < 8; ++e) x.o[g][e] *= r;
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      float f[8];
      const u32x4_t none = {0u, 0u, 0u, 0u};
      unpack8(seen[i] ? v[i] : none, f);         // (what a page holds behind the context need not be finite)
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const float p = __builtin_amdgcn_exp2f(s[i][g] - x.m[g]);
        x.l[g] += p;
#pragma unroll
        for (int e = 0; e < 8; ++e) x.o[g][e] += p * f[e];
      }
    }
  }

  // q heads h * 2, h * 2 + 1 normed and rotated (first fetching wavefront), the new key and value (second one, the last part's)
  __device__ __forceinline__ void fetch_heads(int l, const Place& at, bool last) {
    const int fw = wave - kMulWaves, sub = lane & 15, r = lane >> 4;
    if (fw > 1 || (fw == 1 && !last) || at.len <= 0) return;
    const int64_t pos = at.len - 1 >= a.max_pos ? a.max_pos - 1 : at.len - 1;
    const RopeRegs rr = load_rope_regs(a.cos_sin + pos * 128, sub);
    const bf16_t* nw = fw == 0 ? a.layer[l].qn : a.layer[l].kn;
    u32x4_t wraw = {0u, 0u, 0u, 0u};
    if (nw != nullptr) wraw = *reinterpret_cast<const u32x4_t*>(nw + sub * 8);
    const int head = fw == 0 ? at.h * 2 + (r & 1) : a.hq + (r & 1) * a.hkv + at.h;
    const auto rs = words(slot(l) + ex.qkv + at.b * (a.hq + 2 * a.hkv) * 64, (a.hq + 2 * a.hkv) * 64);
    u32x4_t raw;
    for (int asks = 0;; ++asks) {
      asm volatile("" ::: "memory");
      raw = __builtin_amdgcn_raw_buffer_load_b128(rs, head * 256 + sub * 16, 0, kPastCaches);
      if (__all(there(raw))) break;
      if (broken || asks >= a.asks) {
        give_up();
        break;
      }
    }
    const bool odd = broken || __any((raw[0] & 0x7FFFu) > 0x7F80u);        // words that were given up elsewhere make NaN of a whole row
    const u32x4_t turned = norm_rope_head_regs(raw, nw != nullptr, wraw, a.eps, rr, sub);
    const u32x4_t row = fw == 1 && (r & 1) ? raw : turned;
    if (r < 2) *reinterpret_cast<u32x4_t*>(&sh.head[fw * 2 + r][sub * 4]) = row;
    bool keep = true;
    if (odd) {                                   // (an answer takes 0.7 us: no other row asks. Us a step of one sequence of 700 tokens, never asking 495.6, so 497.5, in every row 505)
      asm volatile("" ::: "memory");
      keep = __hip_atomic_load(a.ws + 4, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0;
    }
    if (fw == 1 && r < 2 && keep) *reinterpret_cast<u32x4_t*>((r == 0 ? a.layer[l].kc : a.layer[l].vc) + row_of(at, at.len - 1)) = row;        // for later steps
  }

  __device__ __forceinline__ void attention_fetch(int l, const Place& at) {
    afresh();
    fetch_heads(l, at, at.last);
    group_barrier();
    group_barrier();
    group_barrier();
  }
  // (the first chunks' keys and values have been requested)
  __device__ __forceinline__ void attention(int l, const Place& at) {
    afresh();
    const bool last = at.last;
    const int sub = lane & 15, r = lane >> 4, first = at.first, end = at.end;
    group_barrier();
    float q[2][8];
#pragma unroll
    for (int g = 0; g < 2; ++g) unpack8(*reinterpret_cast<const u32x4_t*>(&sh.head[g][sub * 4]), q[g]);
    Online x;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      x.m[g] = kNegBig, x.l[g] = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) x.o[g][e] = 0.f;
    }
    // two chunks at a time, the next two of their place requested behind them
    const auto two = [&](u32x4_t* k, u32x4_t* v, int key0) {
      bool seen[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int key = key0 + i * kChunk + wave * 4 + r;
        seen[i] = key < end;
        if (last && key == at.len - 1) {         // the new token: its place in the cache is not read
          k[i] = *reinterpret_cast<const u32x4_t*>(&sh.head[2][sub * 4]);
          v[i] = *reinterpret_cast<const u32x4_t*>(&sh.head[3][sub * 4]);
        }
      }
      if (end - key0 <= kChunk) attend<1>(x, q, k, v, seen);
      else attend<2>(x, q, k, v, seen);
      if (key0 + kHeld * kChunk < end) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int64_t from = row_of(at, min(key0 + (kHeld + i) * kChunk + wave * 4 + r, end - 1));
          k[i] = *reinterpret_cast<const u32x4_t*>(a.layer[l].kc + from);
          v[i] = *reinterpret_cast<const u32x4_t*>(a.layer[l].vc + from);
        }
      }
    };
#pragma unroll 1
    for (int key0 = first; key0 < end; key0 += kHeld * kChunk) {
      two(kr, vr, key0);
      if (key0 + 2 * kChunk < end) two(kr + 2, vr + 2, key0 + 2 * kChunk);
    }
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const float top = rows_max(x.m[g]), f = __builtin_amdgcn_exp2f(x.m[g] - top);
      x.m[g] = top;
      x.l[g] = rows_sum(x.l[g] * f);
#pragma unroll
      for (int e = 0; e < 8; ++e) x.o[g][e] = rows_sum(x.o[g][e] * f);
    }
    if (r < 2) {
      float* to = &sh.red[(wave * 2 + r) * 128 + sub * 8];
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        f32x4_t o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = r == 0 ? x.o[0][e + i] : x.o[1][e + i];
        *reinterpret_cast<f32x4_t*>(to + e) = o;
      }
      if (sub == 0) sh.ml[wave][r][0] = r == 0 ? x.m[0] : x.m[1], sh.ml[wave][r][1] = r == 0 ? x.l[0] : x.l[1];
    }
    group_barrier();
    if (tid < 256) {
      const int g = tid >> 7, d = tid & 127;
      float M = kNegBig, num = 0.f, den = 0.f;
  #pragma unroll
      for (int w = 0; w < kMulWaves; ++w) M = fmaxf(M, sh.ml[w][g][0]);
  #pragma unroll
      for (int w = 0; w < kMulWaves; ++w) {
        const float f = __builtin_amdgcn_exp2f(sh.ml[w][g][0] - M);
        num += f * sh.red[(w * 2 + g) * 128 + d];
        den += f * sh.ml[w][g][1];
      }
      const int row = at.b * a.hq + at.h * 2 + g, place = (at.h * 2 + g) * a.rows * a.parts + at.at;
      if (at.whole) {
        const float o = at.len > 0 ? num / den : 0.f;        // (len 0: a row that fills up a captured step)
        const float next = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(o), 0xB1, 0xf, 0xf, false));
        if (!(d & 1)) hand(slot(l) + ex.att + row * 64 + d / 2, pack_bf16x2(o, next));
      } else {
        hand(slot(l) + ex.po + place * 128 + d, num);
        if (d < 2) hand(slot(l) + ex.ml + place * 2 + d, d == 0 ? M : den);
      }
    }
    group_barrier();
  }

  // a head's n parts, the first of them at place `from` (head by head, all rows' parts)
  __device__ __forceinline__ int parts_of(int row) const { return (row % a.hq) * a.rows * a.parts + before(row / a.hq); }
  __device__ __forceinline__ void merge_fetch(int l, int from, int n) {
    afresh();
    const int fw = wave - kMulWaves;
    const auto ro = words(slot(l) + ex.po + from * 128, n * 128), rm = words(slot(l) + ex.ml + from * 2, n * 2);
    u32x2_t o[kMaxParts / 4], w;
    for (int asks = 0;; ++asks) {
      asm volatile("" ::: "memory");
      w = __builtin_amdgcn_raw_buffer_load_b64(rm, lane * 8, 0, kPastCaches);
      bool ok = there(w);
#pragma unroll
      for (int i = 0; i < kMaxParts / 4; ++i) o[i] = __builtin_amdgcn_raw_buffer_load_b64(ro, ((i * 4 + fw) * 64 + lane) * 8, 0, kPastCaches);
#pragma unroll
      for (int i = 0; i < kMaxParts / 4; ++i) ok = ok && there(o[i]);
      if (__all(ok)) break;
      if (broken || asks >= a.asks) {
        give_up();
        break;
      }
    }
    const float m = lane < n ? __uint_as_float(w[0]) : kNegBig;
    const float M = wave_allreduce_max(m);
    const float f = lane < n ? __builtin_amdgcn_exp2f(m - M) : 0.f, den = wave_allreduce_sum(lane < n ? f * __uint_as_float(w[1]) : 0.f);
    float lo = 0.f, hi = 0.f;
#pragma unroll
    for (int i = 0; i < kMaxParts / 4; ++i) {
      const float fi = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f), i * 4 + fw));        // (0 behind the last part)
      lo += fi * __uint_as_float(o[i][0]), hi += fi * __uint_as_float(o[i][1]);
    }
    *reinterpret_cast<float2*>(&sh.red[fw * 128 + lane * 2]) = make_float2(lo, hi);
    if (fw == 0 && lane == 0) sh.den = den;
    group_barrier();
    group_barrier();
  }
  __device__ __forceinline__ void merge(int l, int row) {
    afresh();
    group_barrier();
    if (wave == 0) {
      float2 s = make_float2(0.f, 0.f);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float2 p = *reinterpret_cast<const float2*>(&sh.red[i * 128 + lane * 2]);
        s.x += p.x, s.y += p.y;
      }
      hand(slot(l) + ex.att + row * 64 + lane, pack_bf16x2(s.x / sh.den, s.y / sh.den));
    }
    group_barrier();                             // (the sums' place is free again)
  }

  __device__ __forceinline__ void load_norms(int l) {
    afresh();
    n1 = *reinterpret_cast<const u32x2_t*>(a.layer[l].norm1 + l4 * 4);
    n2 = *reinterpret_cast<const u32x2_t*>(a.layer[l].norm2 + l4 * 4);
  }

  // every workgroup is there: each takes the share of its number
  __device__ __forceinline__ void run_fixed() {
    const int me = blockIdx.x;
    const bool att = me < before(a.rows) * a.hkv, has_qkv = me < shares_qkv();
    const Place at = place(att ? me : 0);
    const int first_merge = kGroups - shares_merge();        // (the workgroups behind the attention's: step_parts leaves them)
    const int row = me >= first_merge ? me - first_merge : 0;
    const int n = parts(row / a.hq), parts_at = parts_of(row);
    const bool merges = me >= first_merge && n > 1, parted = before(a.rows) > a.rows;
    if (multiplies()) {                          // (two loops: neither holds the other's registers)
      int64_t from[kHeld];
      first_keys(at, from);
      // A request waits for those in front of it, of the whole workgroup: the words that are handed on, and those of the next phase, for weights. So weights are asked for behind
      // a phase's words, most of them where the next phase is far away (behind the attention, whose parts are merged first). In us, one sequence of 700 tokens: every
      // matrix in front of its own phase 579, behind the fetch of the phase before 576, behind its words 539, gate|up and down behind the attention's 499; qkv in parts
      // of 1 + 3, 2 + 2, 4 + 0 and 0 + 4 of its four pieces 497 497 520 511.
      const int qkv_item = has_qkv ? me : 0;
      load_qkv<0, 4>(0, qkv_item);
      load_kv(0, from, at.per);
#pragma unroll 1
      for (int l = 0; l < a.layers; ++l) {
        const int after = min(l + 1, a.layers - 1);
        if (has_qkv) qkv(l, me);
        load_quarters(wo, a.layer[l].wo, a.hq * 128, me);
        if (att) attention(l, at);
        else pause(kPauseIdle);                  // (the others' queries first)
        load_gate_up(l, me);
        load_quarters(wd, a.layer[l].wd, a.ff, me);
        if (merges) merge(l, row);
        out_projection(l, me);
        load_qkv<0, 1>(after, qkv_item);
        gate_up(l, me);
        load_qkv<1, 4>(after, qkv_item);
        down(l, me);
        load_kv(after, from, at.per);
      }
    } else {
#pragma unroll 1
      for (int l = 0; l < a.layers; ++l) {
        load_norms(l);
        if (l > 0) pause(kPause);
        if (has_qkv) qkv_fetch(l);
        pause(kPause);
        if (att) attention_fetch(l, at);
        if (merges) {                            // (it has no attention)
          pause(kPauseMerge);
          merge_fetch(l, parts_at, n);
        }
        pause(merges ? kPauseMerged : parted ? kPauseParts : kPause);
        out_fetch(l, me);
        pause(kPauseGateUp);
        gate_up_fetch(l);
        pause(kPause);
        down_fetch(l, me);
      }
    }
  }
  __device__ __forceinline__ static void pause(int n) {
    for (int i = 0; i < n; ++i) __builtin_amdgcn_s_sleep(1);
  }

  // shares in order from a counter
  int share = 0;
  __device__ __forceinline__ void next() {
    group_barrier();
    if (tid == 0) sh.item = (int)__hip_atomic_fetch_add(a.ws + 2, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    group_barrier();
    share = __builtin_amdgcn_readfirstlane(sh.item);
  }
  __device__ __forceinline__ void run_dealt() {
    const bool muls = multiplies();
    int base = 0;
    next();
#pragma unroll 1
    for (int l = 0; l < a.layers; ++l) {
#pragma unroll 1
      for (; share < base + shares_qkv(); next()) {
        if (muls) load_qkv<0, 4>(l, share - base), qkv(l, share - base);
        else load_norms(l), qkv_fetch(l);
      }
      base += shares_qkv();
#pragma unroll 1
      for (; share < base + shares_attention(); next()) {
        if (share - base >= before(a.rows) * a.hkv) continue;
        const Place at = place(share - base);
        if (muls) {
          int64_t from[kHeld];
          first_keys(at, from);
          load_kv(l, from, at.per);
          attention(l, at);
        } else {
          attention_fetch(l, at);
        }
      }
      base += shares_attention();
#pragma unroll 1
      for (; share < base + shares_merge(); next()) {
        const int row = share - base, n = parts(row / a.hq);
        if (n == 1) continue;
        if (muls) merge(l, row);
        else merge_fetch(l, parts_of(row), n);
      }
      base += shares_merge();
#pragma unroll 1
      for (; share < base + kGroups; next()) {
        if (muls) load_quarters(wo, a.layer[l].wo, a.hq * 128, share - base), out_projection(l, share - base);
        else out_fetch(l, share - base);
      }
      base += kGroups;
#pragma unroll 1
      for (; share < base + kGroups; next()) {
        if (muls) load_gate_up(l, share - base), gate_up(l, share - base);
        else load_norms(l), gate_up_fetch(l);
      }
      base += kGroups;
#pragma unroll 1
      for (; share < base + kGroups; next()) {
        if (muls) load_quarters(wd, a.layer[l].wd, a.ff, share - base), down(l, share - base);
        else down_fetch(l, share - base);
      }
      base += kGroups;
    }
  }
};

template <int MR>
__global__ __launch_bounds__(kThreads) void decode_step_kernel(const StepArgs a) {
  __shared__ StepShared<MR> sh;
  Step<MR> step(a, sh);
  if (threadIdx.x == 0) {
    const unsigned int come = __hip_atomic_fetch_add(a.ws, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
    unsigned int none = 0;
    if (come == kGroups) __hip_atomic_compare_exchange_strong(a.ws + 1, &none, 1u, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    unsigned int mode;
    const int most = (int)a.ws[3];
    for (int asks = 0;; ++asks) {
      mode = __hip_atomic_load(a.ws + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (mode != 0) break;
      if (asks >= most) {
        none = 0;
        __hip_atomic_compare_exchange_strong(a.ws + 1, &none, 2u, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);        // (then the next look sees whose word it is)
      }
    }
    sh.mode = (int)mode;
  }
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(sh.mode) == 1) step.run_fixed();
}

// behind it: the step where not every workgroup was there (a kernel of its own, so that the other keeps its registers; it leaves at once otherwise)
template <int MR>
__global__ __launch_bounds__(kThreads) void decode_step_dealt_kernel(const StepArgs a) {
  __shared__ StepShared<MR> sh;
  if (a.ws[1] != 2) return;
  Step<MR> step(a, sh);
  step.run_dealt();
}

// empty exchange words, the sync words, the step's input as v in front of the first layer
__global__ __launch_bounds__(256) void decode_step_begin_kernel(unsigned int* ws, int64_t exchange, const bf16_t* __restrict__ x, int n, unsigned int patience,
                                                                unsigned int asks, int32_t* gave_up, const int32_t* __restrict__ ctx,
                                                                int rows, int parts) {
  const int64_t at = (int64_t)blockIdx.x * 256 + threadIdx.x, stride = (int64_t)gridDim.x * 256;
  u32x4_t* words = reinterpret_cast<u32x4_t*>(ws + kSyncWords);
  for (int64_t i = at; i < exchange / 4; i += stride) words[i] = u32x4_t{kEmpty, kEmpty, kEmpty, kEmpty};
  for (int64_t i = at; i < n; i += stride) {
    const unsigned int v = __float_as_uint((float)x[i]);
    ws[kSyncWords + exchange + i] = v == kEmpty ? 0x7FFF7FFFu : v;
  }
  if (at < kCutKeys) ws[at] = at == 1 ? (patience == 0 ? 2u : 0u) : at == 3 ? patience : at == 4 ? asks == 0 : 0u;
  if (at == 256) cut_contexts(ws, ctx, rows, parts);
  if (at == 0 && asks == 0 && gave_up) *gave_up = 1;        // (no wait at all is allowed: given up from the start)
}

int step_parts(int64_t batch, int hkv) {
  const int64_t parts = (kGroups - batch * hkv * 2) / (batch * hkv);
  return (int)(parts < kMaxParts ? parts : kMaxParts);
}

bool step_covers(int64_t batch, int layers, int hidden, int ff, int hq, int hkv) {
  return batch >= 1 && batch <= 4 && layers >= 1 && layers <= kMaxLayers && hidden == kWidth && ff > 0 && ff % 1024 == 0 && ff <= kMaxFf && hkv > 0 && hq == 2 * hkv &&
         (hq == 8 || hq == 16);
}

}  // namespace

extern "C" size_t nvl_decode_step_workspace_bytes(int64_t batch, int num_layers, int hidden, int ff, int num_q_heads, int num_kv_heads) {
  if (!step_covers(batch, num_layers, hidden, ff, num_q_heads, num_kv_heads)) return 0;
  const Exchange ex((int)batch, num_q_heads, num_kv_heads, ff, step_parts(batch, num_kv_heads));
  return (size_t)(kSyncWords + (int64_t)num_layers * ex.total + batch * kWidth) * 4;
}

extern "C" int nvl_decode_step(const void* x, const void* const* layers, int num_layers, float eps, const float* cos_sin, int64_t max_pos, const int32_t* block_tables,
                               int64_t bt_stride, const int32_t* context_lens, int64_t batch, int hidden, int ff, int num_q_heads, int num_kv_heads, int block_size,
                               float softmax_scale, float* hidden_out, void* residual_out, void* workspace, size_t workspace_bytes, int patience, int asks, int32_t* gave_up,
                               void* stream) {
  const size_t need = nvl_decode_step_workspace_bytes(batch, num_layers, hidden, ff, num_q_heads, num_kv_heads);
  NVL_REQUIRE(need > 0,
              "nvl_decode_step: %lld rows, %d layers of width %d, %d and %d / %d heads (up to 4 rows and %d layers, width %d, 1,024 to %d in thousands, 8 or 16 heads in pairs)",
              (long long)batch, num_layers, hidden, ff, num_q_heads, num_kv_heads, kMaxLayers, kWidth, kMaxFf);
  NVL_REQUIRE(x && layers && cos_sin && block_tables && context_lens && hidden_out && residual_out && workspace && block_size > 0 && max_pos > 0 && bt_stride > 0 && patience >= 0 &&
                  asks >= 0 && (uintptr_t)gave_up % 4 == 0,
              "nvl_decode_step: null pointer, block_size, max_pos, bt_stride, patience, asks or gave_up");
  NVL_REQUIRE(workspace_bytes >= need && (uintptr_t)workspace % 256 == 0, "nvl_decode_step: workspace of %zu bytes (%zu needed, 256-byte aligned)", workspace_bytes, need);
  StepArgs a;
  for (int l = 0; l < num_layers; ++l) {
    const void* const* p = layers + l * 10;
    for (int i = 0; i < 10; ++i) {
      const bool head_norm = i == 2 || i == 3;
      NVL_REQUIRE((p[i] != nullptr || head_norm) && (uintptr_t)p[i] % 16 == 0, "nvl_decode_step: layer %d: a pointer is null or not 16-byte aligned", l);
    }
    NVL_REQUIRE((p[2] == nullptr) == (p[3] == nullptr), "nvl_decode_step: layer %d: q/k norm weights come as a pair", l);
    a.layer[l] = StepLayer{(const bf16_t*)p[0], (const bf16_t*)p[1], (const bf16_t*)p[2], (const bf16_t*)p[3], (const bf16_t*)p[4],
                           (const bf16_t*)p[5], (const bf16_t*)p[6], (const bf16_t*)p[7], (bf16_t*)p[8], (bf16_t*)p[9]};
  }
  for (int l = num_layers; l < kMaxLayers; ++l) a.layer[l] = a.layer[0];
  a.cos_sin = cos_sin, a.tables = block_tables, a.ctx = context_lens, a.ws = (unsigned int*)workspace, a.hidden = hidden_out, a.residual = (bf16_t*)residual_out, a.gave_up = gave_up, a.asks = asks;
  a.bt_stride = bt_stride, a.max_pos = max_pos, a.eps = eps, a.scale_log2e = softmax_scale * 1.4426950408889634f;
  a.layers = num_layers, a.rows = (int)batch, a.hq = num_q_heads, a.hkv = num_kv_heads, a.ff = ff, a.block_size = block_size, a.parts = step_parts(batch, num_kv_heads);
  const Exchange ex(a.rows, a.hq, a.hkv, a.ff, a.parts);
  const int64_t exchange = (int64_t)num_layers * ex.total;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(decode_step_begin_kernel, dim3(512), dim3(256), 0, s, a.ws, exchange, (const bf16_t*)x, a.rows * kWidth, (unsigned int)patience, (unsigned int)asks, gave_up,
                     context_lens, a.rows, a.parts);
  const int rc = nvl_check_launch("nvl_decode_step");
  if (rc != NVL_OK) return rc;
  const auto launch = [&](auto fixed, auto dealt) {
    hipLaunchKernelGGL(fixed, dim3(kGroups), dim3(kThreads), 0, s, a);
    hipLaunchKernelGGL(dealt, dim3(kGroups), dim3(kThreads), 0, s, a);
  };
  if (batch == 1) launch(decode_step_kernel<1>, decode_step_dealt_kernel<1>);
  else if (batch == 2) launch(decode_step_kernel<2>, decode_step_dealt_kernel<2>);
  else launch(decode_step_kernel<4>, decode_step_dealt_kernel<4>);
  return nvl_check_launch("nvl_decode_step");
}
