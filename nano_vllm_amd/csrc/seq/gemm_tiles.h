// Products of many 16-bit rows: rows X [n, K] times W [features, K]^T in tiles of 256 rows x 256 weight rows, for grouped expert products and dense
// layers. Included by moe.hip behind the helpers that it shares with the other products.
//
// What bounds it: the chip's power. At 1.2 to 1.5 PFLOP/s the clock falls from 2.4 to 1.7-2.0 GHz as the matrix pipe fills, so that what counts is the energy of a
// product and the issue slots beside it, not the pipe's idle time alone (the loop before this one had 56 % of the pipe's cycles at 2.2 GHz, with wider instructions and the
// requests spread it had 68 % at 1.8 GHz and took as long). Measured on MI355X, 14,600 rows, K 4096, 6,144 weight rows, without the results' end:
//   v_mfma_f32_32x32x16_bf16 538 us, v_mfma_f32_16x16x32_bf16 493 us: the smaller one moves half the accumulators per product.
//   Requests one by one between the products, and half of them a half step earlier: 12 % less than in bursts behind the step's barrier, where they also queue up for
//   the path into LDS (64 KB a step, 64 bytes a clock).
//   Products in an order in which one operand of two is the one before, either in turn: 1 % less than all of one row of blocks behind the other (8,192 x 24,576 x 4096 1125 -> 1112 us).
//   Results stored as a stream: they do not push out the operands that neighbours share (the same 1112 -> 1043 us; outputs below 130 MB the same either way).
//   Addresses as 32-bit offsets of a buffer, one LDS base for four requests, no branch in the loop: a step of 128 products takes 2,360 clocks, 2,715 before; 128 products
//   back to back 2,176.
//
// Four wavefronts, 128 x 128 each (one per SIMD, 256 accumulators: per 32 of k 16 operand reads for 64 products, which is half of what LDS gives). A step is 64 of
// k, 128 bytes of every row. LDS (160 KB) is a ring of five parts of 256 rows: rows of X take turns in three of them, rows of W in two. Rows of X of the step
// after the next are requested during a step's first half, rows of W during its second one, behind the step's one barrier: it says that the next step's parts are there (all but the
// eight youngest requests) and that this step's have been read. Operands of a half are read during the half before. 16-byte unit c of a row r sits at c ^ swizzle(r), so the 16 rows
// that an operand read touches lie on different banks.
//
// 256 workgroups go on from tile to tile: the last two steps of a tile ask for the first ones of the next. Results go through the ring's free part and out as whole rows of 128
// or 256 bytes; the number of stores does not depend on the rows that are there (those that are not go nowhere), so the next tile's waits can count them and none waits for them to drain.
// Tiles that are left for a last pass of at most 128 workgroups are halved: 14,600 rows and 24 feature tiles are 5.4 passes, not 6 (gate|up at K 1024 7 % of its time).
//
// us before (moe_gemm_pipe_kernel's tiles of 256 rows) / now, whole calls on one card: gate|up and SiLU, 14,600 rows, ff 3072, K 1024 185 / 155, K 4096 581 / 495; rows, 14,175 x 4096 x 4096
// 399 / 324 (the library 331), 14,600 x 4096 x 1024 128 / 107, 14,600 x 1024 x 3072 92 / 77. Against the library: ops_seq.py (tiles_rule, silu_linear_rows).
#pragma once
#include "tiles_reach.h"

// ring of five parts
constexpr int TILE_ROW = 128, TILE_PART = 256 * TILE_ROW, TILE_RING = 5 * TILE_PART;
constexpr uint32_t TILE_NOWHERE = 0xF0000000u, TILE_SKEW = 4096;

template <int MODE, bool PLAN>
__global__ __launch_bounds__(256, 1) void gemm_tiles_kernel(const bf16_t* __restrict__ X, int64_t ldx, const bf16_t* __restrict__ W, int nout, int K,
                                                            const int32_t* __restrict__ tile_expert, const int32_t* __restrict__ row_token, int tiles_m,
                                                            int tiles_n, uint32_t band_inverse, int rows, const bf16_t* __restrict__ bias,
                                                            bf16_t* __restrict__ out, int64_t ldo) {
  constexpr bool GLU = MODE == 1, GATHER = MODE == 1 || MODE == 2;    // (0: rows, 1: SiLU of gate times up, 2: squares of positive results, 3: rows plus a bias)
  constexpr int NG = GLU ? 2 : 1, BN = 256 / NG, R = 8;               // features of a tile, requests of a wavefront per part
  extern __shared__ __attribute__((aligned(128))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15;
  const int wn = wave & 1, wm = wave >> 1;
  const auto expert = [&](int tile) { return PLAN ? tile_expert[tile] : 0; };
  const auto token = [&](int64_t r) { return PLAN ? row_token[r] : (int)r < rows ? (int)r : -1; };
  if constexpr (PLAN) {                       // the row tiles that hold rows come first in a plan: how many are there
    int lo = 0, hi = tiles_m;                 // (the answer is in [lo, hi])
    while (lo < hi) {
      const int stride = (hi - lo + 63) / 64, at = lo + lane * stride;
      const int held = __builtin_popcountll(__ballot(at < hi && tile_expert[at < hi ? at : lo] >= 0));
      if (!held) hi = lo;
      else lo += (held - 1) * stride + 1, hi = min(hi, lo - 1 + stride);
    }
    tiles_m = lo;
  }
  // passes of 256 tiles, one per workgroup; a last pass of at most half as many goes in halves of 128 rows. Workgroups go to the eight XCDs
  // round-robin: each XCD takes a run of neighbours
  const int tiles = tiles_m * tiles_n, whole = tiles / 256, rest = tiles % 256;
  const bool halves = rest && rest <= 128;
  int pass = 0, rt = 0, ft = 0, sub = 0;
  bool low = false;                           // a tile of 128 rows
  const auto find = [&] {
    const bool last = pass >= whole;
    const int slots = !last ? 256 : halves ? 2 * rest : rest, per = (slots + 7) / 8, slot = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (pass > whole || (int)(blockIdx.x / 8) >= per || slot >= slots) return false;
    low = last && halves;
    const int t = pass * 256 + (low ? slot / 2 : slot);
    int band = (int)__umulhi((uint32_t)t, band_inverse), k = t - band * 8 * tiles_n;
    if (k < 0) --band, k += 8 * tiles_n;
    const int high = min(8, tiles_m - band * 8);
    ft = high == 8 ? k / 8 : k / high, rt = band * 8 + (high == 8 ? k % 8 : k % high), sub = low ? slot % 2 * 128 : 0;
    return true;
  };
  if (!find()) return;
  int e = expert(rt);
  // Request i of a wavefront brings eight rows of a part, lane l unit (l & 7) ^ swizzle of row l >> 3. A tile of 128 rows has 64 for either pair of wavefronts. The
  // offsets leave out what the instruction adds to both of its addresses
  uint32_t xoff[R], woff[R];
  int tok[R];
  const auto look = [&] {
    if constexpr (GATHER) {
      int l = lane;
      asm volatile("" : "+v"(l));             // (what follows from the lane alone is worked out here, not kept over the loop)
      const int64_t first = (int64_t)rt * 256 + sub + (low ? (wave >> 1) * 64 : wave * 64) + (l >> 3);
#pragma unroll
      for (int i = 0; i < R; ++i) tok[i] = low && (wave & 1) ? -1 : token(first + i * 8);
    }
  };
  const auto near = [&](const bf16_t* p, uint32_t n) { return __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)p - TILE_SKEW), 0, (int)n, 0x00020000); };
  __amdgpu_buffer_rsrc_t xs = near(X, TILE_REACH), ws;
  const auto point = [&] {
    int l = lane;
    asm volatile("" : "+v"(l));
    ws = near(W + (int64_t)e * NG * nout * K, TILE_REACH);
    const uint32_t x2 = (uint32_t)ldx * 2, w2 = (uint32_t)K * 2;
    const int l3 = l >> 3, u = l & 7, f = ft * BN + wave * 64 % BN + l3;
    const uint32_t wfirst = (uint32_t)(wave * 64 / BN * nout + f) * w2 + TILE_SKEW;
    const int first = rt * 256 + sub + (low ? (wave >> 1) * 64 : wave * 64) + l3;
    const uint32_t xfirst = (uint32_t)first * x2 + TILE_SKEW;
    const bool none = low && (wave & 1);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const uint32_t xunit = (u ^ ((i * 4 & 4) | l3 >> 1)) * 16 - i % 4 * 1024, wunit = (u ^ ((l3 >> 1 & 1) | (i * 2 & 6))) * 16 - i % 4 * 1024;
      if constexpr (!GATHER) xoff[i] = none || (!PLAN && first + i * 8 >= rows) ? TILE_NOWHERE : xfirst + i * 8 * x2 + xunit;
      else xoff[i] = tok[i] < 0 ? TILE_NOWHERE : (uint32_t)tok[i] * x2 + TILE_SKEW + xunit;
      woff[i] = f + i * 8 < nout ? wfirst + i * 8 * w2 + wunit : TILE_NOWHERE;
    }
  };
  look();
  point();
  const auto request = [&](bool w, int i, int at, int step) {          // request i of a part of rows of X or W into the slot at byte `at`
    lds_void_t* to = (lds_void_t*)(lds + at + (wave * R + i / 4 * 4) * 8 * TILE_ROW);
    if (i % 4 == 0) __builtin_amdgcn_raw_ptr_buffer_load_lds(w ? ws : xs, to, 16, w ? woff[i] : xoff[i], step * TILE_ROW, 0, 0);
    if (i % 4 == 1) __builtin_amdgcn_raw_ptr_buffer_load_lds(w ? ws : xs, to, 16, w ? woff[i] : xoff[i], step * TILE_ROW, 1024, 0);
    if (i % 4 == 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(w ? ws : xs, to, 16, w ? woff[i] : xoff[i], step * TILE_ROW, 2048, 0);
    if (i % 4 == 3) __builtin_amdgcn_raw_ptr_buffer_load_lds(w ? ws : xs, to, 16, w ? woff[i] : xoff[i], step * TILE_ROW, 3072, 0);
  };
  struct Operands {
    u32x4_t x[8], w[8];
  };
  const int unit0 = ((lane >> 4) ^ ((li >> 1) & 7)) * 16;
  const char* wrow = lds + (wn * (GLU ? 64 : 128) + (li >> 2) * 8 + (li & 3)) * TILE_ROW;
  const char* xrow = lds + (wm * 128 + li) * TILE_ROW;
  const auto read = [&](Operands& o, bool w, int i, int half, int at) {
    const int place = at + (unit0 ^ (half * 64));
    if (w) o.w[i] = *(const u32x4_t*)(wrow + place + (GLU ? i / 4 * 128 + i % 4 / 2 * 32 + i % 2 * 4 : i / 2 * 32 + i % 2 * 4) * TILE_ROW);
    else o.x[i] = *(const u32x4_t*)(xrow + place + i * 16 * TILE_ROW);
  };
  // A half of a step: 8 RB products. The next half's operands are read and requests go out between them
  const auto half_step = [&](auto RBC, auto FIRST, auto& acc, const Operands& now, Operands& next, int half, int xat, int wat, bool w, int ask_at, int ask_step) {
    constexpr int RB = decltype(RBC)::value, READS = RB + 8;
#pragma unroll
    for (int n = 0; n < 8 * RB; ++n) {
      const int m = n / 2 % RB, pair = n / 2 / RB, b = pair % 2 ? RB - 1 - m : m, a = pair * 2 + (m % 2 ? 1 - n % 2 : n % 2);      // (either operand in turn is the one before)
      if constexpr (decltype(FIRST)::value) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(acc[a][b]) : "v"(now.w[a]), "v"(now.x[b]));
      else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[a][b]) : "v"(now.w[a]), "v"(now.x[b]));
      __builtin_amdgcn_sched_barrier(0);
      constexpr int EVERY = RB == 8 ? 3 : 2;
      if (n % EVERY == 0 && n / EVERY < READS) {
        const int k = n / EVERY;
        if (k < 2 * RB) read(next, k % 2, k / 2, half, k % 2 ? wat : xat);
        else read(next, true, k - RB, half, wat);
      }
      if (n % RB == RB - 1) request(w, n / RB, ask_at, ask_step);
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
  };
  // the ring: rows of X go round in the first three slots, rows of W in the other two
  int x0 = 0, x1 = TILE_PART, x2 = 2 * TILE_PART, w0 = 3 * TILE_PART, w1 = 4 * TILE_PART;
  const int steps = K / 64;
  Operands a, b;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int i = 0; i < R; ++i) request(false, i, s ? x1 : x0, s);
#pragma unroll
    for (int i = 0; i < R; ++i) request(true, i, s ? w1 : w0, s);
  }
  __builtin_amdgcn_s_waitcnt(0x4F70);         // vmcnt(16): the first step is there
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) read(a, false, i, 0, x0), read(a, true, i, 0, w0);
  __builtin_amdgcn_s_waitcnt(0xC07F);
  constexpr int STORES = GLU ? 16 : 32;       // of a tile of 256 rows, younger than the requests its end left (nothing follows one of 128)
  bool stored = false;
  const auto tile = [&](auto RBC) {
    constexpr int RB = decltype(RBC)::value;
    const int64_t row0 = (int64_t)rt * 256 + sub + wm * RB * 16;
    const int f0 = ft * BN + wn * (BN / 2);
    ++pass;
    const bool more = find();
    int e_next = more ? expert(rt) : -1;
    if (more) look();
    f32x4_t acc[8][RB];                       // [block of 16 weight rows][block of 16 rows]
    int live[RB];
    u32x4_t offset[4];                        // the bias of a lane's features
    int s = 0, ahead = 2;
#pragma unroll 1
    do {
      if (ahead == steps) {
        ahead = 0;
        if (more) {
          e = e_next;
          point();
        } else {                              // nothing follows: the last requests bring nothing
          xs = near(X, 0), ws = near(W, 0);
        }
        if constexpr (MODE == 3) {
#pragma unroll
          for (int j = 0; j < 4; ++j) offset[j] = *(const u32x4_t*)(bias + min(f0 + j * 32 + (lane >> 4) * 8, nout - 8));
        }
        if constexpr (PLAN) {
#pragma unroll
          for (int i = 0; i < RB; ++i) live[i] = token(row0 + i * 16 + li);
        }
      }
      if (s == 0) {
        half_step(RBC, std::true_type{}, acc, a, b, 1, x0, w0, false, x2, ahead);
        if (!stored) __builtin_amdgcn_s_waitcnt(0x0F78);               // vmcnt(8): the next step's parts are there
        else __builtin_amdgcn_s_waitcnt(0x0F78 + STORES / 16 * 0x4000);          // ... (8 + STORES)
      } else {
        half_step(RBC, std::false_type{}, acc, a, b, 1, x0, w0, false, x2, ahead);
        __builtin_amdgcn_s_waitcnt(0x0F78);
      }
      __builtin_amdgcn_s_barrier();           // ... everybody's, and this step's have been read
      __builtin_amdgcn_sched_barrier(0);
      half_step(RBC, std::false_type{}, acc, b, a, 0, x1, w1, true, w0, ahead);
      const int x = x0, w = w0;
      x0 = x1, x1 = x2, x2 = x, w0 = w1, w1 = w;
      ++ahead;
    } while (++s < steps);
    int l = lane;
    asm volatile("" : "+v"(l));
    asm volatile("s_nop 15\n\ts_nop 15");     // the last products are written before they are read: every read depends on one of
#pragma unroll                            // these statements, and volatile ones keep their order
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < RB; ++j) asm volatile("" : "+a"(acc[i][j]));
    // a row block's results go through the ring's free slot (where this wavefront's next requests go) and out as whole rows
    constexpr int UNITS = GLU ? 8 : 16, PER = 64 / UNITS;              // 16-byte units of a row, rows of a store
    u32x4_t* turn = (u32x4_t*)(lds + x2 + wave * R * 8 * TILE_ROW);
    const auto place = [&](int r, int u) { return r * UNITS + (u ^ ((UNITS == 16 ? r : r >> 1) & (UNITS - 1))); };
    const int unit = l % UNITS, line = l / UNITS;
    const uint32_t to = (uint32_t)(line * (int)ldo + unit * 8) * 2;
    const bool inside = f0 + unit * 8 < nout;
    const __amdgpu_buffer_rsrc_t os = __builtin_amdgcn_make_buffer_rsrc((void*)(out + row0 * ldo + f0), 0, (int)TILE_REACH, 0x00020000);
    const auto turn_in = [&](int rb) {        // (two row blocks have room: one is read while the next one's results are worked out)
#pragma unroll
      for (int j = 0; j < UNITS / 4; ++j) {
        union { bf16_t v[8]; u32x4_t q; } o;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float y = acc[2 * j + i / 4][rb][i % 4];
          if constexpr (GLU) o.v[i] = (bf16_t)silu_times<bf16_t>(y, acc[2 * j + i / 4 + 4][rb][i % 4]);
          else if constexpr (MODE == 3) o.v[i] = (bf16_t)(y + __builtin_bit_cast(float, i % 2 ? offset[j][i / 2] & 0xFFFF0000u : offset[j][i / 2] << 16));
          else o.v[i] = (bf16_t)plain_value(y, MODE);
        }
        turn[rb % 2 * 16 * UNITS + place(l & 15, j * 4 + (l >> 4))] = o.q;
      }
    };
    turn_in(0);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      u32x4_t q[16 / PER];
#pragma unroll
      for (int p = 0; p < 16 / PER; ++p) q[p] = turn[rb % 2 * 16 * UNITS + place(p * PER + line, unit)];
      __builtin_amdgcn_sched_barrier(0);
      if (rb + 1 < RB) turn_in(rb + 1);
      __builtin_amdgcn_sched_barrier(0);
      const uint32_t on = (uint32_t)__ballot((PLAN ? live[rb] : token(row0 + rb * 16 + (l & 15))) >= 0);
#pragma unroll
      for (int p = 0; p < 16 / PER; ++p)      // (2: not to be kept in the caches)
        __builtin_amdgcn_raw_buffer_store_b128(q[p], os, (on >> (p * PER + line) & 1) && inside ? to : TILE_NOWHERE, (rb * 16 + p * PER) * (int)ldo * 2, 2);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    static_assert(RB == 4 || RB * 16 / PER == STORES, "the next tile's first wait counts them");
    stored = true;
    return more;
  };
  bool more = true;
#pragma unroll 1
  while (more && !low) more = tile(std::integral_constant<int, 8>{});
  if (more) tile(std::integral_constant<int, 4>{});
  __builtin_amdgcn_s_waitcnt(0x0F70);         // (requests that bring nothing still write)
}

// the calls that the tiles take: rows of whole 128-byte pieces (two at least), results in whole 16-byte units, offsets within 32 bits
inline bool tiles_fit(int64_t ldx, int64_t rows, int nout, int K, int64_t weights, const void* out, int64_t ldo) {
  return K % 64 == 0 && K >= 128 && ((nout | ldo) & 7) == 0 && ((uintptr_t)out & 15) == 0 && tiles_reach(rows, ldx, weights, ldo) &&
         (rows + 255) / 256 * ((nout + 127) / 128) < (1ll << 31);
}

template <int MODE, bool PLAN>
int launch_tiles(const void* X, int64_t ldx, const void* W, int nout, int K, const int32_t* tile_expert, const int32_t* row_token, int64_t cap, void* out,
                 int64_t ldo, hipStream_t st, const char* who, int rows = 0, const void* bias = nullptr) {
  constexpr int BN = MODE == 1 ? 128 : 256;
  const int64_t tiles_m = (cap + 255) / 256, tiles_n = (nout + BN - 1) / BN;
  const auto kernel = gemm_tiles_kernel<MODE, PLAN>;
  NVS_LDS_ROOM(kernel, TILE_RING, who);
  kernel<<<dim3(256), dim3(256), TILE_RING, st>>>((const bf16_t*)X, ldx, (const bf16_t*)W, nout, K, tile_expert, row_token, (int)tiles_m, (int)tiles_n, (uint32_t)((1ull << 32) / (8 * tiles_n) + 1), rows,
                                                  (const bf16_t*)bias, (bf16_t*)out, ldo);
  return nvs_check_launch(who);
}
