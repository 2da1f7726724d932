// Shared helpers of libnvl_seq.so (gfx950 only: 64-wide wavefronts are assumed throughout).
#pragma once
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <atomic>
#include "../../../include/nvl_seq.h"

typedef __bf16 bf16_t;

void nvs_set_error(const char* fmt, ...);
int nvs_check_launch(const char* what);

#define NVS_REQUIRE(cond, ...)       \
  do {                               \
    if (!(cond)) {                   \
      nvs_set_error(__VA_ARGS__);    \
      return NVS_EINVAL;             \
    }                                \
  } while (0)

// Room for a kernel's dynamic LDS, once on each device that the process launches it on
#define NVS_LDS_ROOM(kernel, bytes, what)                                                                                                                     \
  do {                                                                                                                                                        \
    static std::atomic<uint64_t> nvs_room{0};                                                                                                                 \
    int nvs_device = 0;                                                                                                                                       \
    (void)hipGetDevice(&nvs_device);                                                                                                                          \
    if (!(nvs_room.load(std::memory_order_relaxed) >> (nvs_device & 63) & 1)) {                                                                               \
      NVS_REQUIRE(hipFuncSetAttribute((const void*)(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess,                                \
                  "%s: %d bytes of LDS were refused", what, (int)(bytes));                                                                                \
      nvs_room.fetch_or(1ull << (nvs_device & 63), std::memory_order_relaxed);                                                                                \
    }                                                                                                                                                         \
  } while (0)

// element access in 32-bit whatever the storage type
__device__ __forceinline__ float ldf(const float* p) { return *p; }
__device__ __forceinline__ float ldf(const bf16_t* p) { return (float)*p; }
__device__ __forceinline__ void stf(float* p, float v) { *p = v; }
__device__ __forceinline__ void stf(bf16_t* p, float v) { *p = (bf16_t)v; }   // round to nearest even

// VEC consecutive elements at once (16 / 8 bytes for VEC 4; the address is aligned to VEC elements)
template <int VEC>
__device__ __forceinline__ void ldv(const float* p, float (&v)[VEC]) {
  if constexpr (VEC == 4) {
    const float4 f = *(const float4*)p;
    v[0] = f.x, v[1] = f.y, v[2] = f.z, v[3] = f.w;
  } else {
#pragma unroll
    for (int i = 0; i < VEC; ++i) v[i] = p[i];
  }
}
template <int VEC>
__device__ __forceinline__ void ldv(const bf16_t* p, float (&v)[VEC]) {
  if constexpr (VEC == 4) {
    typedef __attribute__((ext_vector_type(4))) __bf16 b4_t;
    const b4_t b = *(const b4_t*)p;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (float)b[i];
  } else {
#pragma unroll
    for (int i = 0; i < VEC; ++i) v[i] = (float)p[i];
  }
}
template <int VEC>
__device__ __forceinline__ void stv(float* p, const float (&v)[VEC]) {
  if constexpr (VEC == 4) *(float4*)p = make_float4(v[0], v[1], v[2], v[3]);
  else {
#pragma unroll
    for (int i = 0; i < VEC; ++i) p[i] = v[i];
  }
}
template <int VEC>
__device__ __forceinline__ void stv(bf16_t* p, const float (&v)[VEC]) {
  if constexpr (VEC == 4) {
    typedef __attribute__((ext_vector_type(4))) __bf16 b4_t;
    b4_t b;
#pragma unroll
    for (int i = 0; i < 4; ++i) b[i] = (bf16_t)v[i];
    *(b4_t*)p = b;
  } else {
#pragma unroll
    for (int i = 0; i < VEC; ++i) p[i] = (bf16_t)v[i];
  }
}

// N (a power of two up to 8) consecutive elements in one piece (the address is aligned to the piece)
template <int N, typename T>
__device__ __forceinline__ void ldp(const T* p, float (&v)[N]) {
  typedef __attribute__((ext_vector_type(N))) T vec_t;
  const vec_t f = *(const vec_t*)p;
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = (float)f[i];
}
template <int N, typename T>
__device__ __forceinline__ void stp(T* p, const float (&v)[N]) {
  typedef __attribute__((ext_vector_type(N))) T vec_t;
  vec_t f;
#pragma unroll
  for (int i = 0; i < N; ++i) f[i] = (T)v[i];
  *(vec_t*)p = f;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
// sum over a workgroup of up to 1024 threads; `red` is LDS for 16 floats; every thread gets the result
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  const int w = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  __syncthreads();                       // `red` may still be read from a previous call
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  float s = 0.f;
  for (int i = 0; i < nw; ++i) s += red[i];
  return s;
}

// e^x from the hardware's 2^x of a fraction in [-1/2, 1/2], to a unit in the last place; x is taken as no less than -100 and no more than 88
// (by comparisons that a NaN fails: fmaxf would make it -100). The fraction is taken off in one fused step: x log2 e rounded first, and what
// rounding took added back, is what the compiler's own fusing of that difference adds twice (27 x 2^-24 at e^28).
__device__ __forceinline__ float exp_hw(float x) {
  const float c = x < -100.f ? -100.f : x > 88.f ? 88.f : x, n = rintf(c * 1.44269504088896341f);
  const float f = fmaf(c, 1.92596299112661747e-8f, fmaf(c, 1.44269504088896341f, -n));
  return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(f), (int)n);
}
// 1 / (1 + e^-x), the reciprocal with one step of Newton
__device__ __forceinline__ float sigmoid_hw(float x) {
  const float d = 1.f + exp_hw(-x), r = __builtin_amdgcn_rcpf(d);
  return fmaf(fmaf(-d, r, 1.f), r, r);
}
// (e^x - 1 - x) / x^2 for x in [-1, 0]: the Taylor polynomial
__device__ __forceinline__ float expm1_tail(float x) {
  float p = 2.50521083854417188e-8f;                // 1 / 11!, 1 / 10!, ..., 1 / 2!
  p = fmaf(p, x, 2.75573192239858907e-7f), p = fmaf(p, x, 2.75573192239858907e-6f), p = fmaf(p, x, 2.48015873015873016e-5f);
  p = fmaf(p, x, 1.98412698412698413e-4f), p = fmaf(p, x, 1.38888888888888889e-3f), p = fmaf(p, x, 8.33333333333333333e-3f);
  p = fmaf(p, x, 4.16666666666666667e-2f), p = fmaf(p, x, 1.66666666666666667e-1f), p = fmaf(p, x, 0.5f);
  return p;
}
// e^x - 1 - x for x <= 0, and 1 - e^x, both without the cancellation near 0
__device__ __forceinline__ float expm1_less_x(float x) { return x > -1.f ? expm1_tail(x) * x * x : exp_hw(x) - 1.f - x; }
__device__ __forceinline__ float one_less_exp(float x) { return x > -1.f ? -fmaf(expm1_tail(x) * x, x, x) : 1.f - exp_hw(x); }

// one token and channel of the real-gated linear recurrence S <- a S + add: la = log a. sp = softplus(lam)
struct RglruTerms {
  float la, a, add;
};
__device__ __forceinline__ RglruTerms rglru_terms(float gr, float gi, float u, float sp, float c) {
  RglruTerms v;
  v.la = -c * sigmoid_hw(gr) * sp;
  v.a = exp_hw(v.la);
  const float om = fmaxf(one_less_exp(2.f * v.la), 0.f);            // 1 - a^2, without cancellation near a = 1; then its root
  const float rs = __builtin_amdgcn_rsqf(om), s0 = om * rs;
  v.add = (om > 1e-30f ? fmaf(fmaf(-s0, s0, om) * 0.5f, rs, s0) : sqrtf(om)) * (sigmoid_hw(gi) * u);
  return v;
}

// A portion and its tokens [t0, t1) in the step
struct PortionSpan {
  int s, t0, t1;
};

// The portion that is number `rank` by length (in chunks of 16 tokens), longest first, of 2 to 64: workgroups start in the order of their numbers, so what is left for
// the end of a launch is short. Its length is found bit by bit, a ballot each: counting for every portion how many are longer took a workgroup 1 us, which is as
// long as a short portion's scan. All lanes of the wavefront call it.
__device__ __forceinline__ PortionSpan portion_by_length(const int32_t* __restrict__ cu_q, int nseq, int rank) {
  const int lane = threadIdx.x & 63, t0 = cu_q[lane < nseq ? lane : 0], t1 = cu_q[lane < nseq ? lane + 1 : 0];
  const int mine = lane < nseq ? (t1 - t0 + 15) >> 4 : -1;
  int longest = (__builtin_amdgcn_readlane(t1, nseq - 1) - __builtin_amdgcn_readfirstlane(t0) + 15) >> 4, v = 0;        // (not more than all of them)
  for (int bit = 31 - __builtin_clz(longest | 1); bit >= 0; --bit) {
    const int more = v | 1 << bit;
    if (__builtin_popcountll(__ballot(mine >= more)) > rank) v = more;
  }
  const uint64_t as_long = __ballot(mine == v);       // (ties in the order they come; all ballots by all lanes)
  const int longer = __builtin_popcountll(__ballot(mine > v));
  const int before = __builtin_amdgcn_mbcnt_hi((uint32_t)(as_long >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)as_long, 0));
  const int s = __builtin_ctzll(__ballot(mine == v && longer + before == rank));
  return {s, __builtin_amdgcn_readlane(t0, s), __builtin_amdgcn_readlane(t1, s)};
}

__device__ __forceinline__ float sigmoidf_(float x) { return 1.f / (1.f + __expf(-x)); }
__device__ __forceinline__ float softplusf_(float x) { return x > 20.f ? x : log1pf(expf(x)); }
// x / (1 + e^-x) with the hardware's exponential and reciprocal: what the rounding of x log2 e took (up to |x| units of 2^-24) is added back, and so is the quotient's
// remainder (far below 1, and no number behind an infinite x). Within 4 x 2^-24 above -30; 0 below -87
__device__ __forceinline__ float silu_hw(float x) {
  const float c = __builtin_amdgcn_fmed3f(x, -88.f, 88.f), t = c * -1.44269504088896341f;
  const float left = fmaf(t, 1.90465429995776804e-9f, fmaf(t, -0.693147182464599609f, -c));       // -c - t ln 2
  const float e = __builtin_amdgcn_exp2f(t), d = fmaf(e, left, e) + 1.f, r = __builtin_amdgcn_rcpf(d), q = x * r;
  return fmaf(__builtin_amdgcn_fmed3f(fmaf(-d, q, x), -1.f, 1.f), r, q);
}
__device__ __forceinline__ float siluf_(float x) { return x / (1.f + expf(-x)); }
__device__ __forceinline__ float gelu_tanhf_(float z) {
  return 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}

__device__ __forceinline__ float glu_value(float g, float u, int kind, float limit, float alpha) {
  if (kind == 0) return g / (1.f + expf(-g)) * u;               // silu(g) * u
  if (kind == 2) return gelu_tanhf_(g);                         // ungated: the tanh form of GELU (u is not read)
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g / (1.f + expf(-alpha * g)) * (u + 1.f);              // clamped: g sigmoid(alpha g) (u + 1)
}

#define NVS_DISPATCH(dtype, ...)                       \
  do {                                                 \
    if ((dtype) == NVS_BF16) {                         \
      typedef bf16_t T;                                \
      __VA_ARGS__;                                     \
    } else {                                           \
      typedef float T;                                 \
      __VA_ARGS__;                                     \
    }                                                  \
  } while (0)
