// How a context is cut into parts (decode attention of few sequences, and the projection that merges its open parts). Plain C++: the split is enumerated on the host as well.
#pragma once

#ifdef __HIPCC__
#define NVL_FEW_FN __host__ __device__ __forceinline__
#else
#define NVL_FEW_FN inline
#endif

constexpr int NVL_OPEN_PART_TILES = 8;           // tiles of 32 tokens of a part that is left open

// ceil(a / b), a up to 2^20: (a + b - 1/2) / b is half a b-th away from the next whole number, which the reciprocal's error (2^-22) does not reach. (An integer division
// is some 30 instructions in the chain in front of the first request: 0.2 us a layer.)
NVL_FEW_FN int nvl_few_div(int a, int b) {
#if defined(__HIP_DEVICE_COMPILE__)
  return (int)(((float)(a + b) - 0.5f) * __builtin_amdgcn_rcpf((float)b));
#else
  return (int)(((float)(a + b) - 0.5f) * (1.f / (float)b));
#endif
}

// Parts of a context of `tiles` tiles: part_tiles tiles each, more where `parts` do not suffice. Part p takes tiles [p per, p per + per) with per = ceil(tiles / n):
// none is empty, so the part that ends with the last tile, which brings the new token, is one. (Of `parts` parts themselves the last ones may be empty: 129 tiles
// in 16 are 15 of 9.)
NVL_FEW_FN int nvl_few_split(int tiles, int part_tiles, int parts) {
  const int n = (tiles + part_tiles - 1) / part_tiles;
  if (n <= parts) return n < 1 ? 1 : n;
  return nvl_few_div(tiles, nvl_few_div(tiles, parts));
}
