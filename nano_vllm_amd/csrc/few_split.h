// How a context is cut into parts (decode attention of few sequences, and the projection that merges its open parts). Plain C++: the split is enumerated on the host as well.
#pragma once

#ifdef __HIPCC__
#define NVL_FEW_FN __host__ __device__ __forceinline__
#else
#define NVL_FEW_FN inline
#endif

constexpr int NVL_OPEN_PART_TILES = 8;           // tiles of 32 tokens of a part that is left open

// Parts of a context of `tiles` tiles: part_tiles tiles each, more where `parts` do not suffice. Part p takes tiles [p per, p per + per) with per = ceil(tiles / n):
// none is empty, so the part that ends with the last tile, which brings the new token, is one. (Of `parts` parts themselves the last ones may be empty: 129 tiles
// in 16 are 15 of 9.)
NVL_FEW_FN int nvl_few_split(int tiles, int part_tiles, int parts) {
  const int n = (tiles + part_tiles - 1) / part_tiles;
  if (n <= parts) return n < 1 ? 1 : n;
  const int per = (tiles + parts - 1) / parts;
  return (tiles + per - 1) / per;
}
