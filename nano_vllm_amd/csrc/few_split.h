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

// Whose parts come in fours: nvl_paged_attn_decode_open_fours', as nvl_linear_decode_open_fours asks for them (a second part costs it as much as a fourth, and the parts' tiles
// come in on more compute units, 28 bytes a clock each), and those of fused steps of up to four sequences. nvl_paged_attn_decode_open and nvl_linear_decode_open keep parts of
// eight tiles. Decode steps of Qwen3-0.6B in us, parts of eight tiles / fours, merged by the projection: one sequence, contexts of 300, 400, 700,
// 1,200, 1,600 and 2,000 tokens 806 813 823 850 853 852 / 791 803 811 829 846 854; two of 400, 700, 1,200, 2,000 832 843 866 873 / 818 829 850 875; three of up to 600, 1,000,
// 1,500, 2,000 876 884 910 922 / 836 859 888 905; four of 257 to 300, of up to 600, 1,000, 1,500, 2,000 857 897 882 922 961 / 844 858 878 924 948, of 100 to 300 896 / 900 (the one loss, 0.2 us a
// layer. With two parts instead of four for four sequences of up to 512 tokens it stays, 899, and the others lose: 257 to 300 858, 300 to 600 874). In a launch of their own:
// one of 300, 700, 2,000 tokens 842 867 870 / 834 853 871, two of up to 700 867 / 865, three of up to 1,000 907 / 908, four of up to 300, 600, 1,500, 2,000 934 907 943 986 /
// 941 893 943 986. More sequences stay as they were (fours for six of 600 964 / 953, eight of 1,200 1056 / 1061).
NVL_FEW_FN bool nvl_few_fours(int sequences) { return sequences <= 4; }

// Parts of a context of `tiles` tiles: part_tiles tiles each, more where `parts` do not suffice, fewer where that makes whole `fours`. Part p takes tiles [p per, p per + per) with
// per = ceil(tiles / n): none is empty, so the part that ends with the last tile, which brings the new token, is one. (Of `parts` parts themselves the last ones may be
// empty: 129 tiles in 16 are 15 of 9.) A single part is told first: the shortest contexts pay for no division.
NVL_FEW_FN int nvl_few_split(int tiles, int part_tiles, int parts, bool fours = false) {
  const int n = (tiles + part_tiles - 1) / part_tiles;
  if (n <= 1) return 1;
  const int up = fours ? 3 : 0, more = (n + up) & ~up;
  if (more == n && n <= parts) return n;
  return nvl_few_div(tiles, nvl_few_div(tiles, more < parts ? more : parts));
}
