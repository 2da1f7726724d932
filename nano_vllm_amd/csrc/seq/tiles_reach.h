// What the products in tiles of 256 rows (gemm_tiles.h) reach with 32-bit offsets of a buffer. Plain C++: the callers' rule (ops_seq.py) is held against it on the host.
#pragma once
#include <cstdint>

// bytes of a buffer that offsets may name; 8 KiB of them are left for what is added to a row's and for the skew of the base
constexpr uint32_t TILE_REACH = 0xC0000000u;
constexpr int64_t TILE_OPERAND = (int64_t)TILE_REACH - 8192;

// rows X of `rows` x ldx entries, `weights` entries of W, results ldo entries apart (a row block's 128 rows lie within 1 GiB)
inline bool tiles_reach(int64_t rows, int64_t ldx, int64_t weights, int64_t ldo) {
  return rows * ldx * 2 < TILE_OPERAND && weights * 2 < TILE_OPERAND && ldo < (1 << 22);
}
