// Which operands the general tile stages in whole chunks (GeneralTile, gemm_general.h).  Plain C++, so
// that the rule can be compiled and checked without a GPU.
#pragma once

#include <cstdint>

namespace moegemm {

// A chunk is 8 elements along an operand's unit stride; rows run along K, or (cols) along M or N.
struct ChunkRoute {
  bool a_rows, a_cols, b_rows, b_cols;
  constexpr bool chunked() const { return (a_rows || a_cols) && (b_rows || b_cols); }
};

// Strides in elements of `es` bytes, of any sign.  The chunks' addresses are a 64-bit base plus an unsigned
// 32-bit offset that spans a tile's rows (rows along K) or a slice's, so a pitch must not be negative (such
// an offset would land 4 GiB past its row) and a tile's rows must span less than 2^31 bytes; an operand
// that does not meet the rule is staged element by element with signed 64-bit indices.
constexpr ChunkRoute chunk_route(bool f32, int es, int bm, int bn, int64_t m, int64_t n, int64_t k, int64_t sam,
                                 int64_t sak, int64_t sbk, int64_t sbn) {
  // A pitch that is too large or negative has one of these bits.  (Two scalar instructions a pitch: signed
  // compares took registers that the split kernels spill, 28.7 -> 31.3 us on fp16 [777,2881]@[2881,1443].)
  const uint64_t past = ~((uint64_t(1) << 31) / (bm > bn ? bm : bn) / es - 1);
  const bool k_fits = k >= 8 && k * es < (int64_t(1) << 31);
  const bool deep = !f32 || k >= 8;  // shorter fp32 sums are closer with the fp32 instruction
  ChunkRoute r{};
  r.a_rows = sak == 1 && k_fits && (uint64_t(sam) & past) == 0;
  r.a_cols = deep && bm >= 32 && sam == 1 && m >= 8 && (uint64_t(sak) & past) == 0;
  r.b_rows = sbk == 1 && k_fits && (uint64_t(sbn) & past) == 0;
  r.b_cols = deep && sbn == 1 && n >= 8 && (uint64_t(sbk) & past) == 0;
  return r;
}

}  // namespace moegemm
