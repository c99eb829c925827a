// Device helpers shared by the fp16 MFMA GEMM kernels.
#pragma once

#include "mnb_kernels.h"

namespace mnb {
namespace gemm {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kBK = 64;              // k per tile
constexpr int kUnits = kBK / 8;      // 16-byte units per LDS row

__device__ __forceinline__ int Swz(int row, int unit) {
  return row * kUnits + (unit ^ ((row >> 1) & 7));
}

__device__ __forceinline__ uint32_t PackHalf2(float lo, float hi) {
  const half2v h = {static_cast<_Float16>(lo), static_cast<_Float16>(hi)};
  return __builtin_bit_cast(uint32_t, h);
}

__device__ __forceinline__ uint32_t PkMulF16(uint32_t a, uint32_t b) {
  const half2v r = __builtin_bit_cast(half2v, a) * __builtin_bit_cast(half2v, b);
  return __builtin_bit_cast(uint32_t, r);
}

// Per (row, k-tile) operands of DequantWord: -(1024 + zp) and -(64 + zp)
// (exact in fp16) and the block scale in fp16.
struct DequantRow {
  uint32_t neg_lo, neg_hi, s;
};
__device__ __forceinline__ DequantRow MakeDequantRow(float s, uint32_t zp) {
  const float z = static_cast<float>(zp);
  return DequantRow{PackHalf2(-(1024.f + z), -(1024.f + z)), PackHalf2(-(64.f + z), -(64.f + z)),
                    PackHalf2(s, s)};
}

// One packed word of 8 nibbles (k order) -> 8 fp16 weights in [0,4,1,5,2,6,3,7]
// order, with no per-nibble shift: in fp16, 1024.0 (0x6400) has an ulp of 1
// and 64.0 (0x5400) an ulp of 1/16, so (w & 0x000F000F) | 0x6400.. is the
// pair 1024 + q of nibbles 0 | 4 and (w & 0x00F000F0) | 0x5400.. the pair
// 64 + q of nibbles 1 | 5, both exact; the same of w >> 8 gives nibbles
// 2 | 6 and 3 | 7. Adding -(1024 + zp) or -(64 + zp) leaves q - zp exactly,
// and one multiply by the fp16 scale rounds the weight once. Per word: one
// shift, four v_and_or_b32, four packed adds and four packed multiplies.
__device__ __forceinline__ uint4 DequantWord(uint32_t w, const DequantRow &r,
                                             const Masks &c) {
  const uint32_t w8 = w >> 8;
  const uint32_t h0 = (w & c.lo) | c.e1024;   // nibbles 0 | 4: 1024 + q
  const uint32_t h1 = (w & c.hi) | c.e64;     // nibbles 1 | 5: 64 + q
  const uint32_t h2 = (w8 & c.lo) | c.e1024;  // nibbles 2 | 6
  const uint32_t h3 = (w8 & c.hi) | c.e64;    // nibbles 3 | 7
  return make_uint4(PkMulF16(PkAddF16(h0, r.neg_lo), r.s), PkMulF16(PkAddF16(h1, r.neg_hi), r.s),
                    PkMulF16(PkAddF16(h2, r.neg_lo), r.s), PkMulF16(PkAddF16(h3, r.neg_hi), r.s));
}

// (scale fp16 | zp << 16 | zp << 28) -> the operands of DequantWord, one byte
// permute each: fp16 -(1024 + z) is 0xE400 | z (ulp 1 at 1024) and -(64 + z)
// 0xD400 | z << 4 (ulp 1/16 at 64), so the word's bytes 2 and 3 are their low
// bytes.
template <bool HAS_ZP>
__device__ __forceinline__ DequantRow RowFromSz(uint32_t w) {
  DequantRow r;
  r.s = __builtin_amdgcn_perm(w, w, 0x01000100u);  // the fp16 scale in both halves
  if constexpr (HAS_ZP) {
    constexpr uint32_t kHigh = 0x0000D4E4u;  // the high bytes
    r.neg_lo = __builtin_amdgcn_perm(w, kHigh, 0x00060006u);
    r.neg_hi = __builtin_amdgcn_perm(w, kHigh, 0x01070107u);
  } else {
    r.neg_lo = 0xE408E408u;  // -(1024 + 8)
    r.neg_hi = 0xD480D480u;  // -(64 + 8)
  }
  return r;
}

} // namespace gemm
} // namespace mnb
