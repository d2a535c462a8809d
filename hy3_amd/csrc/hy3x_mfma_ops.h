// hy3x_mfma_ops.h -- the Q4_K x fp16 MFMA building blocks shared by the
// grouped-GEMM tile kernels (hy3x_mfma.hip, hy3x_mfma_big.hip): operand
// types, the weight copy, the Q4_K scale unpack, the exact integer weight
// operands and the mins operand.
#pragma once
#include "hy3x_kernels.h"
#include "hy3x_q4k.h"
#include "hy3x_dma.h"

namespace hy3x {

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));  // 16 bytes as a native vector
typedef uint32_t u2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pk_fma_f16(uint32_t a, h2_t b, h2_t c) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(as_h2(a), b, c));
}

// The 6-bit scales and mins of a Q4_K block (hy3.c:1001-1009) as bytes:
// sc[0] = sc_0..3, sc[1] = sc_4..7, mn[0] = m_0..3, mn[1] = m_4..7.
struct Scales6 {
  uint32_t sc[2], mn[2];
};
__device__ __forceinline__ Scales6 unpack_scales(const u4_t &h) {
  // j < 4: sc_j = s[j] & 63, m_j = s[j+4] & 63
  // j >= 4: sc_j = (s[j+4] & 15) | (s[j-4] >> 6) << 4, m_j = (s[j+4] >> 4) | (s[j] >> 6) << 4
  Scales6 r;
  r.sc[0] = h.y & 0x3F3F3F3Fu;
  r.mn[0] = h.z & 0x3F3F3F3Fu;
  r.sc[1] = (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u);
  r.mn[1] = ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u);
  return r;
}

// The two bytes of w that `sel` picks (a v_perm selector: their indices in its
// bytes 0 and 2, 4 in bytes 1 and 3) as the fp16 pair 1024 + byte: each byte
// goes into the mantissa of 1024.0.
__device__ __forceinline__ h2_t bytes_h2(uint32_t w, uint32_t sel) {
  return as_h2(__builtin_amdgcn_perm(0x64646464u, w, sel));
}
// The selector of bytes 2 i and 2 i + 1.
__device__ __forceinline__ uint32_t bytes_sel(int i) {
  return 0x04000400u | (uint32_t)(2 * i + 1) << 16 | (uint32_t)(2 * i);
}

// The scales of a lane's sub-block pair (a low- and a high-nibble sub-block) as
// the operands of dequant_run: (sc_lo, sc_hi / 16) and -(1024 sc_lo, 64 sc_hi).
struct PairScale {
  h2_t mul, add;
};
__device__ __forceinline__ PairScale pair_scale(uint32_t scw, uint32_t sel) {
  const h2_t sc = bytes_h2(scw, sel) - (h2_t){(_Float16)1024.0f, (_Float16)1024.0f};
  PairScale r;
  r.mul = sc * (h2_t){(_Float16)1.0f, (_Float16)0.0625f};
  r.add = sc * (h2_t){(_Float16)-1024.0f, (_Float16)-64.0f};
  return r;
}

// Weight operands of one 8-byte run of qs: the low nibbles (sub-block scale
// sc_lo) and the high nibbles (sc_hi) as exact integers sc*q in fp16
// (sc*q <= 945). Low: 0x6400 | q = 1024 + q, times sc_lo, minus 1024 sc_lo.
// High, left in place: 0x6400 | 16q = 1024 + 16q, times sc_hi/16, minus
// 64 sc_hi. Each is one fused multiply-add whose exact result is
// representable, so it is exact.
__device__ __forceinline__ void dequant_run(u2_t q, const PairScale &ps, h8_t &w_lo,
                                            h8_t &w_hi) {
  const h2_t ml = {ps.mul[0], ps.mul[0]}, al = {ps.add[0], ps.add[0]};
  const h2_t mh = {ps.mul[1], ps.mul[1]}, ah = {ps.add[1], ps.add[1]};
  const uint32_t mag = 0x64006400u, m_lo = 0x000F000Fu, m_hi = 0x00F000F0u;
  const uint32_t x8 = q.x >> 8, y8 = q.y >> 8;
  u4_t lo, hi;
  lo.x = pk_fma_f16(and_or(q.x, m_lo, mag), ml, al);
  lo.y = pk_fma_f16(and_or(x8, m_lo, mag), ml, al);
  lo.z = pk_fma_f16(and_or(q.y, m_lo, mag), ml, al);
  lo.w = pk_fma_f16(and_or(y8, m_lo, mag), ml, al);
  hi.x = pk_fma_f16(and_or(q.x, m_hi, mag), mh, ah);
  hi.y = pk_fma_f16(and_or(x8, m_hi, mag), mh, ah);
  hi.z = pk_fma_f16(and_or(q.y, m_hi, mag), mh, ah);
  hi.w = pk_fma_f16(and_or(y8, m_hi, mag), mh, ah);
  w_lo = __builtin_bit_cast(h8_t, lo);
  w_hi = __builtin_bit_cast(h8_t, hi);
}

// The mins operand of a row-block (header hd) for the lane's sub-blocks j = 2g
// and 2g + 1 (their mins in the bytes of mw that sel picks): -dmin * m_j, each
// split exactly into two fp16 parts hi + lo (dmin: 11 significant bits, m: 6;
// the product's rounding error is one fused multiply-add away), laid out (hi, hi,
// hi, hi, lo, lo, lo, lo) over the two sub-blocks in turn against the staged
// activation sums (Sh, Sh, Sl, Sl, Sh, Sh, Sl, Sl: store_subsum): the four cross
// products of the two splits fill the MFMA's k slots. dmin is used as the half it is
// stored as:
// hy3.c's decode (fp16_quirk) reads a half with exponent 0 as 2^-15 (1 + mant /
// 1024), half of the half with exponent 1 and the same mantissa, so there m / 2
// (exact) meets that one. In packed fp16 this takes nine vector instructions;
// through fp32 conversions it took 28, of about 260 per wave and column.
__device__ __forceinline__ h8_t mins_operand(uint32_t hx, uint32_t mw, uint32_t sel) {
  const bool z = (hx & 0x7C000000u) == 0u;
  const _Float16 dmin = __builtin_bit_cast(_Float16, (uint16_t)((hx >> 16) | (z ? 0x0400u : 0u)));
  const _Float16 f1 = z ? (_Float16)0.5f : (_Float16)1.0f;
  const _Float16 f0 = z ? (_Float16)-512.0f : (_Float16)-1024.0f;
  const h2_t nd = {-dmin, -dmin};
  const h2_t m = __builtin_elementwise_fma(bytes_h2(mw, sel), (h2_t){f1, f1}, (h2_t){f0, f0});
  const h2_t hi = m * nd;
  const h2_t lo = __builtin_elementwise_fma(m, nd, -hi);
  return (h8_t){hi[0], hi[1], hi[0], hi[1], lo[0], lo[1], lo[0], lo[1]};
}

// Launch order -> work item (workgroups are dealt to the 8 XCDs round-robin).
// The first `shared` items, the shared expert's, go round the XCDs at the start
// of the launch: with Q8 weights they take twice as long as a routed expert's,
// and at the end of one XCD's work they were the launch's tail (8 tokens, Q8:
// gate/up 95.7 us and down 46.8, first and spread 83.4 and 40.4; 20: 146.8 and
// 86.5, 139.7 and 69.4). The rest: consecutive items on one XCD, so that the row
// tiles of one expert tile share its activations in that XCD's L2, and
// consecutive token tiles of one expert share its weights.
__device__ __forceinline__ int xcd_remap(int bid, int nblocks, int shared) {
  const int s8 = shared & ~7;
  if (bid < s8) return bid;
  nblocks -= s8;
  bid -= s8;
  const int q = nblocks >> 3, r = nblocks & 7, x = bid & 7, i = bid >> 3;
  return s8 + x * q + (x < r ? x : r) + i;
}

// Launch order -> work item with whole tiles dealt round-robin to the XCDs:
// tile j's nrt row tiles run consecutively on XCD j % 8 (sharing the tile's
// activations in that L2), and neighbouring tiles go to different XCDs. Work
// item w < n_tiles * nrt is block ((w / nrt / 8) * nrt + w % nrt) * 8 +
// (w / nrt) % 8, which is below (n_tiles + 7) * nrt: the grid needs
// XCD_TILE_RR_MARGIN = 7 tiles of margin; blocks whose item is past the work
// leave.
__device__ __forceinline__ int xcd_tile_rr(int bid, int nrt) {
  const int x = bid & 7, i = bid >> 3;
  return ((i / nrt) * 8 + x) * nrt + i % nrt;
}

// fp16 weights (exact q) of 8 consecutive bytes, in the staged activations'
// run order (0, 2, 1, 3, 4, 6, 5, 7).
__device__ __forceinline__ h8_t q8_run(u2_t b) {
  const uint32_t ex = 0x64646464u, a = b.x ^ 0x80808080u, c = b.y ^ 0x80808080u;
  const h2_t m1152 = {(_Float16)-1152.0f, (_Float16)-1152.0f};
  u4_t w;
  w.x = __builtin_bit_cast(uint32_t, as_h2(__builtin_amdgcn_perm(ex, a, 0x04020400u)) + m1152);
  w.y = __builtin_bit_cast(uint32_t, as_h2(__builtin_amdgcn_perm(ex, a, 0x04030401u)) + m1152);
  w.z = __builtin_bit_cast(uint32_t, as_h2(__builtin_amdgcn_perm(ex, c, 0x04020400u)) + m1152);
  w.w = __builtin_bit_cast(uint32_t, as_h2(__builtin_amdgcn_perm(ex, c, 0x04030401u)) + m1152);
  return __builtin_bit_cast(h8_t, w);
}

}  // namespace hy3x
